"""Inverted residual blocks in one launch (fp16, channels-last): which blocks the call takes, and programs around it
against the fp32 oracle on the same fp16-representable values."""
import ctypes as C

import numpy as np
import pytest

from helpers import ORACLE_PATH
from occamy_amd import _abi, compiler
from occamy_amd.ops import Ops
from test_gpu_e2e import as_fp32_graph, close16, run

pytestmark = pytest.mark.gpu

FLAGS = dict(fusion=True, fuse_residual=True, fuse_activations=True, fuse_matmul_bias=True, channels_last=True, alias_copies=True, compact_pool=True)


class ExecBlock(C.Structure):
    _fields_ = ([(n, C.c_void_p) for n in ("x", "w1", "b1", "wd", "bd", "w3", "b3", "z", "y")]
                + [(n, C.c_int64) for n in ("n", "cin", "h", "w", "ch", "r", "s", "stride", "pad_h", "pad_w", "p", "q", "cout", "act1", "actd", "act")]
                + [(n, C.c_float) for n in ("coef1", "coefd", "coef")] + [(n, C.c_int32) for n in ("expand", "dtype", "format", "filter_layout")])


def block(n, cin, h, w, ch, cout, stride, pad_h, pad_w, **kw):
    b = ExecBlock(n=n, cin=cin, h=h, w=w, ch=ch, r=3, s=3, stride=stride, pad_h=pad_h, pad_w=pad_w, cout=cout, expand=1, dtype=_abi.F16, format=_abi.NHWC,
                  p=(h + 2 * pad_h - 3) // stride + 1, q=(w + 2 * pad_w - 3) // stride + 1, act1=_abi.ACT_CLIPPED_RELU, actd=_abi.ACT_CLIPPED_RELU,
                  act=_abi.ACT_IDENTITY, coef1=6.0, coefd=6.0)
    for k, v in kw.items():
        setattr(b, k, v)
    return b


def test_which_blocks_the_call_takes():
    """Any padding the tiles can hold, and no other: wider ones, and results of another size than the geometry gives, stay
    with the three calls."""
    ops = Ops()
    applies = lambda b: ops.lib.dnnrtExecBlockApplies(ops.handle, C.byref(b))  # noqa: E731
    for stride in (1, 2):
        for ph in range(6):
            for pw in range(6):
                assert applies(block(64, 24, 56, 56, 144, 32, stride, ph, pw)) == (ph <= 2 and pw <= 2), (stride, ph, pw)
    assert not applies(block(64, 24, 56, 56, 144, 32, 1, -1, 0))
    assert not applies(block(64, 24, 56, 56, 144, 32, 1, 1, 1, p=57))
    assert not applies(block(64, 24, 56, 56, 144, 32, 2, 1, 1, q=29))
    assert not applies(block(64, 24, 2, 56, 144, 32, 1, 0, 0))
    ops.close()


def small_net(batch, height, width, stride, pads, dtype=np.float16, cin=24, hidden=144, cout=32, residual=False):
    """A 3x3 layer, one inverted residual block with the given depthwise padding, a 1x1 layer and a pooled result."""
    r = np.random.default_rng(batch * height + width + stride)
    g = compiler.Graph()
    c = lambda *s, f=1.0: g.constant((r.standard_normal(s) * f).astype(dtype))  # noqa: E731
    x = g.input("x", (batch, 3, height, width), dtype)

    def conv(v, ci, co, k, s, p, group=1):
        return g.node("Conv", [v, c(co, ci // group, k, k, f=np.sqrt(2.0 / (ci // group * k * k))), c(co, f=0.3)], kernel_shape=[k, k], pads=[p[0], p[1], p[0], p[1]],
                      strides=[s, s], group=group)

    def relu6(v):
        return g.node("Clip", [v, g.constant(np.array(0.0, dtype)), g.constant(np.array(6.0, dtype))])

    v = y = relu6(conv(x, 3, cin, 3, 1, (1, 1)))
    v = relu6(conv(v, cin, hidden, 1, 1, (0, 0)))
    v = relu6(conv(v, hidden, hidden, 3, stride, pads, hidden))
    v = conv(v, hidden, cout, 1, 1, (0, 0))
    if residual:
        v = g.node("Add", [v, y])
    v = relu6(conv(v, cout, 48, 1, 1, (0, 0)))
    g.output(g.node("Flatten", [g.node("GlobalAveragePool", [v])], axis=1))
    return g, [r.standard_normal((batch, 3, height, width)).astype(dtype)]


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("pads", [(0, 0), (1, 2), (2, 0), (2, 2), (3, 1), (1, 3), (4, 4), (5, 3)], ids=str)
def test_any_depthwise_padding(pads, stride):
    """Paddings the block call takes and paddings it leaves to the three calls; images down to a pixel or two."""
    for batch, height, width in ((8, 28, 31), (16, 9, 2), (16, 1, 12)):
        if height + 2 * pads[0] < 3 or width + 2 * pads[1] < 3:
            continue
        build = lambda: small_net(batch, height, width, stride, pads)  # noqa: E731
        ref, _ = run(lambda: as_fp32_graph(*build()), ORACLE_PATH, fusion=True)
        for mode in (compiler.MODE_OCCAMY, compiler.MODE_RESIDENT):
            got, _ = run(build, mode=mode, **FLAGS)
            close16(got[0], ref[0])
