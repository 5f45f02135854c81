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
                + [(n, C.c_float) for n in ("coef1", "coefd", "coef")] + [(n, C.c_int32) for n in ("expand", "dtype", "format")])


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


def small_net(batch, height, width, stride, pads, dtype=np.float16, cin=24, hidden=144, cout=32):
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

    v = relu6(conv(x, 3, cin, 3, 1, (1, 1)))
    v = relu6(conv(v, cin, hidden, 1, 1, (0, 0)))
    v = relu6(conv(v, hidden, hidden, 3, stride, pads, hidden))
    v = conv(v, hidden, cout, 1, 1, (0, 0))
    v = relu6(conv(v, cout, 48, 1, 1, (0, 0)))
    g.output(g.node("Flatten", [g.node("GlobalAveragePool", [v])], axis=1))
    return g, [r.standard_normal((batch, 3, height, width)).astype(dtype)]


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("pads", [(0, 0), (1, 2), (2, 0), (2, 2), (3, 1), (1, 3), (4, 4), (5, 3)], ids=str)
def test_any_depthwise_padding(pads, stride):
    """Paddings the block call takes and paddings it leaves to the three calls; images down to a pixel or two."""
    ops = Ops()
    for batch, height, width in ((128, 28, 31), (512, 9, 2), (512, 1, 12)):
        if height + 2 * pads[0] < 3 or width + 2 * pads[1] < 3:
            continue
        sizes = dict(cin=16, hidden=96, cout=24)
        if stride == 1 or height == 28:
            b = block(batch, 16, height, width, 96, 24, stride, *pads)
            assert ops.lib.dnnrtExecBlockApplies(ops.handle, C.byref(b)) == (max(pads) <= 2)
        build = lambda: small_net(batch, height, width, stride, pads, **sizes)  # noqa: E731
        ref, _ = run(lambda: as_fp32_graph(*build()), ORACLE_PATH, fusion=True)
        for mode in (compiler.MODE_OCCAMY, compiler.MODE_RESIDENT):
            got, _ = run(build, mode=mode, **FLAGS)
            close16(got[0], ref[0])
    ops.close()


def test_operands_at_any_address():
    """A block some of whose operands are the program's arguments, or whose result lies in the tensor that is returned: a
    run in place hands those over at the caller's addresses, which are aligned to an element only."""
    import torch
    batch, cin, hidden, cout, side = 32, 24, 144, 24, 28
    r = np.random.default_rng(5)
    half = lambda *s, f=1.0: (r.standard_normal(s) * f).astype(np.float16)  # noqa: E731
    values = {"x": half(batch, 3, side, side), "b1": half(hidden), "wd": half(hidden, 1, 3, 3, f=0.4), "bd": half(hidden), "b3": half(cout)}

    def build(args, dtype=np.float16):
        r2 = np.random.default_rng(6)
        g = compiler.Graph()
        c = lambda *s: g.constant((r2.standard_normal(s) * np.sqrt(2.0 / np.prod(s[1:]))).astype(np.float16).astype(dtype))  # noqa: E731
        v = {n: g.input(n, a.shape, dtype) if n == "x" or n in args else g.constant(a.astype(dtype)) for n, a in values.items()}
        clip = lambda t: g.node("Clip", [t, g.constant(np.array(0.0, dtype)), g.constant(np.array(6.0, dtype))])  # noqa: E731
        one = dict(kernel_shape=[1, 1], pads=[0] * 4, strides=[1, 1], group=1)
        t = clip(g.node("Conv", [v["x"], c(cin, 3, 3, 3), g.constant(np.zeros(cin, dtype))], kernel_shape=[3, 3], pads=[1] * 4, strides=[1, 1], group=1))
        t = clip(g.node("Conv", [t, c(hidden, cin, 1, 1), v["b1"]], **one))
        t = clip(g.node("Conv", [t, v["wd"], v["bd"]], kernel_shape=[3, 3], pads=[1] * 4, strides=[1, 1], group=hidden))
        t = g.node("Conv", [t, c(cout, hidden, 1, 1), v["b3"]], **one)
        t = clip(g.node("Conv", [t, c(40, cout, 1, 1), g.constant(np.zeros(40, dtype))], **one))
        g.output(g.node("Flatten", [g.node("GlobalAveragePool", [t])], axis=1))
        return g, [values[n] for n in g.input_shapes]

    def closing_layer(dtype=np.float16):  # a block's result is added to in place by the layer whose result is returned
        r2 = np.random.default_rng(7)
        g = compiler.Graph()
        c = lambda *s: g.constant((r2.standard_normal(s) * 0.2).astype(np.float16).astype(dtype))  # noqa: E731
        clip = lambda t: g.node("Clip", [t, g.constant(np.array(0.0, dtype)), g.constant(np.array(6.0, dtype))])  # noqa: E731
        conv = lambda t, ci, co, k=1, group=1: g.node("Conv", [t, c(co, ci // group, k, k), c(co)], kernel_shape=[k, k], pads=[k // 2] * 4, strides=[1, 1], group=group)  # noqa: E731
        y = clip(conv(g.input("x", (64, 16, 1, 1), dtype), 16, 24))
        y = conv(clip(conv(clip(conv(y, 24, 48)), 48, 48, 3, 48)), 48, 24)
        g.output(g.node("Add", [conv(y, 24, 24), y]))
        return g, [np.random.default_rng(8).standard_normal((64, 16, 1, 1)).astype(dtype)]

    ops = Ops()
    for b in (block(batch, cin, side, side, hidden, cout, 1, 1, 1), block(64, 24, 1, 1, 48, 24, 1, 1, 1)):
        assert ops.lib.dnnrtExecBlockApplies(ops.handle, C.byref(b))
    ops.close()
    nets = [lambda args=args: build(args) for args in ((), ("b1",), ("wd",), ("bd",), ("b3",), ("b1", "wd", "bd", "b3"))]
    for net in nets + [closing_layer]:
        ref, _ = run(lambda: as_fp32_graph(*net()), ORACLE_PATH, fusion=True)
        g, inputs = net()
        s = g.compile(inplace_residual=True, **FLAGS).session(compiler.MODE_RESIDENT)
        n = ref[0].size
        for off in (0, 1):
            bufs = [torch.zeros(a.size + 8, dtype=torch.float16, device="cuda") for a in inputs]
            for b, a in zip(bufs, inputs):
                b[off:off + a.size] = torch.from_numpy(a.reshape(-1)).cuda()
            out = torch.zeros(n + 8, dtype=torch.float16, device="cuda")
            for use_graph in (False, True, True):
                out.zero_()
                torch.cuda.synchronize()
                s.run_device([b.data_ptr() + 2 * off for b in bufs], [out.data_ptr() + 2 * off], use_graph=use_graph, in_place=True)
                s.sync()
                close16(out[off:off + n].cpu().numpy().reshape(ref[0].shape), ref[0])
        s.close()


def test_profile_and_variants_know_blocks():
    """MobileNetV2 with blocks: the session says which operations run in whose launch, times are those of launches, a
    block's work is its three convolutions' without the tensors between them, and variants are kept only for
    convolutions that have a call of their own."""
    import torch
    from occamy_amd import models
    g, inputs = models.mobilenet_v2(32, np.float16, seed=4, classes=100)
    p = g.compile(inplace_residual=True, **FLAGS)
    s = p.session(compiler.MODE_RESIDENT)
    plain = s.run(*inputs)[0]
    ops, prog = s.compute_ops(), p.compute_ops()
    assert [o[0] for o in ops] == [o[0] for o in prog]
    blocks = [i for i, o in enumerate(ops) if o[1] == "inverted_block" and o[4] == i]
    inner = [i for i, o in enumerate(ops) if o[4] != i]
    assert len(blocks) >= 5 and all(ops[i][4] in blocks and ops[i][2:4] == (0.0, 0.0) for i in inner) and len(inner) >= len(blocks)
    for b in blocks:
        members = [i for i, o in enumerate(ops) if o[4] == b]
        assert members == list(range(members[0], b + 1)) and len(members) in (2, 3)
        assert ops[b][2] == sum(prog[i][2] for i in members) and 0 < ops[b][3] < 0.6 * sum(prog[i][3] for i in members)
    for by_class in (False, True):
        for _ in range(2):
            ms = s.profile(inputs, by_class=by_class)
        assert all((m > 0) == (o[4] == i) for i, (m, o) in enumerate(zip(ms, ops)))
    rates = [ops[b][3] / ms[b] / 1e6 for b in blocks]  # GB/s
    assert max(rates) < 8000, rates
    np.testing.assert_array_equal(s.run(*inputs)[0], plain)
    s.set_algos([(3, 0)] * len(ops))
    kept = s.algos()
    assert all(kept[i] == (0, 0) for i in [*inner, *blocks]) and (3, 0) in kept
    close16(s.run(*inputs)[0], plain.astype(np.float32))
    s.set_algos([(0, 0)] * len(ops))
    np.testing.assert_array_equal(s.run(*inputs)[0], plain)
    changed = s.tune(inputs, reps=3)
    kept = s.algos()
    assert changed == sum(a != (0, 0) for a in kept) and all(kept[i] == (0, 0) for i in [*inner, *blocks])
    x = [torch.from_numpy(a).cuda() for a in inputs]
    out = torch.empty(plain.shape, dtype=torch.float16, device="cuda")
    for _ in range(2):
        s.run_device([t.data_ptr() for t in x], [out.data_ptr()], in_place=True)
        s.sync()
        close16(out.cpu().numpy(), plain.astype(np.float32))
    s.close()


def test_profile_knows_copies_that_are_not_launched():
    from occamy_amd import models
    g, inputs = models.alexnet(2, np.float32, image=224)
    s = g.compile(fusion=True, fuse_matmul_bias=True).session(compiler.MODE_RESIDENT)
    s.run(*inputs)
    ops, ms = s.compute_ops(), s.profile(inputs)
    elided = [i for i, o in enumerate(ops) if o[4] < 0]
    assert elided and all(ops[i][0] in ("dnn.flatten", "dnn.reshape", "dnn.squeeze", "dnn.unsqueeze") for i in elided)
    assert all((m > 0) == (o[4] == i) for i, (m, o) in enumerate(zip(ms, ops)))
    s.close()


@pytest.mark.parametrize("batch,height,width,stride,pads", [(1, 56, 57, 1, (1, 1)), (3, 31, 30, 2, (2, 1)), (4, 60, 5, 1, (2, 1)), (1, 28, 28, 1, (3, 3))], ids=str)
def test_fp32_blocks_in_programs(batch, height, width, stride, pads):
    """fp32 programs with a block in one launch (and one with a padding that it does not take), per inference and resident, against
    the oracle; every mode and a replay the same bits."""
    import torch
    flags = dict(FLAGS, channels_last=False)
    build = lambda: small_net(batch, height, width, stride, pads, dtype=np.float32)  # noqa: E731
    ref, _ = run(build, ORACLE_PATH, fusion=True)
    g, inputs = build()
    p = g.compile(**flags)
    s = p.session(compiler.MODE_RESIDENT)
    assert any(o[1] == "inverted_block" for o in s.compute_ops()) == (max(pads) <= 2)
    out = s.run(*inputs)[0]
    np.testing.assert_allclose(out, ref[0], rtol=1e-4, atol=1e-5 * float(np.abs(ref[0]).max()))
    x, y = torch.from_numpy(inputs[0]).cuda(), torch.empty(out.shape, device="cuda")
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        s.run_device([x.data_ptr()], [y.data_ptr()])
        s.sync()
        np.testing.assert_array_equal(y.cpu().numpy(), out)
    s.close()
    np.testing.assert_array_equal(run(build, mode=compiler.MODE_OCCAMY, **flags)[0][0], out)


@pytest.mark.parametrize("batch,side,sizes", [(1, 14, dict(cin=96, hidden=576, cout=96)), (10, 7, dict(cin=160, hidden=960, cout=160))], ids=str)
def test_fp16_blocks_in_parts_in_programs(batch, side, sizes):
    """Few tiles, so the hidden channels of a block go to several workgroups: close to the oracle, and the same bits run after run
    (the parts are added in order, and their counters are back at zero)."""
    build = lambda: small_net(batch, side, side, 1, (1, 1), **sizes)  # noqa: E731
    ref, _ = run(lambda: as_fp32_graph(*build()), ORACLE_PATH, fusion=True)
    g, inputs = build()
    s = g.compile(**FLAGS).session(compiler.MODE_RESIDENT)
    assert any(o[1] == "inverted_block" for o in s.compute_ops())
    out = s.run(*inputs)[0]
    close16(out, ref[0])
    for _ in range(4):
        np.testing.assert_array_equal(s.run(*inputs)[0], out)
    s.close()
