"""Which inverted residual blocks a session takes, on the CPU: the oracle runtime, claiming to be a device runtime whose block call takes
every fp32 block, makes it out of the three convolutions and counts it."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import graph_eval
from helpers import ROOT
from occamy_amd import compiler

SHIM = r"""
#define dnnrtIsHostBackend dnnrt_oracle_is_host_backend
#define dnnrtSetFilterLayout dnnrt_oracle_set_filter_layout
#define dnnrtConvBiasActiv dnnrt_oracle_conv_bias_activ
#include "%(oracle)s"
#undef dnnrtIsHostBackend
#undef dnnrtSetFilterLayout
#undef dnnrtConvBiasActiv
#include "%(exec)s"
static int layout, blocks_run;
int blocks_so_far(void) { return blocks_run; }
int32_t dnnrtIsHostBackend(void) { return 0; }
int32_t dnnrtSetFilterLayout(dnnrtHandle_t h, int32_t l) { (void)h; layout = l; return 0; }
int32_t dnnrtExecFenceCreate(void **event) { return dnnrtEventCreate(event); }
int32_t dnnrtExecStreamWait(dnnrtStream_t stream, void *event) { (void)stream; (void)event; return 0; }
int32_t dnnrtExecUpload(void *dst, const void *src, int64_t bytes, dnnrtStream_t stream) { (void)stream; memcpy(dst, src, (size_t)bytes); return 0; }
void *dnnrtConvBiasActiv(dnnrtHandle_t h, const void *X, const int64_t *dX, const void *W, const int64_t *dW, const void *B, const int64_t *dB, void *ws, int64_t wsBytes,
                         int64_t algo, int64_t group, const int64_t *pads, const int64_t *strides, int64_t act, void *Y, int32_t dtype) {
  const int64_t K = dW[0], CRS = dW[1] * dW[2] * dW[3];
  if (layout == DNNRT_FILTER_KCRS) return dnnrt_oracle_conv_bias_activ(h, X, dX, W, dW, B, dB, ws, wsBytes, algo, group, pads, strides, act, Y, dtype);
  float *rows = malloc((size_t)(K * CRS) * 4);
  for (int64_t k = 0; k < K; k++)
    for (int64_t j = 0; j < CRS; j++) rows[k * CRS + j] = ((const float *)W)[j * K + k];
  void *r = dnnrt_oracle_conv_bias_activ(h, X, dX, rows, dW, B, dB, ws, wsBytes, algo, group, pads, strides, act, Y, dtype);
  free(rows);
  return r;
}
/* the layout that the block call reads its 1x1 filters in: as they come */
void dnnrtExecBlockFilter(void *dst, const void *src, int64_t rows, int64_t cols) { memcpy(dst, src, (size_t)(rows * cols) * 4); }
void dnnrtExecBlockFilterF32(void *dst, const void *src, int64_t rows, int64_t cols) { memcpy(dst, src, (size_t)(rows * cols) * 4); }
int32_t dnnrtExecBlockApplies(dnnrtHandle_t h, const dnnrtExecBlock *k) { (void)h; return k->dtype == DNNRT_F32 && k->expand && !k->z; }
int32_t dnnrtExecRunBlock(dnnrtHandle_t h, const dnnrtExecBlock *k) {
  float *wide = malloc((size_t)(k->n * k->ch * k->h * k->w) * 4), *mid = malloc((size_t)(k->n * k->ch * k->p * k->q) * 4);
  const int64_t none[2] = {0, 0}, one[2] = {1, 1}, pads[2] = {k->pad_h, k->pad_w}, strides[2] = {k->stride, k->stride};
  const int64_t dx[4] = {k->n, k->cin, k->h, k->w}, dwide[4] = {k->n, k->ch, k->h, k->w}, dmid[4] = {k->n, k->ch, k->p, k->q};
  const int64_t d1[4] = {k->ch, k->cin, 1, 1}, dd[4] = {k->ch, 1, k->r, k->s}, d3[4] = {k->cout, k->ch, 1, 1}, bh[4] = {1, k->ch, 1, 1}, bo[4] = {1, k->cout, 1, 1};
  const int was = layout;
  layout = DNNRT_FILTER_CRSK;
  const int ok = dnnrtConvBiasActiv(h, k->x, dx, k->w1, d1, k->b1, bh, 0, 0, 0, 1, none, one, k->act1, wide, k->dtype) &&
                 dnnrtConvBiasActiv(h, wide, dwide, k->wd, dd, k->bd, bh, 0, 0, 0, k->ch, pads, strides, k->actd, mid, k->dtype) &&
                 dnnrtConvBiasActiv(h, mid, dmid, k->w3, d3, k->b3, bo, 0, 0, 0, 1, none, one, k->act, k->y, k->dtype);
  layout = was;
  free(wide);
  free(mid);
  blocks_run++;
  return !ok;
}
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("no host compiler")
    at = tmp_path_factory.mktemp("blocks")
    (at / "runtime.c").write_text(SHIM % {"oracle": os.path.join(ROOT, "oracle", "dnnrt_oracle.c"), "exec": os.path.join(ROOT, "occamy_amd", "csrc", "dnnrt_exec.h")})
    subprocess.check_call(["gcc", "-O1", "-fPIC", "-shared", "-std=gnu11", "-ffp-contract=off", "-fopenmp", "-I", os.path.join(ROOT, "oracle"),
                           "-o", str(at / "runtime.so"), str(at / "runtime.c"), "-lm"])
    return str(at / "runtime.so")


def _net(side, blocks, last):
    """A chain of blocks (input channels, hidden ones, output ones), each on a map of half the side, and a 3x3 layer of `last` channels."""
    r = np.random.default_rng(11)
    g = compiler.Graph()

    def conv(v, cin, cout, k, stride, group=1, relu=True):
        w = (r.standard_normal((cout, cin // group, k, k)) * np.sqrt(2.0 / (cin // group * k * k))).astype(np.float32)
        v = g.node("Conv", [v, g.constant(w), g.constant(r.uniform(-0.3, 0.3, cout).astype(np.float32))], kernel_shape=[k, k], pads=[k // 2] * 4,
                   strides=[stride, stride], group=group)
        return g.node("Relu", [v]) if relu else v

    x = v = g.input("x", (1, 8, side, side))
    v, channels = conv(v, 8, blocks[0][0], 3, 1), blocks[0][0]
    for cin, hidden, cout in blocks:
        assert cin == channels
        v = conv(v, cin, hidden, 1, 1)
        v = conv(v, hidden, hidden, 3, 2, hidden)
        v, channels = conv(v, hidden, cout, 1, 1, relu=False), cout
    g.output(conv(v, channels, last, 3, 1))
    return g, [r.standard_normal((1, 8, side, side)).astype(np.float32)]


SMALL, NEXT, WIDE = (16, 48, 24), (24, 48, 160), (160, 960, 160)


@pytest.mark.parametrize("net,taken", [
    ((32, [SMALL], 16), 1),
    ((48, [SMALL, NEXT, WIDE], 384), 3),        # the last layer's filter makes the pool large enough
    ((48, [SMALL, NEXT, WIDE], 16), 2),         # ... and here not: 1.31 MB where the filters of the widest block alone are 1.26
    ((32, [SMALL, NEXT, WIDE, WIDE], 192), 2),  # two that do not fit
], ids=str)
def test_a_block_whose_filters_do_not_fit_goes_alone(runtime, net, taken):
    """The same blocks in both modes: those that a per-inference program has with its constants uploaded ahead."""
    g, inputs = _net(*net)
    want = graph_eval.evaluate(g, inputs)[0]
    lib = C.CDLL(runtime)
    p = g.compile(fusion=True, fuse_activations=True, compact_pool=True)
    outs = []
    for mode in (compiler.MODE_OCCAMY, compiler.MODE_RESIDENT):
        s = p.session(mode, runtime_library=runtime)
        for _ in range(2):
            before = lib.blocks_so_far()
            outs.append(s.run(*inputs)[0])
            assert lib.blocks_so_far() - before == taken, mode
            np.testing.assert_allclose(outs[-1], want, rtol=1e-3, atol=1e-4 * float(np.abs(want).max()))
        s.close()
    for o in outs[1:]:
        np.testing.assert_array_equal(o, outs[0])
