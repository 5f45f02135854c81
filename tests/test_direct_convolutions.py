"""Which `algo` operand the executor gives a convolution: the oracle runtime, claiming to be a device runtime, notes it."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import graph_eval
from helpers import ROOT
from occamy_amd import _abi, compiler

NOTING = r"""
#define dnnrtIsHostBackend dnnrt_oracle_is_host_backend
#define dnnrtConvBiasActiv dnnrt_oracle_conv_bias_activ
#define dnnrtSetFilterLayout dnnrt_oracle_set_filter_layout
#include "%(oracle)s"
#undef dnnrtIsHostBackend
#undef dnnrtConvBiasActiv
#undef dnnrtSetFilterLayout
static int64_t seen[64];
static int n_seen, crsk;
int algos_seen(int64_t *out) { int n = n_seen; for (int i = 0; i < n; i++) out[i] = seen[i]; n_seen = 0; return n; }
int32_t dnnrtIsHostBackend(void) { return 0; }
int32_t dnnrtSetFilterLayout(dnnrtHandle_t h, int32_t layout) { (void)h; crsk = layout == DNNRT_FILTER_CRSK; return 0; }
void *dnnrtConvBiasActiv(dnnrtHandle_t h, const void *X, const int64_t *dX, const void *W, const int64_t *dW, const void *B, const int64_t *dB,
                         void *ws, int64_t wsBytes, int64_t algo, int64_t group, const int64_t *pads, const int64_t *strides, int64_t activ, void *Y, int32_t dtype) {
  if (n_seen < 64) seen[n_seen++] = algo;
  int64_t K = dW[0], J = dW[1] * dW[2] * dW[3];
  float *w = malloc((size_t)(K * J) * sizeof(float));
  for (int64_t k = 0; k < K; k++)
    for (int64_t j = 0; j < J; j++) w[k * J + j] = crsk ? ((const float *)W)[j * K + k] : ((const float *)W)[k * J + j];
  void *r = dnnrt_oracle_conv_bias_activ(h, X, dX, w, dW, B, dB, ws, wsBytes, algo, group, pads, strides, activ, Y, dtype);
  free(w);
  return r;
}
"""


@pytest.fixture(scope="module")
def noting(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("no host compiler")
    at = tmp_path_factory.mktemp("noting")
    (at / "runtime.c").write_text(NOTING % {"oracle": os.path.join(ROOT, "oracle", "dnnrt_oracle.c")})
    subprocess.check_call(["gcc", "-O1", "-fPIC", "-shared", "-std=c11", "-ffp-contract=off", "-fopenmp", "-I", os.path.join(ROOT, "oracle"),
                           "-o", str(at / "runtime.so"), str(at / "runtime.c"), "-lm"])
    return str(at / "runtime.so")


@pytest.mark.parametrize("mode", [compiler.MODE_OCCAMY, compiler.MODE_RESIDENT])
@pytest.mark.parametrize("asked", [False, True])
def test_direct_sums_where_asked_for_or_filters_are_mostly_zero(noting, mode, asked):
    """Four convolutions: dense 3x3, 3x3 with half its values zero, 3x3 with more, and a sparse 1x1."""
    r = np.random.default_rng(5)
    g = compiler.Graph()
    y = g.input("x", (1, 4, 9, 9))
    for k, zeros in ((3, 0), (3, 72), (3, 73), (1, 14)):
        w = r.standard_normal((4, 4, k, k)).astype(np.float32) / k
        w.reshape(-1)[:zeros] = 0
        conv = g.node("Conv", [y, g.constant(w), g.constant(r.standard_normal(4).astype(np.float32))], kernel_shape=[k, k], pads=[k // 2] * 4, strides=[1, 1], group=1)
        y = g.node("Relu", [conv])
    g.output(y)
    inputs = [r.standard_normal((1, 4, 9, 9)).astype(np.float32)]
    want = graph_eval.evaluate(g, inputs)[0]
    s = g.compile(fusion=True, direct_convolutions=asked).session(mode, runtime_library=noting)
    seen, L = (C.c_int64 * 64)(), C.CDLL(noting)
    L.algos_seen(seen)
    np.testing.assert_allclose(s.run(*inputs)[0], want, rtol=1e-4, atol=1e-5)
    n = L.algos_seen(seen)
    s.close()
    direct = _abi.CONV_ALGO_DIRECT
    assert list(seen[:n]) == ([direct] * 4 if asked else [1, 1, direct, 1])
