"""Per-inference sessions that upload their constants ahead of the operations, on the CPU: the oracle runtime, claiming
to be a device runtime and given the entry points that the executor looks for, does every upload at the moment it is
issued.  Bytes that the plan gives to a constant while something that lies there is still to be read are then wrong in
the results, every time."""
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
#include "%(oracle)s"
#undef dnnrtIsHostBackend
static long n_uploads;
long uploads_issued(void) { return n_uploads; }
int32_t dnnrtIsHostBackend(void) { return 0; }
int32_t dnnrtExecFenceCreate(void **event) { return dnnrtEventCreate(event); }
int32_t dnnrtExecStreamWait(dnnrtStream_t stream, void *event) { (void)stream; (void)event; return 0; }
int32_t dnnrtExecUpload(void *dst, const void *src, int64_t bytes, dnnrtStream_t stream) {
  (void)stream;
  n_uploads++;
  memcpy(dst, src, (size_t)bytes);
  return 0;
}
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("no host compiler")
    at = tmp_path_factory.mktemp("uploading")
    (at / "runtime.c").write_text(SHIM % {"oracle": os.path.join(ROOT, "oracle", "dnnrt_oracle.c")})
    subprocess.check_call(["gcc", "-O1", "-fPIC", "-shared", "-std=c11", "-ffp-contract=off", "-fopenmp", "-I", os.path.join(ROOT, "oracle"),
                           "-o", str(at / "runtime.so"), str(at / "runtime.c"), "-lm"])
    return str(at / "runtime.so")


def _graph(kinds, returned):
    """A chain of products, and a constant that is reshaped in front of it and added behind it."""
    r = np.random.default_rng(3)
    g = compiler.Graph()
    side = 32
    x = g.input("x", (side, side))
    late = g.constant(r.standard_normal((1, side * side)).astype(np.float32))
    shape = g.constant(np.array([side, side], np.int64))
    for kind in kinds:
        if kind == "reshape":
            late = g.node("Reshape", [late, shape])
        elif kind == "unsqueeze":
            late = g.node("Unsqueeze", [late], axes=[0])
        else:
            late = g.node("Squeeze", [late], axes=[0])
    h = x
    for _ in range(6):
        w = g.constant((r.standard_normal((side, side)) / 6).astype(np.float32))
        h = g.node("Relu", [g.node("MatMul", [h, w])])
    g.output(g.node("Add", [h, late]))
    if returned:
        g.output(late)
    return g, [r.standard_normal((side, side)).astype(np.float32)]


@pytest.mark.parametrize("returned", [False, True])
@pytest.mark.parametrize("kinds", [("reshape",), ("reshape", "unsqueeze", "squeeze"), ("unsqueeze", "squeeze", "reshape")])
@pytest.mark.parametrize("flags", [dict(), dict(alias_copies=True), dict(alias_copies=True, compact_pool=True), dict(alias_copies=True, fuse_matmul_bias=True)])
def test_a_constant_read_through_copies_that_are_not_made_stays_until_its_last_reader(runtime, kinds, flags, returned):
    g, inputs = _graph(kinds, returned)
    want = graph_eval.evaluate(g, inputs)
    s = g.compile(**flags).session(compiler.MODE_OCCAMY, runtime_library=runtime)
    uploads = C.CDLL(runtime).uploads_issued
    before = uploads()
    for _ in range(2):
        for got, ref in zip(s.run(*inputs), want):
            np.testing.assert_allclose(got, ref, rtol=1e-4, atol=1e-4)
    assert uploads() > before  # the plan under test is the one that ran
    s.close()
