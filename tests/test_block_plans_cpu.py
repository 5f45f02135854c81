"""How the inverted residual block calls cut their problems, on the CPU: conv_f32_block.hip and conv_f16_block.hip compiled for the host, the
HIP runtime left out, their planners asked for a device of 256 compute units."""
import os
import shutil
import subprocess

import pytest

import test_gpu_ops
from test_untracked_reads import CSRC, HIPCC

COMMON = r"""
#include <cstdio>
#include <cstring>
extern "C" void **__hipRegisterFatBinary(const void *) { static void *none; return &none; }
extern "C" void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
extern "C" void __hipUnregisterFatBinary(void **) {}
using namespace dnnrt;
static dnnrtContext device() {
  dnnrtContext c{};
  c.num_cu = 256;
  c.splitk_partial_bytes = SPLITK_PARTIAL_BYTES;
  c.splitk_max_tiles = SPLITK_MAX_TILES;
  return c;
}
// n cin h w ch cout stride pad_h pad_w expand
static bool read(dnnrtExecBlock &k, int dtype, int format) {
  long long v[10];
  for (long long &x : v) if (scanf("%lld", &x) != 1) return false;
  k = dnnrtExecBlock{};
  k.n = v[0]; k.cin = v[1]; k.h = v[2]; k.w = v[3]; k.ch = v[4]; k.cout = v[5]; k.stride = v[6]; k.pad_h = v[7]; k.pad_w = v[8]; k.expand = (int)v[9];
  k.r = k.s = 3;
  k.p = (k.h + 2 * k.pad_h - 3) / k.stride + 1;
  k.q = (k.w + 2 * k.pad_w - 3) / k.stride + 1;
  k.act1 = k.actd = DNNRT_ACT_CLIPPED_RELU;
  k.act = DNNRT_ACT_IDENTITY;
  k.coef1 = k.coefd = 6.f;
  k.dtype = dtype;
  k.format = format;
  return true;
}
"""

F32 = r"""
#include "conv_f32_block.hip"
namespace dnnrt {
const dnnrtBlockCut *find_block_cut(const dnnrtContext *, const int64_t (&)[11]) { return nullptr; }
void keep_block_cut(const dnnrtContext *, const int64_t (&)[11], dnnrtBlockCut) {}
}
""" + COMMON + r"""
// The last float of LDS that an expansion of the kernel reads, its loops as they stand there: chunks of KG steps up to KC, blocks of
// 16 pixels, two at a time while more than one is left.
static int last_read(int KC, int XS, int NP) {
  const int KG = block32_kg(KC);
  int last = 0;
  auto expand = [&](int p, int blocks) {
    auto read = [&](int k0) {
      for (int k = 0; k < KG; k++)
        for (int l4 = 0; l4 < 4; l4++) last = std::max(last, 2 * l4 * XS + p + 15 + (8 * ((k0 + k) >> 1) + (k & 1)) * XS + 16 * (blocks - 1));
    };
    read(0);
    for (int k0 = 0; k0 < KC; k0 += KG)
      if (k0 + KG < KC) read(k0 + KG);
  };
  int p = 0;
  for (; p + 16 < NP; p += 32) expand(p, 2);
  if (p < NP) expand(p, 1);
  return last;
}
int main() {
  const dnnrtContext ctx = device();
  dnnrtExecBlock k;
  while (read(k, DNNRT_F32, DNNRT_NCHW)) {
    BlockF32Args a{}, t{};
    BlockF32Cut c{}, u{};
    if (!plan_block_f32(&ctx, k, false, a, c)) { printf("refused\n"); continue; }
    int cuts = 0, outside = 0;
    for (int nb = 1; nb <= 2; nb++)  // every cut that the planner may pick, on this device or another
      for (int qw = 1; qw <= 4 * nb; qw++)
        for (int G = 4; G <= 8; G += 4)
          for (int splits = 1; splits <= 32; splits++)
            if (cut_block_f32(&ctx, k, nb, qw, G, splits, t, u)) {
              cuts++;
              if (u.kc > 0 && 4 * last_read(u.kc, block32_xs((int)k.stride, nb), u.np) + 4 > u.lds) outside++;
            }
    printf("%d %d %d %d %d %d %d\n", c.kc, c.mb, c.nb, c.G, a.splits, cuts, outside);
  }
}
"""

F16 = r"""
#include "conv_f16_block.hip"
""" + COMMON + r"""
int main() {
  dnnrtExecBlock k;
  while (read(k, DNNRT_F16, DNNRT_NHWC)) {
    const dnnrtContext ctx = device();
    BlockF16Args a{};
    int kc, gy, g, parts;
    if (!plan_block_f16(&ctx, k, false, a, kc, gy, g, parts)) { printf("refused\n"); continue; }
    printf("%d %d %d %d\n", kc, gy, g, parts);
  }
}
"""


def _planner(tmp_path_factory, name, source):
    if not os.path.exists(HIPCC) or not shutil.which("g++"):
        pytest.skip("no compiler")
    at = tmp_path_factory.mktemp(name)
    (at / "plan.cpp").write_text(source)
    subprocess.check_call([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-fPIC", "-I", CSRC, "-c", "-o", str(at / "plan.o"), str(at / "plan.cpp")],
                          stderr=subprocess.DEVNULL)
    subprocess.check_call(["g++", "-o", str(at / "plan"), str(at / "plan.o"), "-Wl,--unresolved-symbols=ignore-all"])

    def ask(problems):
        text = "".join(" ".join(str(int(v)) for v in p) + "\n" for p in problems)
        lines = subprocess.run([str(at / "plan")], input=text, capture_output=True, text=True, check=True).stdout.split("\n")[:-1]
        assert len(lines) == len(problems)
        return [None if line == "refused" else tuple(int(v) for v in line.split()) for line in lines]
    return ask


@pytest.fixture(scope="module")
def f32(tmp_path_factory):
    return _planner(tmp_path_factory, "f32", F32)


@pytest.fixture(scope="module")
def f16(tmp_path_factory):
    return _planner(tmp_path_factory, "f16", F16)


def test_expansions_read_inside_the_workgroups_lds(f32):
    """Whatever cut is taken, and also where the block has fewer k-steps than the kernel was made for: few input channels and many output ones."""
    problems = [(n, cin, side, side + 1, 96, cout, stride, 1, 1, 1) for n in (1, 16) for cin in (8, 16, 32, 40, 64, 72, 96, 104, 160) for side in (5, 14, 56)
                for cout in (8, 40, 96, 104, 160, 328) for stride in (1, 2)]
    plans = f32(problems)
    assert all(p is not None and p[5] > 0 for p in plans)
    assert not [q for q, p in zip(problems, plans) if p[6]]


def _cases(name):
    mark, = (m for m in getattr(test_gpu_ops, name).pytestmark if m.name == "parametrize")
    return mark.args[1]


def test_the_fp32_tests_reach_every_kernel(f32):
    """The cases of the tests on the GPU are for the kernels that the planner's estimate sends them to: if it is fitted anew, they may need others."""
    cases = _cases("test_inverted_residual_block_fp32") + _cases("test_inverted_residual_block_fp32_kernels")
    plans = f32([(n, cin, h, w, ch, cout, stride, *pads, expand) for n, cin, h, w, ch, cout, stride, pads, expand, _, _ in cases])
    got = {(c[6], p[0], p[2], p[3], p[4] > 1) for c, p in zip(cases, plans)}  # stride, k-steps, blocks of pixels, wavefronts, in parts
    want = {(s, kc, nb, g, parts) for s in (1, 2) for kc in (24, 40) for nb in (1, 2) for g in (4, 8) for parts in (False, True)}
    want -= {(2, 40, 2, 8, False), (2, 40, 2, 8, True)}  # no room for eight wavefronts, or never the fastest
    want |= {(s, 8, 2, 4, parts) for s in (1, 2) for parts in (False, True)} - {(2, 8, 2, 4, False)} | {(2, 8, 2, 8, False), (1, 0, 2, 4, False), (2, 0, 2, 4, False)}
    assert want <= got, sorted(want - got)


def test_the_fp16_tests_reach_every_kernel(f16):
    cases = [c for name in ("", "_in_parts", "_kernels") for c in _cases("test_inverted_residual_block_fp16" + name)]
    plans = f16([(n, cin, h, w, ch, cout, stride, 1, 1, expand) for n, cin, h, w, ch, cout, stride, expand, _ in cases])
    got = {(c[6], p[0], p[3] > 1) for c, p in zip(cases, plans)}  # stride, steps of input channels, in parts
    want = {(s, kc, parts) for s in (1, 2) for kc in (0, 1, 2, 4, 6, 10) for parts in (False, True)}
    assert want <= got, sorted(want - got)
    in_parts = len(_cases("test_inverted_residual_block_fp16"))
    assert all(p[3] > 1 for p in plans[in_parts:in_parts + len(_cases("test_inverted_residual_block_fp16_in_parts"))])
