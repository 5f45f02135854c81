"""Parity of the gfx950 library with the CPU oracle, operator by operator,
through the C ABI on the same seeded inputs.

Bars: bit-exact for copies, index work, max, clip, negate, ReLU, two-operand
add/mul, reciprocal and sqrt (no reassociation is involved); fp32 reductions
and transcendental functions within rtol 1e-4 / atol 1e-5 of the oracle
(which accumulates in double); fp16 storage within rtol 2e-2.
"""
import ctypes as C

import numpy as np
import pytest

import opcases as oc
from helpers import GpuBackend, OracleBackend, rng
from occamy_amd import _abi

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-4, 1e-5


@pytest.fixture(scope="module")
def gpu():
    return GpuBackend()


@pytest.fixture(scope="module")
def cpu():
    return OracleBackend()


def close(got, ref, rtol=RTOL, atol=ATOL):
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)


# ---- convolution ----------------------------------------------------------------

CONV_CASES = [
    # N, C, H, W, K, R, S, stride, pad, group
    (1, 64, 56, 56, 64, 3, 3, 1, 1, 1),     # the single-conv configuration (Kaiming-uniform below)
    (1, 3, 224, 224, 64, 7, 7, 2, 3, 1),    # ResNet stem
    (1, 64, 56, 56, 256, 1, 1, 1, 0, 1),
    (1, 256, 56, 56, 512, 1, 1, 2, 0, 1),   # strided 1x1 downsample
    (1, 128, 56, 56, 128, 3, 3, 2, 1, 1),
    (1, 512, 7, 7, 512, 3, 3, 1, 1, 1),     # 49 pixels: ragged column tile
    (1, 2048, 7, 7, 512, 1, 1, 1, 0, 1),
    (2, 16, 9, 11, 24, 3, 3, 1, 1, 1),      # batch > 1, ragged everything
    (3, 5, 8, 8, 7, 2, 3, 1, 0, 1),         # generic filter size, odd channels
    (1, 8, 12, 12, 16, 5, 5, 1, 2, 1),
    (1, 16, 10, 10, 32, 3, 3, 1, 1, 4),     # grouped
    (1, 32, 112, 112, 32, 3, 3, 1, 1, 32),  # MobileNetV2 depthwise
    (1, 96, 112, 112, 96, 3, 3, 2, 1, 96),  # depthwise stride 2
    (2, 6, 7, 7, 12, 3, 3, 1, 1, 6),        # depthwise with channel multiplier 2
    (1, 1, 5, 5, 1, 3, 3, 1, 1, 1),         # smallest
    (1, 64, 96, 80, 3, 3, 3, 1, 1, 1),      # image-producing last layer: three output channels
    (2, 16, 21, 17, 4, 3, 3, 2, 1, 1),      # four output channels, stride 2
    (2, 24, 9, 9, 2, 1, 1, 1, 0, 1),        # two output channels, 1x1
    # 3x3 layers that fill the chip (the LDS-tiled 3x3 kernel): 128x128 tiles with an odd channel count and
    # ragged rows; 64x64 tiles, stride 2, no padding; groups
    (1, 5, 190, 180, 130, 3, 3, 1, 1, 1),
    (2, 8, 260, 130, 64, 3, 3, 2, 0, 1),
    (1, 8, 182, 182, 256, 3, 3, 1, 1, 2),
]


@pytest.mark.parametrize("case", CONV_CASES, ids=lambda c: "x".join(map(str, c)))
def test_conv_f32(gpu, cpu, case):
    N, C, H, W, K, R, S, st, pd, g = case
    r = rng(hash(case) % (2 ** 31))
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    bound = np.sqrt(6.0 / (C // g * R * S))
    w = r.uniform(-bound, bound, (K, C // g, R, S)).astype(np.float32)
    b = r.uniform(-0.1, 0.1, K).astype(np.float32)
    args = ((pd, pd), (st, st), g)
    close(oc.conv(gpu, x, w, None, *args), oc.conv(cpu, x, w, None, *args))
    ref = oc.conv(cpu, x, w, b, *args, _abi.ACT_RELU)
    got = oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU)
    close(got, ref)
    assert (got >= 0).all()
    close(oc.conv(gpu, x, w, b, *args, _abi.ACT_IDENTITY), oc.conv(cpu, x, w, b, *args, _abi.ACT_IDENTITY))
    # the same filter handed over C,R,S,K: same kernels' K,C,R,S result up to
    # the summation order of the tile shapes each layout selects
    close(oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=True), ref)
    close(oc.conv(gpu, x, w, None, *args, crsk=True), oc.conv(cpu, x, w, None, *args))
    # residual operand: relu((conv + b) + z); bit-equal to this library's own
    # conv -> add -> relu chain, which forms the same sums in the same order
    z = r.standard_normal(ref.shape).astype(np.float32)
    fused = oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, z=z)
    close(fused, oc.conv(cpu, x, w, b, *args, _abi.ACT_RELU, z=z))
    lin = oc.conv(gpu, x, w, b, *args, _abi.ACT_IDENTITY)
    np.testing.assert_array_equal(fused, oc.unary(gpu, "relu", oc.tensor_op(gpu, _abi.OP_ADD, lin, z)))
    close(oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=True, z=z), fused)
    # the result written over the residual operand (Z == Y): the same bits, from the kernels of either filter layout
    np.testing.assert_array_equal(oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, z=z, inplace=True), fused)
    np.testing.assert_array_equal(oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=True, z=z, inplace=True),
                                  oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=True, z=z))
    np.testing.assert_array_equal(oc.conv(cpu, x, w, b, *args, _abi.ACT_RELU, z=z, inplace=True), oc.conv(cpu, x, w, b, *args, _abi.ACT_RELU, z=z))


# N, C, H, W, K, stride, pad: 3x3 depthwise layers with outputs enough for strips of four rows (N K ceil(P/4) Q from
# 2048 threads per compute unit on): rows that leave one, two or three over, one row, no padding and more than needed,
# two results per channel, stride 2 with even and odd sides, the last strip and image together.
DW_ROWS_CASES = [(4, 96, 113, 111, 96, 1, 1), (3, 160, 78, 79, 160, 1, 0), (2, 64, 119, 121, 128, 1, 2), (600, 64, 1, 14, 64, 1, 1),
                 (6, 64, 150, 149, 64, 2, 1), (4, 96, 151, 152, 96, 2, 0), (257, 576, 14, 14, 576, 2, 1)]


@pytest.mark.parametrize("case", DW_ROWS_CASES, ids=lambda c: "x".join(map(str, c)))
def test_conv_f32_depthwise_strips(gpu, cpu, case):
    """Depthwise layers computed in strips of rows against the oracle, both filter layouts, with a residual and over it."""
    N, C, H, W, K, st, pd = case
    r = rng(sum(case))
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((K, 1, 3, 3)) / 3).astype(np.float32)
    b = r.uniform(-0.3, 0.3, K).astype(np.float32)
    args = ((pd, pd), (st, st), C)
    lin = oc.conv(cpu, x, w, b, *args, _abi.ACT_IDENTITY)
    close(oc.conv(gpu, x, w, None, *args), lin - b[:, None, None], atol=1e-5)
    z = r.standard_normal(lin.shape).astype(np.float32)
    for crsk in (False, True):
        gotz = oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=crsk, z=z)
        close(gotz, np.maximum(lin + z, 0))
        np.testing.assert_array_equal(oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=crsk, z=z, inplace=True), gotz)


def random_conv_cases(seed, count, f16):
    """Seeded shapes around the kernels' boundaries: channel counts on both sides of the multiples of 8, 32 and
    64 the fast paths ask for, filter sizes 1 / 2 / 3 / 5 / 7, strides 1-3 (different along the two axes now and
    then), padding up to the filter's half and beyond, a few hundred to a few thousand output pixels."""
    r = np.random.default_rng(seed)
    cases = []
    while len(cases) < count:
        R, S = (int(v) for v in r.choice([1, 1, 2, 3, 3, 3, 5, 7], 2)) if r.random() < 0.3 else (int(r.choice([1, 3, 3, 5])),) * 2
        grp = int(r.choice([1, 1, 1, 1, 2, 4])) if not f16 or r.random() < 0.3 else 1
        cg = int(r.choice([1, 3, 8, 16, 31, 32, 33, 64, 96, 128, 160, 192, 256])) if f16 else int(r.choice([1, 2, 3, 5, 8, 16, 24, 33, 64, 100]))
        kg = int(r.choice([1, 2, 8, 24, 40, 64, 72, 128, 136, 200, 256])) if f16 else int(r.choice([1, 2, 3, 4, 7, 16, 33, 64, 130]))
        if grp > 1:
            cg, kg = min(cg, 32), min(kg, 40)
        N, H, W = int(r.integers(1, 5)), int(r.integers(1, 30)), int(r.integers(1, 30))
        sh, sw = (int(r.integers(1, 4)),) * 2 if r.random() < 0.8 else (int(r.integers(1, 4)), int(r.integers(1, 4)))
        ph, pw = int(r.integers(0, R // 2 + 2)), int(r.integers(0, S // 2 + 2))
        P, Q = (H + 2 * ph - R) // sh + 1, (W + 2 * pw - S) // sw + 1
        if P < 1 or Q < 1 or H + 2 * ph < R or W + 2 * pw < S or N * cg * grp * H * W > 2_000_000 or N * kg * grp * P * Q > 2_000_000:
            continue
        cases.append((N, cg * grp, H, W, kg * grp, R, S, sh, sw, ph, pw, grp))
    return cases


def test_conv_f32_random_shapes(gpu, cpu):
    """120 seeded shapes through dnnrtConvBiasActiv / dnnrtConvBiasAddActiv on fp32 N,C,H,W tensors against the
    oracle (rtol 1e-4, atol 1e-5), with both filter layouts, each activation mode once in a while, and the residual
    form also written over its residual operand."""
    for i, (N, C, H, W, K, R, S, sh, sw, ph, pw, grp) in enumerate(random_conv_cases(2024, 120, False)):
        r = rng(1000 + i)
        x = r.standard_normal((N, C, H, W)).astype(np.float32)
        w = (r.standard_normal((K, C // grp, R, S)) * np.sqrt(2.0 / (C // grp * R * S))).astype(np.float32)
        b = r.uniform(-0.3, 0.3, K).astype(np.float32)
        activ, coef = [(_abi.ACT_RELU, None), (_abi.ACT_IDENTITY, None), (_abi.ACT_CLIPPED_RELU, 0.7), (_abi.ACT_LEAKY_RELU, 0.1)][i % 4]
        what = f"case {i}: x {x.shape} w {w.shape} strides {(sh, sw)} pads {(ph, pw)} group {grp} act {activ}"
        ref = oc.conv(cpu, x, w, b, (ph, pw), (sh, sw), grp, activ, coef=coef)
        for crsk in (False, True):
            got = oc.conv(gpu, x, w, b, (ph, pw), (sh, sw), grp, activ, crsk=crsk, coef=coef)
            np.testing.assert_allclose(got, ref, rtol=RTOL, atol=ATOL, err_msg=what)
        z = r.standard_normal(ref.shape).astype(np.float32)
        refz = oc.conv(cpu, x, w, b, (ph, pw), (sh, sw), grp, activ, z=z, coef=coef)
        gotz = oc.conv(gpu, x, w, b, (ph, pw), (sh, sw), grp, activ, z=z, coef=coef)
        np.testing.assert_allclose(gotz, refz, rtol=RTOL, atol=ATOL, err_msg=what + " + z")
        np.testing.assert_array_equal(oc.conv(gpu, x, w, b, (ph, pw), (sh, sw), grp, activ, z=z, coef=coef, inplace=True), gotz, err_msg=what + " in place")


# N, C, H, W, K, R, stride, pad: the tiles whose operands go straight into LDS (C,R,S,K filters, problems that fill the
# chip).  K off the tile and off multiples of four, pixels per image odd (pairs of pixels that straddle two images) and
# in fours (16-byte loads), channels fewer than a step, not a multiple of a step, not a multiple of four, filters of one
# tap with padding, 16 to 32 filters, tiles left over and split along the reduction, one reduction step.
DMA_F32_CASES = [(3, 20, 75, 75, 66, 3, 1, 1), (2, 64, 90, 117, 130, 3, 1, 1), (4, 4, 80, 80, 64, 3, 2, 1), (1, 12, 130, 131, 70, 5, 1, 2),
                 (2, 3, 190, 190, 64, 7, 2, 3), (1, 5, 150, 120, 64, 4, 1, 0), (4, 64, 56, 56, 128, 1, 1, 0), (3, 36, 75, 75, 96, 1, 1, 0),
                 (2, 30, 75, 75, 132, 1, 1, 1), (8, 16, 32, 32, 256, 1, 2, 0), (3, 256, 38, 38, 24, 3, 1, 1), (3, 512, 19, 19, 486, 3, 1, 1),
                 (16, 256, 14, 14, 256, 3, 1, 1), (33, 8, 24, 24, 64, 1, 1, 0)]


@pytest.mark.parametrize("case", DMA_F32_CASES, ids=lambda c: "x".join(map(str, c)))
def test_conv_f32_direct_to_lds_tiles(gpu, cpu, case):
    """fp32 convolutions on the direct-to-LDS tiles against the oracle, plain, with a residual and over it; twice (the
    arrival counters of split tiles must be back at zero), the second result bit-identical."""
    N, C, H, W, K, R, st, pd = case
    r = rng(sum(case))
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((K, C, R, R)) * np.sqrt(2.0 / (C * R * R))).astype(np.float32)
    b = r.uniform(-0.3, 0.3, K).astype(np.float32)
    args = ((pd, pd), (st, st), 1)
    got = oc.conv(gpu, x, w, b, *args, _abi.ACT_LEAKY_RELU, crsk=True, coef=0.1)
    ref = oc.conv(cpu, x, w, b, *args, _abi.ACT_IDENTITY)
    np.testing.assert_allclose(got, np.where(ref < 0, np.float32(0.1) * ref, ref), rtol=RTOL, atol=ATOL)
    np.testing.assert_array_equal(oc.conv(gpu, x, w, b, *args, _abi.ACT_LEAKY_RELU, crsk=True, coef=0.1), got)
    z = r.standard_normal(ref.shape).astype(np.float32)
    gotz = oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=True, z=z)
    np.testing.assert_allclose(gotz, np.maximum(ref + z, 0), rtol=RTOL, atol=ATOL)
    np.testing.assert_array_equal(oc.conv(gpu, x, w, b, *args, _abi.ACT_RELU, crsk=True, z=z, inplace=True), gotz)


# 168, 65 and 8 tiles in three, seven and six parts, runs of neighbouring tiles per XCD: rounds of parts that are multiples of
# eight workgroups and one that is not; 32 tiles in eight parts with more filters than activations, every eighth tile on one XCD
@pytest.mark.parametrize("case", [(8, 128, 41, 41, 192, 3, 2, 1), (4, 512, 28, 28, 320, 3, 2, 1), (5, 64, 57, 57, 256, 3, 2, 1),
                                  (2, 1024, 14, 14, 1024, 3, 2, 1)], ids=lambda c: "x".join(map(str, c)))
def test_conv_f32_split_tiles_on_their_xcd(gpu, cpu, case):
    test_conv_f32_direct_to_lds_tiles(gpu, cpu, case)


# channel counts around the four rows a wavefront loads at a time; sizes that fill the chip, whole tiles and split ones
@pytest.mark.parametrize("C", [1, 2, 3, 5, 29, 30, 33, 47])
@pytest.mark.parametrize("N,H,W,K,stride", [(3, 75, 75, 66, 1), (6, 56, 56, 64, 1), (10, 60, 60, 128, 2)])
def test_pointwise_conv_f32_any_channel_count(gpu, cpu, C, N, H, W, K, stride):
    """fp32 1x1 layers without padding whose channels are no multiple of four: against the oracle, and an image of
    infinities leaves the images beside it as they are, bit for bit (the rows past an image's last channel are the next
    image's first ones)."""
    r = rng(100 * C + H)
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    w = (r.standard_normal((K, C, 1, 1)) * np.sqrt(1.0 / C)).astype(np.float32)
    b = r.uniform(-0.3, 0.3, K).astype(np.float32)
    args = ((0, 0), (stride, stride), 1, _abi.ACT_IDENTITY)
    got = oc.conv(gpu, x, w, b, *args, crsk=True)
    np.testing.assert_allclose(got, oc.conv(cpu, x, w, b, *args), rtol=RTOL, atol=ATOL)
    for bad in (np.inf, np.nan):
        xi = x.copy()
        xi[N - 2] = bad
        goti = oc.conv(gpu, xi, w, b, *args, crsk=True)
        for n in range(N):
            if n == N - 2:
                assert not np.isfinite(goti[n]).any()
            else:
                np.testing.assert_array_equal(goti[n], got[n])


def test_conv_f16_random_shapes(gpu, cpu):
    """120 seeded shapes through the fp16 convolution, channels-last (every fast path's boundary: channel counts
    around the multiples of 8 / 32 / 64, a few steps or many, padded or not, grouped and depthwise) and, every
    third case, N,C,H,W; against the oracle to one fp16 rounding (rtol 2e-3, atol 2e-3; 4e-3 with a residual),
    the residual form also in place."""
    for i, (N, C, H, W, K, R, S, sh, sw, ph, pw, grp) in enumerate(random_conv_cases(4048, 120, True)):
        if R != S or sh != sw or ph != pw:  # the fp16 helper takes square geometry
            S, sw, pw = R, sh, ph
            if (W + 2 * pw - S) // sw + 1 < 1 or W + 2 * pw < S:
                continue
        r = rng(3000 + i)
        x = r.standard_normal((N, C, H, W)).astype(np.float16)
        w = (r.standard_normal((K, C // grp, R, R)) * np.sqrt(2.0 / (C // grp * R * R))).astype(np.float16)
        b = r.uniform(-0.3, 0.3, K).astype(np.float16)
        fmt = _abi.NCHW if i % 3 == 2 else _abi.NHWC
        what = f"case {i}: x {x.shape} w {w.shape} stride {sh} pad {ph} group {grp} format {fmt}"
        ref = oc.conv(cpu, x, w, b, (ph, ph), (sh, sh), grp, _abi.ACT_RELU)
        got = conv_f16(gpu, x, w, b, (ph, ph), (sh, sh), grp, _abi.ACT_RELU, fmt)
        np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3, err_msg=what)
        z = r.standard_normal(ref.shape).astype(np.float16)
        refz = oc.conv(cpu, x, w, b, (ph, ph), (sh, sh), grp, _abi.ACT_RELU, z=z)
        gotz = conv_f16(gpu, x, w, b, (ph, ph), (sh, sh), grp, _abi.ACT_RELU, fmt, z=z)
        np.testing.assert_allclose(gotz.astype(np.float32), refz.astype(np.float32), rtol=4e-3, atol=4e-3, err_msg=what + " + z")
        np.testing.assert_array_equal(conv_f16(gpu, x, w, b, (ph, ph), (sh, sh), grp, _abi.ACT_RELU, fmt, z=z, inplace=True), gotz,
                                      err_msg=what + " in place")


def test_conv_f16_pointwise_and_depthwise_random_shapes(gpu, cpu):
    """Seeded channels-last fp16 shapes aimed at the two kernels without a workgroup tile: 1x1 stride-1 layers over
    a multiple of 8 channels up to 256 that is not a multiple of 64 (one to sixteen 16-channel steps, the last one
    half empty every other time; few and many filters, so that results leave both through the staging tile and
    straight from the accumulators; ragged last wavefronts; few pixels, so that the filter blocks are dealt over the
    grid) and 3x3 depthwise layers with stride 1 and 2 and padding 0 to 2; each activation mode in turn, with and
    without a residual, which is also written in place.  Against the oracle to one fp16 rounding."""
    r = np.random.default_rng(909)
    acts = [(_abi.ACT_RELU, None), (_abi.ACT_IDENTITY, None), (_abi.ACT_CLIPPED_RELU, 0.7), (_abi.ACT_LEAKY_RELU, 0.1)]
    for i in range(60):
        N, H, W = int(r.integers(1, 5)), int(r.integers(1, 25)), int(r.integers(1, 25))
        if i % 2 == 0:  # pointwise
            C = 8 * int(r.integers(1, 33))
            if C % 64 == 0:
                C += 8
            K = 8 * int(r.choice([1, 2, 3, 4, 5, 8, 9, 12, 18, 40]))
            R, st, pd, grp = 1, 1, 0, 1
        else:           # depthwise
            C = K = 8 * int(r.integers(1, 40))
            R, st, pd, grp = 3, int(r.integers(1, 3)), int(r.integers(0, 3)), C
            if H + 2 * pd < 3 or W + 2 * pd < 3:
                H, W = H + 3, W + 3
        activ, coef = acts[(i // 2) % 4]
        q = rng(5000 + i)
        x = q.standard_normal((N, C, H, W)).astype(np.float16)
        w = (q.standard_normal((K, C // grp, R, R)) * np.sqrt(2.0 / (C // grp * R * R))).astype(np.float16)
        b = q.uniform(-0.3, 0.3, K).astype(np.float16)
        what = f"case {i}: x {x.shape} w {w.shape} stride {st} pad {pd} group {grp} act {activ}"
        if coef is not None:
            gpu.ops.set_activation_coef(coef)
        ref = oc.conv(cpu, x, w, b, (pd, pd), (st, st), grp, activ, coef=coef)
        got = conv_f16(gpu, x, w, b, (pd, pd), (st, st), grp, activ, _abi.NHWC)
        np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3, err_msg=what)
        z = q.standard_normal(ref.shape).astype(np.float16)
        refz = oc.conv(cpu, x, w, b, (pd, pd), (st, st), grp, activ, z=z, coef=coef)
        gotz = conv_f16(gpu, x, w, b, (pd, pd), (st, st), grp, activ, _abi.NHWC, z=z)
        np.testing.assert_allclose(gotz.astype(np.float32), refz.astype(np.float32), rtol=4e-3, atol=4e-3, err_msg=what + " + z")
        np.testing.assert_array_equal(conv_f16(gpu, x, w, b, (pd, pd), (st, st), grp, activ, _abi.NHWC, z=z, inplace=True), gotz,
                                      err_msg=what + " in place")


def test_rowwise_ops_random_shapes(gpu, cpu):
    """Seeded sweeps of soft-max, LayerNorm, ReduceMean and the poolings over shapes around their kernels'
    boundaries (row lengths on both sides of 4-element groups, of the in-register limit and of a wavefront;
    reductions over an inner, a middle and an outer run), fp32 and fp16, against the oracle."""
    r = np.random.default_rng(77)
    for i in range(60):
        rows = int(r.choice([1, 2, 3, 7, 64, 130]))
        L = int(r.choice([1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 255, 256, 257, 768, 1000, 1024, 2047, 2048, 2049, 2052, 3000, 4100]))
        for dtype, tol in ((np.float32, 1e-4), (np.float16, 4e-3)):
            x = (r.standard_normal((rows, L)) * 2 + 0.5).astype(dtype)
            close(oc.softmax(gpu, x, 1), oc.softmax(cpu, x, 1), tol, tol * 1e-2 if dtype == np.float32 else tol)
            if L > 1:
                g, b = r.standard_normal(L).astype(dtype), r.standard_normal(L).astype(dtype)
                close(oc.layernorm(gpu, x, g, b, 1e-5), oc.layernorm(cpu, x, g, b, 1e-5), max(tol, 2e-4), max(tol, 2e-4) * 4)
    for i in range(40):
        outer, red, inner = (int(v) for v in (r.integers(1, 9), r.choice([1, 2, 5, 7, 49, 64, 100, 257]), r.choice([1, 2, 3, 4, 8, 16, 48, 130])))
        for dtype, tol in ((np.float32, 1e-5), (np.float16, 2e-3)):
            x = r.standard_normal((outer, red, inner)).astype(dtype)
            close(oc.reduce_mean(gpu, x, (outer, 1, inner)), oc.reduce_mean(cpu, x, (outer, 1, inner)), tol, tol)
    for i in range(40):
        N, C, H, W = (int(v) for v in (r.integers(1, 4), r.choice([1, 3, 8, 16, 24, 33]), r.integers(2, 24), r.integers(2, 24)))
        k = (int(r.integers(1, 4)), int(r.integers(1, 4)))
        st = (int(r.integers(1, 4)), int(r.integers(1, 4)))
        pd = (int(r.integers(0, (k[0] + 1) // 2 + (k[0] > 1) - (k[0] == 2))), int(r.integers(0, (k[1] + 1) // 2 + (k[1] > 1) - (k[1] == 2))))
        pd = (min(pd[0], k[0] // 2), min(pd[1], k[1] // 2))
        if H + 2 * pd[0] < k[0] or W + 2 * pd[1] < k[1]:
            continue
        for dtype in (np.float32, np.float16):
            x = r.standard_normal((N, C, H, W)).astype(dtype)
            if i % 5 == 0:
                x[0, 0, H // 2, W // 2] = np.nan
            got, ref = oc.pool(gpu, "max", x, k, pd, st), oc.pool(cpu, "max", x, k, pd, st)
            np.testing.assert_array_equal(got, ref, err_msg=f"max pool {x.shape} k {k} pads {pd} strides {st} {dtype.__name__}")
            if i % 5:
                tol = 1e-5 if dtype == np.float32 else 2e-3
                close(oc.pool(gpu, "avg", x, k, pd, st), oc.pool(cpu, "avg", x, k, pd, st), tol, tol)


def test_products_random_shapes(gpu, cpu):
    """Seeded sweeps of the 2-D product (every layout, alpha / beta, row and matrix C) and the batched product with
    bias, residual and GELU over ragged shapes, fp32 and fp16, against the oracle."""
    r = np.random.default_rng(78)
    dims = [1, 2, 3, 5, 8, 17, 31, 32, 33, 64, 65, 100, 128, 130, 257]
    for i in range(50):
        M, K, N = (int(r.choice(dims)) for _ in range(3))
        tA, tB = int(r.integers(0, 2)), int(r.integers(0, 2))
        for dtype, tol in ((np.float32, (1e-4, 1e-4)), (np.float16, (4e-3, 8e-3))):
            a = r.standard_normal((K, M) if tA else (M, K)).astype(dtype)
            b = (r.standard_normal((N, K) if tB else (K, N)) / np.sqrt(K)).astype(dtype)
            kw = [dict(), dict(alpha=0.5), dict(c=r.standard_normal((M, N)).astype(dtype), alpha=1.5, beta=0.5)][i % 3]
            got, ref = oc.matmul2d(gpu, a, b, transA=tA, transB=tB, **kw), oc.matmul2d(cpu, a, b, transA=tA, transB=tB, **kw)
            np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=tol[0], atol=tol[1],
                                       err_msg=f"[{M},{K}]x[{K},{N}] transA {tA} transB {tB} {kw.keys()} {dtype.__name__}")
    for i in range(40):
        M, K, N = (int(r.choice(dims)) for _ in range(3))
        batch = [(), (2,), (3, 2)][i % 3]
        shared_b = i % 2 == 0
        for dtype, tol in ((np.float32, (1e-4, 1e-4)), (np.float16, (1e-2, 1e-2))):
            a = r.standard_normal(batch + (M, K)).astype(dtype)
            b = (r.standard_normal((() if shared_b else batch) + (K, N)) / np.sqrt(K)).astype(dtype)
            bias = r.standard_normal(N).astype(dtype)
            z = r.standard_normal(batch + (M, N)).astype(dtype)
            kw = [dict(), dict(z=z), dict(gelu=True), dict(z=z, gelu=True)][i % 4]
            got, ref = oc.matmul_nd_bias(gpu, a, b, bias, **kw), oc.matmul_nd_bias(cpu, a, b, bias, **kw)
            np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=tol[0], atol=tol[1],
                                       err_msg=f"{a.shape} x {b.shape} {list(kw)} {dtype.__name__}")
            got, ref = oc.matmul_nd(gpu, a, b), oc.matmul_nd(cpu, a, b)
            np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=tol[0], atol=tol[1], err_msg=f"{a.shape} x {b.shape}")


def test_conv_closed_forms(gpu):
    x = rng(1).standard_normal((1, 3, 8, 8)).astype(np.float32)
    w = np.zeros((3, 3, 3, 3), np.float32)
    for c in range(3):
        w[c, c, 1, 1] = 1
    np.testing.assert_array_equal(oc.conv(gpu, x, w, None, (1, 1), (1, 1)), x)
    w = np.zeros((1, 1, 3, 3), np.float32)
    w[0, 0, 0, 2] = 1
    xi = np.arange(36, dtype=np.float32).reshape(1, 1, 6, 6)
    exp = np.zeros((6, 6), np.float32)
    exp[1:, :-1] = xi[0, 0, :-1, 1:]
    np.testing.assert_array_equal(oc.conv(gpu, xi, w, None, (1, 1), (1, 1))[0, 0], exp)


def test_conv_errors(gpu):
    x = np.zeros((1, 4, 4, 4), np.float32)
    with pytest.raises(RuntimeError):
        oc.conv(gpu, x, np.zeros((4, 3, 1, 1), np.float32))
    with pytest.raises(RuntimeError):
        oc.conv(gpu, x, np.zeros((4, 4, 7, 7), np.float32))


# ---- elementwise -----------------------------------------------------------------

@pytest.mark.parametrize("n", [1, 3, 255, 256, 1025, 200704])
def test_unary_exact(gpu, cpu, n):
    x = np.concatenate([rng(n).standard_normal(n) * 3]).astype(np.float32)
    x[0] = -0.0
    for name, kw in [("relu", {}), ("negative", {}), ("clip", {"lo": 0.0, "hi": 6.0})]:
        np.testing.assert_array_equal(oc.unary(gpu, name, x, **kw), oc.unary(cpu, name, x, **kw))
    nz = np.where(x == 0, np.float32(1), x)
    np.testing.assert_array_equal(oc.unary(gpu, "reciprocal", nz), oc.unary(cpu, "reciprocal", nz))
    np.testing.assert_array_equal(oc.unary(gpu, "sqrt", np.abs(x)), oc.unary(cpu, "sqrt", np.abs(x)))
    np.testing.assert_array_equal(oc.pow_(gpu, x, 2.0), oc.pow_(cpu, x, 2.0))
    for name in ("erf", "gelu", "sigmoid", "tanh"):
        close(oc.unary(gpu, name, x), oc.unary(cpu, name, x))
    close(oc.pow_(gpu, np.abs(x) + 0.5, 1.5), oc.pow_(cpu, np.abs(x) + 0.5, 1.5))


def test_unary_misc(gpu, cpu):
    assert np.isnan(oc.unary(gpu, "relu", np.array([np.nan, 1.0], np.float32))[0])
    i = rng(2).integers(-2 ** 40, 2 ** 40, 777)
    np.testing.assert_array_equal(oc.cast(gpu, i), oc.cast(cpu, i))
    # 4-D shape through dnnrtActive, and an unaligned view (pointer + 4 bytes)
    x = rng(3).standard_normal((2, 3, 5, 7)).astype(np.float32)
    np.testing.assert_array_equal(oc.unary(gpu, "relu", x), oc.unary(cpu, "relu", x))
    t = gpu.put(rng(4).standard_normal(1030).astype(np.float32))
    y = gpu.empty(1030)
    gpu.ops.negative(gpu.ptr(t) + 4, gpu.ptr(y) + 4, [1029])
    gpu.sync()
    np.testing.assert_array_equal(gpu.get(y)[1:], -gpu.get(t)[1:])
    # fp16 storage
    h = (rng(5).standard_normal(5000) * 4).astype(np.float16)
    for name, kw in [("relu", {}), ("negative", {}), ("clip", {"lo": 0.0, "hi": 6.0})]:
        np.testing.assert_array_equal(oc.unary(gpu, name, h, **kw), oc.unary(cpu, name, h, **kw))
    close(oc.unary(gpu, "gelu", h).astype(np.float32), oc.unary(cpu, "gelu", h).astype(np.float32), 2e-2, 1e-3)


def test_tensor_op(gpu, cpu):
    r = rng(7)
    shapes = [((2, 5, 3, 4), (2, 5, 3, 4)), ((2, 5, 3, 4), (1, 5, 1, 1)), ((2, 5, 3, 4), (1, 1, 1, 4)),
              ((2, 5, 3, 4), (2, 1, 3, 1)), ((2, 5, 3, 4), (1, 1, 1, 1)), ((2, 5, 3, 4), (1, 5, 3, 1)),
              ((1, 256, 56, 56), (1, 256, 56, 56)), ((1, 256, 56, 56), (1, 256, 1, 1)),
              ((1, 1000), (1, 1000)), ((1, 128, 768), (1, 1, 768)), ((1, 128, 768), (1, 128, 1)),
              ((3, 7), (1, 7)), ((5,), (5,)), ((5,), (1,))]
    for sa, sb in shapes:
        a = r.standard_normal(sa).astype(np.float32)
        b = r.standard_normal(sb).astype(np.float32)
        for op in (_abi.OP_ADD, _abi.OP_MUL):
            np.testing.assert_array_equal(oc.tensor_op(gpu, op, a, b), oc.tensor_op(cpu, op, a, b))
            np.testing.assert_array_equal(oc.tensor_op(gpu, op, a, b, coef=-2.5), oc.tensor_op(cpu, op, a, b, coef=-2.5))
        np.testing.assert_array_equal(oc.tensor_op(gpu, _abi.OP_ADD, a, b, inplace=True),
                                      oc.tensor_op(cpu, _abi.OP_ADD, a, b, inplace=True))
    with pytest.raises(RuntimeError):
        oc.tensor_op(gpu, _abi.OP_ADD, np.zeros((2, 4), np.float32), np.zeros((2, 3), np.float32))
    a = r.standard_normal((2, 3, 4, 8)).astype(np.float16)
    b = r.standard_normal((1, 3, 1, 1)).astype(np.float16)
    np.testing.assert_array_equal(oc.tensor_op(gpu, _abi.OP_ADD, a, b), oc.tensor_op(cpu, _abi.OP_ADD, a, b))
    # 16-byte broadcast path (innermost run a multiple of 16 bytes) next to the element-wise one, both dtypes
    for dtype in (np.float32, np.float16):
        for sa, sb in [((2, 6, 4, 8), (1, 6, 1, 1)), ((2, 6, 4, 8), (2, 1, 4, 8)), ((2, 6, 4, 8), (2, 6, 1, 1)),
                       ((2, 6, 4, 8), (1, 1, 1, 8)), ((2, 6, 4, 8), (1, 6, 1, 8)), ((2, 6, 4, 8), (1, 1, 4, 1)),
                       ((3, 5, 16), (3, 1, 16)), ((3, 5, 16), (1, 5, 1)), ((4, 24), (1, 1)), ((4, 24), (4, 1)),
                       ((2, 6, 3, 6), (1, 6, 1, 1)), ((1, 64, 96, 96), (1, 1, 1, 1)), ((2, 64, 28, 28), (1, 64, 1, 1))]:
            a = r.standard_normal(sa).astype(dtype)
            b = r.standard_normal(sb).astype(dtype)
            want = (a.astype(np.float32) + b.astype(np.float32)).astype(dtype)
            np.testing.assert_array_equal(oc.tensor_op(gpu, _abi.OP_ADD, a, b), want)
            np.testing.assert_array_equal(oc.tensor_op(gpu, _abi.OP_MUL, a, b), oc.tensor_op(cpu, _abi.OP_MUL, a, b))


# ---- reductions --------------------------------------------------------------------

def test_reduce_mean(gpu, cpu):
    r = rng(9)
    for shape, out in [((1, 2048, 7, 7), (1, 2048, 1, 1)), ((2, 6, 7, 7), (2, 1, 7, 7)), ((2, 6, 7, 7), (1, 6, 7, 7)),
                       ((1, 128, 768), (1, 128, 1)), ((3, 1000), (3, 1)), ((1, 1280, 7, 7), (1, 1280, 1, 1))]:
        x = r.standard_normal(shape).astype(np.float32)
        close(oc.reduce_mean(gpu, x, out), oc.reduce_mean(cpu, x, out))
    # a middle dim reduced over an inner run of whole 8-byte units (what a channels-last global average
    # pool is): 7 + 3, 49 and 5 reduction steps, both element types, against numpy's float64 mean
    for shape, out in [((3, 10, 16), (3, 1, 16)), ((4, 49, 256), (4, 1, 256)), ((2, 5, 3, 8), (2, 1, 3, 8)), ((1, 7, 6), (1, 1, 6))]:
        for dtype, tol in ((np.float32, 1e-5), (np.float16, 2e-3)):
            x = r.standard_normal(shape).astype(dtype)
            got = oc.reduce_mean(gpu, x, out)
            close(got, oc.reduce_mean(cpu, x, out), tol, tol)
            np.testing.assert_allclose(got.astype(np.float64), x.astype(np.float64).mean(1, keepdims=True), rtol=tol, atol=tol)
    with pytest.raises(RuntimeError):
        oc.reduce_mean(gpu, np.zeros((2, 3, 4, 5), np.float32), (1, 3, 1, 5))


def test_softmax(gpu, cpu):
    r = rng(10)
    x = (r.standard_normal((1, 12, 128, 128)) * 3).astype(np.float32)
    got = oc.softmax(gpu, x, 3)
    close(got, oc.softmax(cpu, x, 3), 1e-4, 1e-7)
    close(got.sum(3), 1.0, 1e-5)
    x = (r.standard_normal((2, 3, 5, 17)) * 4).astype(np.float32)
    for axis in (3, -1, 1, 0, 2):
        close(oc.softmax(gpu, x, axis), oc.softmax(cpu, x, axis), 1e-4, 1e-7)
    big = np.array([[1000.0, 1000.0, -1000.0]], np.float32)
    close(oc.softmax(gpu, big, 1), [[0.5, 0.5, 0.0]], 1e-6, 1e-7)


def test_layernorm(gpu, cpu):
    r = rng(12)
    # rows held in registers (L % 4 == 0, up to 2048: one to eight groups of four per lane, few and
    # many rows) and the general kernel (odd L, long rows)
    for shape in [(1, 128, 768), (2, 7, 48), (5, 1000), (3, 1), (3, 4), (2, 300), (1, 2048), (1300, 256), (2, 1540), (2, 4096), (4, 1026)]:
        L = shape[-1]
        x = (r.standard_normal(shape) * 3 + 1).astype(np.float32)
        g = r.standard_normal(L).astype(np.float32)
        b = r.standard_normal(L).astype(np.float32)
        close(oc.layernorm(gpu, x, g, b, 1e-12 if L > 1 else 1e-5), oc.layernorm(cpu, x, g, b, 1e-12 if L > 1 else 1e-5), 1e-4, 1e-4)
    for shape in [(16, 768), (3, 64), (2, 2052)]:
        L = shape[-1]
        x = (r.standard_normal(shape) * 3 + 1).astype(np.float16)
        g, b = r.standard_normal(L).astype(np.float16), r.standard_normal(L).astype(np.float16)
        np.testing.assert_allclose(oc.layernorm(gpu, x, g, b, 1e-5).astype(np.float32), oc.layernorm(cpu, x, g, b, 1e-5).astype(np.float32),
                                   rtol=2e-2, atol=2e-2)


# one lane's group of four to eight wavefronts a row, a last group short of the wavefront and of the row; few rows, and more than share the chip that way
@pytest.mark.parametrize("L", [4, 252, 256, 260, 508, 768, 1028, 1536, 1540, 2044, 2048])
@pytest.mark.parametrize("rows", [1, 130, 400])
def test_layernorm_of_few_rows(gpu, rows, L):
    """Against 64 bits.  Bound: the sums over a row are trees of at most 17 additions, so the mean is within 20 2^-24 of the mean magnitude,
    and the deviations, their mean square, root, quotient and the last two operations round a few times each."""
    r = rng(rows + L)
    x = (r.standard_normal((rows, L)) * 3 + 1).astype(np.float32)
    g, b = r.standard_normal(L).astype(np.float32), r.standard_normal(L).astype(np.float32)
    x6, u = x.astype(np.float64), 2.0 ** -24
    d = x6 - x6.mean(-1, keepdims=True)
    inv = 1 / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-5)
    mean_error = 20 * u * np.abs(x6).mean(-1, keepdims=True)
    bound = inv * np.abs(g) * (2 * mean_error + np.abs(d) * (28 * u + 2 * mean_error * inv)) + 4 * u * np.abs(b)
    assert (np.abs(oc.layernorm(gpu, x, g, b, 1e-5) - (d * inv * g + b)) <= bound).all()


# ---- pooling ---------------------------------------------------------------------------

def test_pooling(gpu, cpu):
    r = rng(13)
    x = r.standard_normal((1, 64, 112, 112)).astype(np.float32)
    np.testing.assert_array_equal(oc.pool(gpu, "max", x, (3, 3), (1, 1), (2, 2)), oc.pool(cpu, "max", x, (3, 3), (1, 1), (2, 2)))
    x = r.standard_normal((2, 3, 13, 12)).astype(np.float32)
    for k, p, s in [(3, 1, 2), (2, 0, 2), (3, 0, 1), (3, 1, 1)]:
        np.testing.assert_array_equal(oc.pool(gpu, "max", x, (k, k), (p, p), (s, s)), oc.pool(cpu, "max", x, (k, k), (p, p), (s, s)))
        close(oc.pool(gpu, "avg", x, (k, k), (p, p), (s, s)), oc.pool(cpu, "avg", x, (k, k), (p, p), (s, s)))
    xn = x.copy()
    xn[0, 0, 0, 0] = np.nan
    np.testing.assert_array_equal(np.isnan(oc.pool(gpu, "max", xn, (3, 3), (1, 1), (2, 2))),
                                  np.isnan(oc.pool(cpu, "max", xn, (3, 3), (1, 1), (2, 2))))


# ---- matrix products --------------------------------------------------------------------

def test_matmul2d(gpu, cpu):
    r = rng(14)
    # the few-row shapes take the dot-product kernel with 1, 4 or 16 wavefronts per output
    for M, K, N in [(1, 2048, 1000), (1, 1280, 1000), (5, 9, 7), (64, 64, 64), (130, 70, 33), (3, 2048, 10), (16, 250, 40),
                    (2, 50176, 496), (8, 8194, 33), (1, 9216, 4096), (7, 2049, 5)]:
        a = r.standard_normal((M, K)).astype(np.float32)
        b = (r.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
        c = r.standard_normal((M, N)).astype(np.float32)
        ref = oc.matmul2d(cpu, a, b)
        close(oc.matmul2d(gpu, a, b), ref)
        close(oc.matmul2d(gpu, a.T.copy(), b, transA=1), ref)
        close(oc.matmul2d(gpu, a, b.T.copy(), transB=1), ref)
        close(oc.matmul2d(gpu, a.T.copy(), b.T.copy(), transA=1, transB=1), ref)
        close(oc.matmul2d(gpu, a, b.T.copy(), c.copy(), alpha=0.5, beta=-2.0, transB=1),
              oc.matmul2d(cpu, a, b.T.copy(), c.copy(), alpha=0.5, beta=-2.0, transB=1))
        # C as one row (a Gemm's bias folded into the product): equal to product-then-add on the GPU, bit for bit
        row = c[0].copy()
        for tb, bb in ((0, b), (1, b.T.copy())):
            fused = oc.matmul2d_row(gpu, a, bb, row, transB=tb)
            close(fused, oc.matmul2d_row(cpu, a, bb, row, transB=tb))
            np.testing.assert_array_equal(fused, oc.tensor_op(gpu, _abi.OP_ADD, oc.matmul2d(gpu, a, bb, transB=tb), row.reshape(1, -1)))
    with pytest.raises(RuntimeError):
        oc.matmul2d(gpu, np.zeros((5, 9), np.float32), np.zeros((9, 7), np.float32), transB=1)


def test_matmul_nd(gpu, cpu):
    r = rng(15)
    cases = [((1, 128, 768), (768, 768)), ((1, 12, 128, 64), (1, 12, 64, 128)), ((1, 12, 128, 128), (1, 12, 128, 64)),
             ((1, 128, 768), (768, 3072)), ((1, 128, 3072), (3072, 768)),
             ((4, 6), (6, 3)), ((2, 4, 6), (6, 3)), ((2, 3, 4, 6), (2, 3, 6, 5)), ((2, 4, 6), (2, 6, 3)), ((4, 6), (3, 6, 2)),
             # the LDS-staged row-major kernel: ragged rows and columns, 1 to 11 reduction splits (odd counts too)
             # (it takes products of 1.5e8 multiply-adds and more)
             ((1, 100, 1056), (1056, 1540)), ((1, 33, 3072), (3072, 1604)), ((200, 2048), (2048, 388)), ((300, 1024), (1024, 512)),
             ((2, 77, 1024), (1024, 1028)), ((1024, 256), (256, 1024)), ((1, 128, 768), (768, 2304))]
    for sa, sb in cases:
        a = r.standard_normal(sa).astype(np.float32)
        b = (r.standard_normal(sb) / np.sqrt(sb[-2])).astype(np.float32)
        ref = oc.matmul_nd(cpu, a, b)
        close(oc.matmul_nd(gpu, a, b), ref)
        close(oc.matmul_nd(gpu, a, b), ref)   # again: the split-reduction counters must be back at zero
    # fp16 tensors (fp32 accumulation, one rounding): the transformer shapes, broadcast batches, ragged tiles
    for sa, sb in [((1, 128, 768), (768, 768)), ((1, 12, 128, 64), (1, 12, 64, 128)), ((1, 12, 128, 128), (1, 12, 128, 64)),
                   ((4, 6), (6, 3)), ((2, 4, 6), (6, 3)), ((2, 3, 4, 6), (2, 3, 6, 5)), ((2, 4, 6), (2, 6, 3)), ((4, 6), (3, 6, 2)),
                   ((2, 77, 130), (130, 70)),
                   # few tiles and long reductions: split over 2 to 16 workgroups (odd step counts too), twice each
                   # (the arrival counters must be back at zero)
                   ((1, 128, 768), (768, 3072)), ((1, 128, 3072), (3072, 768)), ((1, 33, 1100), (1100, 100)), ((3, 64, 4000), (4000, 64))]:
        a = r.standard_normal(sa).astype(np.float16)
        b = (r.standard_normal(sb) / np.sqrt(sb[-2])).astype(np.float16)
        ref = oc.matmul_nd(cpu, a, b).astype(np.float32)
        first = oc.matmul_nd(gpu, a, b)
        np.testing.assert_allclose(first.astype(np.float32), ref, rtol=2e-3, atol=2e-3)
        np.testing.assert_array_equal(oc.matmul_nd(gpu, a, b), first)


def test_split_reduction_hand_over_is_deterministic(gpu, cpu):
    """Reductions split over workgroups meet through partial tiles and arrival counters in the handle's scratch;
    partial tiles are added in split order, so the result does not depend on who arrives last.  The deepest
    split of ResNet-50 at batch 1 (3x3 over 512 channels at 7x7), a 1x1 layer over 2048 channels and the
    768 -> 3072 product, 200 times each on one handle: every repetition bit-identical to the first, which
    matches the oracle."""
    r = rng(91)
    def repeat(call, ref):
        first = call()
        close(gpu.get(first), ref)
        first = first.clone()
        for i in range(200):
            again = call()
            assert gpu.torch.equal(again, first), f"repetition {i} differs"
    for case in [(1, 512, 7, 7, 512, 3, 1, 1), (1, 2048, 7, 7, 512, 1, 1, 0), (1, 1024, 14, 14, 256, 1, 1, 0)]:
        N, C, H, W, K, R, st, pd = case
        x = r.standard_normal((N, C, H, W)).astype(np.float32)
        w = (r.standard_normal((K, C, R, R)) * np.sqrt(2.0 / (C * R * R))).astype(np.float32)
        b = r.uniform(-0.1, 0.1, K).astype(np.float32)
        ref = oc.conv(cpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_RELU)
        P, Q = oc.conv_out_hw(H, W, R, R, (pd, pd), (st, st))
        X, Wt, B, Y = gpu.put(x), gpu.put(w), gpu.put(b), gpu.empty((N, K, P, Q))
        def conv_call():
            gpu.ops.conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (pd, pd), (st, st), _abi.ACT_RELU,
                                    gpu.ptr(Y), 1, _abi.F32)
            gpu.sync()
            return Y
        repeat(conv_call, ref)
    a = r.standard_normal((1, 128, 768)).astype(np.float32)
    b = (r.standard_normal((768, 3072)) / np.sqrt(768)).astype(np.float32)
    ref = oc.matmul_nd(cpu, a, b)
    A, Bm, Y = gpu.put(a), gpu.put(b), gpu.empty((1, 128, 3072))
    def mm_call():
        gpu.ops.matmul_nd(gpu.ptr(A), a.shape, gpu.ptr(Bm), b.shape, gpu.ptr(Y), (1, 128, 3072), _abi.F32)
        gpu.sync()
        return Y
    repeat(mm_call, ref)
    # the fp16 product splits its reduction the same way (3072 -> 768: eleven workgroups per tile, 768 -> 3072: none)
    for K, N in ((3072, 768), (768, 768)):
        a16 = r.standard_normal((1, 128, K)).astype(np.float16)
        b16 = (r.standard_normal((K, N)) / np.sqrt(K)).astype(np.float16)
        ref16 = oc.matmul_nd(cpu, a16, b16).astype(np.float32)
        A16, B16, Y16 = gpu.put(a16), gpu.put(b16), gpu.empty((1, 128, N), np.float16)
        def mm16_call():
            gpu.ops.matmul_nd(gpu.ptr(A16), a16.shape, gpu.ptr(B16), b16.shape, gpu.ptr(Y16), (1, 128, N), _abi.F16)
            gpu.sync()
            return Y16
        first = mm16_call()
        np.testing.assert_allclose(gpu.get(first).astype(np.float32), ref16, rtol=4e-3, atol=8e-3)
        first = first.clone()
        for i in range(200):
            assert gpu.torch.equal(mm16_call(), first), f"fp16 product {K} -> {N}: repetition {i} differs"


def test_matmul_nd_bias(gpu, cpu):
    r = rng(44)
    # transformer Linear layers (one tall product, the dot-product kernel for few rows) and batched products
    for sa, sb in [((1, 128, 768), (768, 768)), ((1, 128, 768), (768, 3072)), ((1, 128, 3072), (3072, 768)), ((5, 7), (7, 3)),
                   ((3, 6, 5), (3, 5, 4)), ((2, 12, 40, 64), (2, 12, 64, 40)), ((1, 3, 33), (33, 130))]:
        a = r.standard_normal(sa).astype(np.float32)
        b = (r.standard_normal(sb) / np.sqrt(sb[-2])).astype(np.float32)
        bias = r.standard_normal(sb[-1]).astype(np.float32)
        close(oc.matmul_nd_bias(gpu, a, b, bias), oc.matmul_nd_bias(cpu, a, b, bias))
        z = r.standard_normal(np.broadcast_shapes(sa[:-2], sb[:-2]) + (sa[-2], sb[-1])).astype(np.float32)
        close(oc.matmul_nd_bias(gpu, a, b, bias, z=z), oc.matmul_nd_bias(cpu, a, b, bias, z=z))
        close(oc.matmul_nd_bias(gpu, a, b, bias, gelu=True), oc.matmul_nd_bias(cpu, a, b, bias, gelu=True))
    # fp16 tensors: the generic fp16 product (fp32 accumulation, bias, residual and GELU before the one rounding;
    # the oracle rounds to fp16 after the product and after each of the three)
    for sa, sb in [((1, 128, 768), (768, 768)), ((5, 7), (7, 3)), ((3, 6, 5), (3, 5, 4)), ((2, 12, 40, 64), (2, 12, 64, 40)), ((1, 3, 33), (33, 130))]:
        a = r.standard_normal(sa).astype(np.float16)
        b = (r.standard_normal(sb) / np.sqrt(sb[-2])).astype(np.float16)
        bias = r.standard_normal(sb[-1]).astype(np.float16)
        z = r.standard_normal(np.broadcast_shapes(sa[:-2], sb[:-2]) + (sa[-2], sb[-1])).astype(np.float16)
        for kw in (dict(), dict(z=z), dict(gelu=True), dict(z=z, gelu=True)):
            np.testing.assert_allclose(oc.matmul_nd_bias(gpu, a, b, bias, **kw).astype(np.float32),
                                       oc.matmul_nd_bias(cpu, a, b, bias, **kw).astype(np.float32), rtol=1e-2, atol=1e-2)


def test_attention(gpu, cpu):
    r = rng(45)
    # BERT-base's shape; key counts around the 32-key wavefront slice and the 128-key block; every head size
    for B, Sq, Sk, H, D in [(1, 128, 128, 12, 64), (2, 50, 77, 3, 32), (1, 300, 300, 2, 128), (1, 1, 5, 1, 64), (1, 33, 129, 4, 64),
                            (3, 64, 31, 2, 64), (1, 40, 512, 2, 64)]:
        q, k, v = (r.standard_normal((B, S, H * D)).astype(np.float32) for S in (Sq, Sk, Sk))
        q *= 2.0                                              # sharper soft-max: the running maximum moves between blocks
        close(oc.attention(gpu, q, k, v, H, 1.0 / np.sqrt(D)), oc.attention(cpu, q, k, v, H, 1.0 / np.sqrt(D)), 1e-4, 1e-5)
    qkv = r.standard_normal((2, 130, 3 * 256)).astype(np.float32)          # Q | K | V per row
    close(oc.attention_packed(gpu, qkv, 4, 0.125), oc.attention_packed(cpu, qkv, 4, 0.125), 1e-4, 1e-5)
    with pytest.raises(RuntimeError):
        oc.attention(gpu, q[:, :, :96], k[:, :, :96], v[:, :, :96], 2, 1.0)   # head size 48
    # fp16 tensors: widened on the way in, fp32 in between, one rounding on the way out (the oracle does the same)
    for B, Sq, Sk, H, D in [(1, 128, 128, 12, 64), (2, 50, 77, 3, 32), (1, 33, 129, 4, 64), (1, 40, 300, 2, 128)]:
        q, k, v = (r.standard_normal((B, S, H * D)).astype(np.float16) for S in (Sq, Sk, Sk))
        np.testing.assert_allclose(oc.attention(gpu, q, k, v, H, 1.0 / np.sqrt(D)).astype(np.float32),
                                   oc.attention(cpu, q, k, v, H, 1.0 / np.sqrt(D)).astype(np.float32), rtol=2e-3, atol=2e-3)
    qkv = r.standard_normal((2, 130, 3 * 256)).astype(np.float16)
    np.testing.assert_allclose(oc.attention_packed(gpu, qkv, 4, 0.125).astype(np.float32),
                               oc.attention_packed(cpu, qkv, 4, 0.125).astype(np.float32), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("dtype", [np.float32, np.float16, np.int64])
@pytest.mark.parametrize("dims,perm", [((2, 3, 2, 2, 5, w), (0, 1, 4, 2, 5, 3)) for w in (1, 2, 3, 4, 6, 8, 234)] +
                         [((2, 12), (1, 0)), ((2, 3, 12), (2, 1, 0)), ((5, 2, 8), (0, 2, 1)), ((2, 5, 8), (1, 2, 0)), ((3, 2, 7, 4), (0, 2, 3, 1))], ids=str)
def test_transpose_rows_in_pairs(gpu, dims, perm, dtype):
    """The last result dim two strided elements, the one before it the input's last: pixel shuffles by two and plain
    transposes of two rows, of widths and strides the wide loads take and do not."""
    x = rng(len(dims)).integers(-999, 999, dims).astype(dtype)
    np.testing.assert_array_equal(oc.transpose(gpu, x, perm), x.transpose(perm))


@pytest.mark.parametrize("case", [(9, 4, 10), (32, 2048, 1000), (33, 20, 31), (64, 1280, 70), (100, 512, 513), (11, 2052, 1)], ids=str)
def test_matmul2d_f32_rows_of_the_right_operand(gpu, case):
    """Batches of dozens against a right operand with its reduction in a row: ragged in both directions, split reductions and
    none, every kind of C.  Bound: K + 3 roundings of at most 2^-24 of the sum of magnitudes."""
    M, K, N = case
    r = rng(sum(case))
    a, b = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((N, K)).astype(np.float32)
    c, row = r.standard_normal((M, N)).astype(np.float32), r.standard_normal(N).astype(np.float32)
    ab, mag = a.astype(np.float64) @ b.T.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).T.astype(np.float64)
    check = lambda got, ref, m: np.testing.assert_array_less(np.abs(got - ref), (K + 3) * 2.0 ** -24 * m + 1e-30)  # noqa: E731
    for _ in range(2):  # twice: the split reduction's counters must be back at zero
        check(oc.matmul2d(gpu, a, b, transB=1), ab, mag)
        check(oc.matmul2d(gpu, a, b, c, 0.5, 2.0, transB=1), 0.5 * ab + 2.0 * c, 0.5 * mag + 2 * np.abs(c))
        check(oc.matmul2d_row(gpu, a, b, row, transB=1), ab + row, mag + np.abs(row))
        check(oc.matmul2d_row(gpu, a, b, row, 1.0, 0.25, transB=1), ab + 0.25 * row, mag + np.abs(row))


@pytest.mark.parametrize("L", [1, 5, 63, 64, 65, 200])
def test_every_lane_counts_once_in_sums_and_maxima_over_a_wavefront(gpu, L):
    """Rows with one element of weight: L * mean is exactly it wherever it lies, and a soft-max over -300 and one 0 is one-hot."""
    x = 2.0 ** 20 * np.eye(L, dtype=np.float32) + np.float32(1)
    np.testing.assert_array_equal(oc.reduce_mean(gpu, x.reshape(L, L), (L, 1)), np.full((L, 1), np.float32(2 ** 20 + L) / np.float32(L)))
    hot = np.where(np.eye(L, dtype=bool), 0, -300).astype(np.float32)
    np.testing.assert_array_equal(oc.softmax(gpu, hot, 1), np.eye(L, dtype=np.float32))


# B, queries, keys, heads, head size: on either side of 16 queries, of a block of 32 keys, of one round of four and of eight wavefronts, of
# the number of workgroups from which 32 queries are taken at a time; wavefronts without keys
@pytest.mark.parametrize("case", [(1, 1, 1, 1, 32), (1, 15, 31, 2, 64), (2, 16, 33, 3, 128), (1, 17, 96, 2, 64), (1, 33, 127, 4, 32), (1, 128, 128, 12, 64), (3, 20, 129, 2, 64),
                                  (1, 50, 255, 3, 128), (1, 64, 257, 12, 64), (2, 31, 300, 2, 32), (1, 8, 700, 1, 64), (1, 337, 40, 12, 64), (1, 320, 40, 13, 64)], ids=str)
def test_attention_f32_of_few_queries(gpu, case):
    """Against 64 bits.  Bound: a score's product of DH terms rounds by at most (DH + 2) 2^-24 of the terms' magnitudes; a probability
    changes by as much, relative, with its sum's, and the two sums over the keys round by 2^-24 a term."""
    B, Sq, Sk, H, D = case
    r = rng(sum(case))
    q, k, v = (r.standard_normal((B, n, H * D)).astype(np.float32) for n in (Sq, Sk, Sk))
    scale = 1.0 / np.sqrt(D)
    split = lambda t: t.astype(np.float64).reshape(B, -1, H, D).transpose(0, 2, 1, 3)  # noqa: E731
    q6, k6, v6 = split(q), split(k), split(v)
    s = scale * (q6 @ k6.transpose(0, 1, 3, 2))
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    u = 2.0 ** -24
    e = (D + 2) * u * (scale * (np.abs(q6) @ np.abs(k6).transpose(0, 1, 3, 2))).max(-1, keepdims=True) + 2 * u * (s.max(-1, keepdims=True) - s).max(-1, keepdims=True)
    merge = lambda t: t.transpose(0, 2, 1, 3).reshape(B, Sq, H * D)  # noqa: E731
    want, bound = merge(p @ v6), merge((4 * e + (2 * Sk + 12) * u) * (p @ np.abs(v6)))
    got = oc.attention(gpu, q, k, v, H, scale)
    assert (np.abs(got - want) <= bound).all()
    np.testing.assert_array_equal(oc.attention(gpu, q, k, v, H, scale), got)


# B, queries, keys, heads, head size, blocks of 32 keys without weight: all that a wavefront has, of four and of eight; its first one, its last
# one; all but a single key of the last block
@pytest.mark.parametrize("case", [(1, 20, 128, 2, 64, (1,)), (1, 20, 128, 2, 32, (0, 2, 3)), (2, 16, 100, 2, 128, (3,)), (1, 33, 512, 2, 64, (2, 10)), (1, 33, 512, 3, 64, (2,)),
                                  (1, 33, 512, 3, 32, (0, 1, 2, 3, 4, 5, 6, 7, 9)), (1, 17, 400, 2, 64, (12,)), (1, 17, 300, 2, 128, (0, 5)), (1, 17, 257, 2, 64, tuple(range(8)))], ids=str)
def test_attention_f32_of_few_queries_and_keys_without_weight(gpu, case):
    """Scores of minus infinity, from keys of minus infinity and queries that are positive there, while others are finite: exactly no weight.
    Against 64 bits; bound as above, over the keys that have a weight."""
    B, Sq, Sk, H, D, blocks = case
    r = rng(Sq + Sk + len(blocks))
    q, k, v = (r.standard_normal((B, n, H * D)).astype(np.float32) for n in (Sq, Sk, Sk))
    weight = np.ones(Sk, bool)
    for b in blocks:
        weight[32 * b:32 * b + 32] = False
    q[:, :, ::D] = np.abs(q[:, :, ::D]) + np.float32(0.5)
    masked = k.copy()
    masked[:, ~weight, ::D] = -np.inf
    scale = 1.0 / np.sqrt(D)
    split = lambda t: t.astype(np.float64).reshape(B, -1, H, D).transpose(0, 2, 1, 3)  # noqa: E731
    q6, k6, v6 = split(q), split(k[:, weight]), split(v[:, weight])
    s = scale * (q6 @ k6.transpose(0, 1, 3, 2))
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    u = 2.0 ** -24
    e = (D + 2) * u * (scale * (np.abs(q6) @ np.abs(k6).transpose(0, 1, 3, 2))).max(-1, keepdims=True) + 2 * u * (s.max(-1, keepdims=True) - s).max(-1, keepdims=True)
    merge = lambda t: t.transpose(0, 2, 1, 3).reshape(B, Sq, H * D)  # noqa: E731
    want, bound = merge(p @ v6), merge((4 * e + (2 * Sk + 12) * u) * (p @ np.abs(v6)))
    assert (np.abs(oc.attention(gpu, q, masked, v, H, scale) - want) <= bound).all()


@pytest.mark.parametrize("case", [(1, 384, 384, 12, 64), (2, 31, 257, 3, 64), (1, 70, 129, 2, 32), (1, 64, 160, 5, 32), (1, 45, 513, 2, 128),
                                  (1, 1, 1, 1, 64), (3, 33, 32, 2, 64), (1, 600, 600, 16, 64)], ids=str)
def test_attention_f16_blocks_and_wavefronts(gpu, cpu, case):
    """Key counts around the 32-key blocks and what four and eight wavefronts take, sharp and flat soft-maxima, rows of
    Q, K and V that are 16-byte aligned and rows that are not."""
    B, Sq, Sk, H, D = case
    r = rng(sum(case))
    q, k, v = (r.standard_normal((B, S, H * D)).astype(np.float16) for S in (Sq, Sk, Sk))
    for scale in (1.0 / np.sqrt(D), 1.0, 1e-3):
        ref = oc.attention(cpu, q, k, v, H, scale).astype(np.float32)
        np.testing.assert_allclose(oc.attention(gpu, q, k, v, H, scale).astype(np.float32), ref, rtol=2e-3, atol=2e-3)
        wide = [np.zeros((B, S, H * D + 4), np.float16) for S in (Sq, Sk, Sk)]
        for w, t in zip(wide, (q, k, v)):
            w[:, :, :H * D] = t
        Q, K, V = (gpu.put(w) for w in wide)
        Y = gpu.empty((B, Sq, H * D), np.float16)
        gpu.ops.attention(gpu.ptr(Q), gpu.ptr(K), gpu.ptr(V), gpu.ptr(Y), B, Sq, Sk, H, D, float(scale), _abi.F16, ld_in=H * D + 4)
        gpu.sync()
        np.testing.assert_allclose(gpu.get(Y).astype(np.float32), ref, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("case", [(1, 33, 384, 2, 64), (1, 20, 129, 2, 32), (2, 32, 97, 1, 128), (1, 7, 32, 3, 64), (1, 600, 300, 16, 64)], ids=str)
def test_attention_infinities(gpu, cpu, case, dtype):
    """A probability times an infinity is that infinity: an Inf in V, at any key, the last one and a lone one among them,
    gives Inf in its column for every query, opposite ones and NaN give NaN, and the other columns and heads stay."""
    B, Sq, Sk, H, D = case
    r = rng(sum(case))
    q, k, v = (r.standard_normal((B, S, H * D)).astype(dtype) for S in (Sq, Sk, Sk))
    scale = 1.0 / np.sqrt(D)
    plain = oc.attention(gpu, q, k, v, H, scale).astype(np.float32)
    for key in sorted({0, Sk // 2, Sk - 1}):
        vi = v.copy()
        vi[0, key, 3] = np.inf
        vi[0, key, D - 1] = -np.inf
        vi[0, key, 5] = np.nan
        vi[0, key, 7], vi[0, (key + 1) % Sk, 7] = np.inf, -np.inf
        want = plain.copy()
        want[0, :, 3], want[0, :, D - 1], want[0, :, 5], want[0, :, 7] = np.inf, -np.inf, np.nan, np.nan
        np.testing.assert_array_equal(np.isfinite(oc.attention(cpu, q, k, vi, H, scale).astype(np.float32)), np.isfinite(want))
        got = oc.attention(gpu, q, k, vi, H, scale).astype(np.float32)
        np.testing.assert_array_equal(np.where(np.isfinite(got), 0, got), np.where(np.isfinite(want), 0, want))
        fine = np.isfinite(want)
        np.testing.assert_allclose(got[fine], want[fine], rtol=1e-3 if dtype == np.float16 else RTOL, atol=1e-6)  # fp16: one rounding apart


# M, K, N: rows, columns and a reduction off the tiles, the reduction's last step partial, fewer steps than ring stages and
# as many, one more, odd and even counts; split reductions; both tile shapes
@pytest.mark.parametrize("case", [(1, 8, 8), (5, 64, 72), (64, 192, 64), (65, 256, 136), (33, 320, 64), (130, 1000, 328), (16, 3072, 768), (197, 768, 2304),
                                  (100, 384, 3072), (1030, 448, 1160)], ids=str)
def test_matmul_f16_direct_to_lds_tiles(gpu, cpu, case):
    """fp16 products on the direct-to-LDS tiles against the oracle: right operand [K,N] with bias, residual and GELU, twice
    (the arrival counters of split tiles must be back at zero), batched, and stored [N,K]."""
    M, K, N = case
    r = rng(sum(case))
    a = r.standard_normal((1, M, K)).astype(np.float16)
    b = (r.standard_normal((K, N)) / np.sqrt(K)).astype(np.float16)
    bias, z = r.standard_normal(N).astype(np.float16), r.standard_normal((1, M, N)).astype(np.float16)
    exact = a[0].astype(np.float64) @ b.astype(np.float64) + bias.astype(np.float64)
    tol = dict(rtol=2e-3, atol=2e-3)
    got = oc.matmul_nd_bias(gpu, a, b, bias)
    np.testing.assert_allclose(got[0].astype(np.float64), exact, **tol)
    np.testing.assert_array_equal(oc.matmul_nd_bias(gpu, a, b, bias), got)
    np.testing.assert_allclose(oc.matmul_nd_bias(gpu, a, b, bias, z=z)[0].astype(np.float64), exact + z[0], **tol)
    np.testing.assert_allclose(oc.matmul_nd_bias(gpu, a, b, bias, gelu=True).astype(np.float32), oc.matmul_nd_bias(cpu, a, b, bias, gelu=True).astype(np.float32),
                               rtol=1e-2, atol=1e-2)
    np.testing.assert_allclose(oc.matmul2d(gpu, a[0], np.ascontiguousarray(b.T), transB=1, alpha=0.5).astype(np.float64), 0.5 * (exact - bias), **tol)
    if M * K * N < 1 << 22:
        a3, b3 = r.standard_normal((3, M, K)).astype(np.float16), (r.standard_normal((3, K, N)) / np.sqrt(K)).astype(np.float16)
        np.testing.assert_allclose(oc.matmul_nd(gpu, a3, b3).astype(np.float64), a3.astype(np.float64) @ b3.astype(np.float64), **tol)


# The kernel whose wavefronts share the reduction: stages of 32 k for one to four wavefronts, a partial last one, one to many
# stages each, parts of a split; and the tiles it leaves to the other kernel (more than one per compute unit), with fewer
# steps than ring stages, as many, and odd and even counts beyond, on 64x64 and 128x128
@pytest.mark.parametrize("case", [(3, 8, 16), (64, 40, 64), (63, 104, 72), (65, 136, 136), (70, 264, 64), (20, 520, 200), (40, 1288, 64), (129, 6000, 128),
                                  (1100, 64, 1024), (1100, 192, 1024), (1090, 320, 1032), (1100, 392, 1024), (2100, 136, 2056)], ids=str)
@pytest.mark.parametrize("trans_b", [False, True])
def test_matmul_f16_shared_reduction(gpu, case, trans_b):
    """Against 64-bit sums of the same fp16 operands: fp32 sums and one rounding to fp16 (2^-11), whatever the kernel."""
    M, K, N = case
    r = rng(sum(case) + trans_b)
    a, b = r.standard_normal((M, K)).astype(np.float16), (r.standard_normal((K, N)) / np.sqrt(K)).astype(np.float16)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    if trans_b:
        got = oc.matmul2d(gpu, a, np.ascontiguousarray(b.T), transB=1).astype(np.float64)
    else:
        got = oc.matmul_nd_bias(gpu, a[None], b, np.zeros(N, np.float16))[0].astype(np.float64)
    np.testing.assert_allclose(got, exact, rtol=2.0 ** -11, atol=2.0 ** -16)


# both heights of its tiles: rows off them, whole and split reductions, a partial last stage, one to four of its wavefronts without any
@pytest.mark.parametrize("case", [(384, 768, 2304), (383, 808, 2312), (385, 776, 776), (200, 3080, 776), (33, 768, 3080), (31, 1032, 64), (97, 72, 8200)], ids=str)
@pytest.mark.parametrize("trans_b", [False, True])
def test_matmul_f16_shared_reduction_heights(gpu, case, trans_b):
    test_matmul_f16_shared_reduction(gpu, case, trans_b)


# rows and columns off the tiles, one stage of 16 k (three wavefronts without any), a few, odd and even counts, whole tiles
# beside split ones, a handful of split tiles
@pytest.mark.parametrize("case", [(4100, 16, 3104), (1030, 48, 4100), (300, 336, 2052), (161, 1296, 1000), (384, 768, 3072), (128, 3072, 768), (65, 6160, 132)], ids=str)
def test_matmul_f32_shared_reduction(gpu, case):
    """Against 64-bit sums: no further from them than a chain of K fp32 additions (2^-25 sqrt(K) / 2.4 in the 2-norm for
    independent products) and a few roundings; bias, residual and Gelu; twice, the arrival counters must be back at zero."""
    M, K, N = case
    r = rng(sum(case))
    a, b = r.standard_normal((M, K)).astype(np.float32), (r.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
    bias, z = r.standard_normal(N).astype(np.float32), r.standard_normal((1, M, N)).astype(np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64) + bias.astype(np.float64)
    bound = 2.0 ** -25 * (np.sqrt(K) / 2.4 + 4)

    def far(got, want):
        return np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want)
    got = oc.matmul_nd_bias(gpu, a[None], b, bias)
    assert far(got[0], exact) <= bound
    np.testing.assert_array_equal(oc.matmul_nd_bias(gpu, a[None], b, bias), got)
    assert far(oc.matmul_nd_bias(gpu, a[None], b, bias, z=z)[0], exact + z[0]) <= bound
    from scipy.special import erfc
    assert far(oc.matmul_nd_bias(gpu, a[None], b, bias, gelu=True)[0], 0.5 * exact * erfc(-exact / np.sqrt(2))) <= 2 * bound


# where tiles of 32 rows are taken: rows and columns off them, one to three stages a wavefront, whole and split tiles side by side
@pytest.mark.parametrize("case", [(128, 768, 2304), (97, 784, 3076), (100, 3088, 772), (161, 752, 2180), (130, 160, 12292), (520, 16, 16404)], ids=str)
def test_matmul_f32_shared_reduction_of_few_rows(gpu, case):
    test_matmul_f32_shared_reduction(gpu, case)


def test_gelu_epilogue_against_64_bits(gpu):
    """A product with the identity is its left operand, so this is the epilogue's Gelu of chosen values: to 3 units of the last
    place of its argument (the formula's last two roundings and the fits' 2e-9), infinities and NaN as 0.5 x (1 + erf) has them."""
    from scipy.special import erfc
    r = rng(21)
    x = np.concatenate([r.standard_normal(4000) * s for s in (1e-6, 0.05, 0.7, 1.0, 3.0, 20.0)] + [np.linspace(-1.1, 1.1, 575)]).astype(np.float32)
    x = np.concatenate([x, [0.0]]).astype(np.float32).reshape(-1, 64)
    got = oc.matmul_nd_bias(gpu, x[None], np.eye(64, dtype=np.float32), np.zeros(64, np.float32), gelu=True)[0]
    x64 = x.astype(np.float64)
    assert (np.abs(got - 0.5 * x64 * erfc(-x64 / np.sqrt(2))) <= 3 * 2.0 ** -24 * np.abs(x64)).all()


# ---- data movement -------------------------------------------------------------------------

def test_data_movement(gpu, cpu):
    r = rng(16)
    x = r.standard_normal((2, 3, 4, 5)).astype(np.float32)
    np.testing.assert_array_equal(oc.flatten(gpu, x, 1), x.reshape(2, 60))
    np.testing.assert_array_equal(oc.reshape(gpu, x, (6, 20)), x.reshape(6, 20))
    for perm in [(0, 2, 1, 3), (0, 2, 3, 1), (3, 2, 1, 0), (1, 0, 2, 3)]:
        np.testing.assert_array_equal(oc.transpose(gpu, x, perm), x.transpose(perm))
    h = r.standard_normal((1, 128, 12, 64)).astype(np.float32)
    np.testing.assert_array_equal(oc.transpose(gpu, h, (0, 2, 1, 3)), h.transpose(0, 2, 1, 3))
    np.testing.assert_array_equal(oc.transpose(gpu, h, (0, 2, 3, 1)), h.transpose(0, 2, 3, 1))
    np.testing.assert_array_equal(oc.transpose(gpu, x[0], (1, 0, 2)), x[0].transpose(1, 0, 2))
    xi = r.integers(-5, 5, (3, 4)).astype(np.int64)
    np.testing.assert_array_equal(oc.transpose(gpu, xi, (1, 0)), xi.T)
    x6 = r.standard_normal((2, 3, 2, 2, 3, 2)).astype(np.float32)
    np.testing.assert_array_equal(oc.transpose(gpu, x6, (0, 1, 4, 2, 5, 3)), x6.transpose(0, 1, 4, 2, 5, 3))
    table = r.standard_normal((30522, 768)).astype(np.float32)
    idx = r.integers(0, 30522, (1, 128))
    np.testing.assert_array_equal(oc.gather(gpu, table, idx, 0), np.take(table, idx, 0))
    np.testing.assert_array_equal(oc.gather(gpu, x, np.array([2, -1]), 2), np.take(x, [2, -1], 2))
    ti = r.integers(-1000, 1000, (70, 3, 20)).astype(np.int64)
    np.testing.assert_array_equal(oc.gather(gpu, ti, np.array([[6, 0], [3, -2]]), 0), np.take(ti, [[6, 0], [3, -2]], 0))
    np.testing.assert_array_equal(oc.gather(gpu, ti, np.array([19, 1]), 2), oc.gather(cpu, ti, np.array([19, 1]), 2))
    # every permutation of a rank-4 tensor whose dims allow 1-, 2-, 4- and 8-element units, each dtype,
    # plus shapes with size-1 dims and runs of dims that stay together
    import itertools
    for dtype in (np.float32, np.float16, np.int64):
        t = r.integers(-999, 999, (4, 6, 8, 16)).astype(dtype)
        for perm in itertools.permutations(range(4)):
            np.testing.assert_array_equal(oc.transpose(gpu, t, perm), t.transpose(perm))
        for shape, perm in [((2, 1, 8, 4), (2, 1, 0, 3)), ((1, 64, 2, 2, 12, 12), (0, 1, 4, 2, 5, 3)), ((3, 5, 7), (2, 0, 1)),
                            ((2, 3, 4, 5, 6), (0, 3, 4, 1, 2)), ((1, 1, 1), (2, 1, 0)), ((6, 8), (0, 1))]:
            t = r.integers(-999, 999, shape).astype(dtype)
            np.testing.assert_array_equal(oc.transpose(gpu, t, perm), t.transpose(perm))
            np.testing.assert_array_equal(oc.transpose(gpu, t, perm), oc.transpose(cpu, t, perm))
    with pytest.raises(RuntimeError):
        oc.transpose(gpu, x, (0, 1, 1, 3))


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_conv_clipped_and_leaky_relu(gpu, cpu, dtype):
    r = rng(43)
    tol = dict(rtol=1e-4, atol=1e-5) if dtype == np.float32 else dict(rtol=2e-2, atol=2e-3)
    # dense 3x3 and 1x1 (the MFMA kernels), a depthwise 3x3, and a product large enough for the LDS-tiled kernel
    for (N, C, H, K, R, st, pd, grp) in [(1, 64, 14, 64, 3, 1, 1, 1), (2, 32, 9, 48, 1, 1, 0, 1), (1, 32, 12, 32, 3, 2, 1, 32),
                                          (4, 64, 28, 128, 3, 1, 1, 1)]:
        if dtype == np.float16 and grp != 1:
            continue
        x = r.standard_normal((N, C, H, H)).astype(dtype)
        w = (r.standard_normal((K, C // grp, R, R)) * (0.5 / np.sqrt(C // grp * R * R))).astype(dtype)
        b = r.standard_normal(K).astype(dtype)
        P = (H + 2 * pd - R) // st + 1
        z = r.standard_normal((N, K, P, P)).astype(dtype)
        for activ, coef in [(_abi.ACT_CLIPPED_RELU, 0.75), (_abi.ACT_LEAKY_RELU, 0.1)]:
            for zz in (None, z):
                got = oc.conv(gpu, x, w, b, (pd, pd), (st, st), grp, activ, z=zz, coef=coef)
                ref = oc.conv(cpu, x, w, b, (pd, pd), (st, st), grp, activ, z=zz, coef=coef)
                np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), **tol)
                if activ == _abi.ACT_CLIPPED_RELU:
                    assert got.max() <= 0.75 and got.min() >= 0
    x = r.standard_normal((3, 5, 7, 2)).astype(dtype)
    X, Y = gpu.put(x), gpu.empty(x.shape, x.dtype)
    gpu.ops.set_activation_coef(0.25)
    gpu.ops.active(gpu.ptr(X), x.shape, _abi.ACT_LEAKY_RELU, gpu.ptr(Y), oc.DT[np.dtype(dtype)])
    gpu.sync()
    np.testing.assert_array_equal(gpu.get(Y), oc.leaky_relu(cpu, x, 0.25))
    with pytest.raises(RuntimeError):
        oc.conv(gpu, x, np.zeros((4, 5, 1, 1), dtype), np.zeros(4, dtype), activ=4)


def test_leaky_relu_prelu(gpu, cpu):
    r = rng(41)
    for dtype in (np.float32, np.float16):
        for shape in [(2, 24, 13, 13), (1, 64, 56, 56), (5,), (3, 7)]:
            x = r.standard_normal(shape).astype(dtype)
            np.testing.assert_array_equal(oc.leaky_relu(gpu, x, 0.1), oc.leaky_relu(cpu, x, 0.1))
            np.testing.assert_array_equal(oc.prelu(gpu, x, np.array([0.25], dtype)), oc.prelu(cpu, x, np.array([0.25], dtype)))
        x = r.standard_normal((2, 24, 13, 13)).astype(dtype)
        for sshape in [(24, 1, 1), (1, 24, 1, 1), (13,), (2, 24, 13, 13), (1, 1, 13, 1)]:
            sl = r.uniform(-0.5, 0.5, sshape).astype(dtype)
            np.testing.assert_array_equal(oc.prelu(gpu, x, sl), oc.prelu(cpu, x, sl))
    with pytest.raises(RuntimeError):
        oc.prelu(gpu, x, np.ones((7, 1, 1), x.dtype))
    # channels-last: the tensor is a dense [N,H,W,C] array, the slope runs along C
    x = r.standard_normal((2, 24, 5, 7)).astype(np.float16)
    sl = r.uniform(-0.5, 0.5, (24, 1, 1)).astype(np.float16)
    gpu.ops.set_format(_abi.NHWC)
    try:
        X, S = gpu.put(np.ascontiguousarray(x.transpose(0, 2, 3, 1))), gpu.put(sl)
        Y = gpu.empty((2, 5, 7, 24), np.float16)
        gpu.ops.prelu(gpu.ptr(X), gpu.ptr(Y), x.shape, gpu.ptr(S), sl.shape, _abi.F16)
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    np.testing.assert_array_equal(gpu.get(Y).transpose(0, 3, 1, 2), oc.prelu(cpu, x, sl))


def test_concat_squeeze_unsqueeze(gpu, cpu):
    r = rng(42)
    for dtype in (np.float32, np.float16, np.int64):
        mk = (lambda s: r.integers(-99, 99, s).astype(np.int64)) if dtype == np.int64 else (lambda s: r.standard_normal(s).astype(dtype))
        for axis in range(4):
            for sizes in [(1, 3, 7), (4, 4), (8, 16, 8)]:         # element-wise and 16-byte paths
                shapes = []
                for k in sizes:
                    sh = [2, 8, 4, 8]
                    sh[axis] = k
                    shapes.append(sh)
                xs = [mk(s) for s in shapes]
                got = oc.concat(gpu, xs, axis)
                np.testing.assert_array_equal(got, np.concatenate(xs, axis))
                np.testing.assert_array_equal(got, oc.concat(cpu, xs, axis))
    many = [r.standard_normal((3, k + 1, 5)).astype(np.float32) for k in range(16)]
    np.testing.assert_array_equal(oc.concat(gpu, many, 1), np.concatenate(many, 1))
    big = [r.standard_normal((2, c, 52, 52)).astype(np.float32) for c in (128, 256)]  # a detection neck's concat
    np.testing.assert_array_equal(oc.concat(gpu, big, 1), np.concatenate(big, 1))
    with pytest.raises(RuntimeError):
        oc.concat(gpu, many + [many[0]], 1)
    with pytest.raises(RuntimeError):
        oc.concat(gpu, [big[0], big[1][:, :, :50]], 1)
    # channels-last: concatenating channels interleaves per pixel
    xs = [r.standard_normal((2, c, 6, 5)).astype(np.float16) for c in (8, 24, 3)]
    gpu.ops.set_format(_abi.NHWC)
    try:
        Xs = [gpu.put(np.ascontiguousarray(x.transpose(0, 2, 3, 1))) for x in xs]
        Y = gpu.empty((2, 6, 5, 35), np.float16)
        gpu.ops.concat([gpu.ptr(X) for X in Xs], [x.shape for x in xs], gpu.ptr(Y), (2, 35, 6, 5), 1, _abi.F16)
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    np.testing.assert_array_equal(gpu.get(Y).transpose(0, 3, 1, 2), np.concatenate(xs, 1))
    s = r.standard_normal((2, 1, 4, 1)).astype(np.float32)
    np.testing.assert_array_equal(oc.squeeze(gpu, s, (2, 4)), s.reshape(2, 4))
    np.testing.assert_array_equal(oc.squeeze(gpu, s.reshape(2, 4), (1, 2, 1, 4), un=True), s.reshape(1, 2, 1, 4))
    with pytest.raises(RuntimeError):
        oc.squeeze(gpu, s, (4, 2))


def test_expand_and_nonzero(gpu, cpu):
    r = rng(43)
    for shape, out in [((3, 1, 5), (3, 1, 5)), ((3, 1, 5), (2, 3, 4, 5)), ((1,), (1000,)), ((64, 1), (64, 300)),
                       ((1, 1, 1), (2, 3, 4)), ((2, 1, 3, 1, 2), (2, 4, 3, 5, 2)), ((1, 1, 128, 128), (2, 12, 128, 128))]:
        for dtype in (np.int64, np.float32, np.float16):
            x = r.integers(-99, 99, shape).astype(dtype)
            got = oc.expand(gpu, x, out)
            np.testing.assert_array_equal(got, np.broadcast_to(x, out))
            np.testing.assert_array_equal(got, oc.expand(cpu, x, out))
    with pytest.raises(RuntimeError):
        oc.expand(gpu, np.zeros((3, 1, 5), np.int64), (3, 4, 6))
    # sizes around the 1024-element chunk and the 64-lane wavefront, sparse and dense
    for n, density in [(1, 1.0), (63, 0.5), (64, 1.0), (65, 0.3), (1023, 0.9), (1024, 1.0), (1025, 0.01), (5000, 0.5),
                       (100_003, 0.1), (4096, 0.0)]:
        for dtype in (np.float32, np.int64, np.float16):
            x = (r.integers(1, 5, (n,)) * (r.random((n,)) < density)).astype(dtype)
            got = oc.nonzero(gpu, x, (n,), -3)
            want = np.flatnonzero(x)
            np.testing.assert_array_equal(got, oc.nonzero(cpu, x, (n,), -3))
            if dtype != np.float16:  # fp16 cannot hold indices above 2048 exactly: the oracle comparison covers it
                np.testing.assert_array_equal(got[: want.size], want.astype(dtype))
            np.testing.assert_array_equal(got[want.size:], np.full(n - want.size, -3, dtype))
    x = (r.random((7, 9, 11)) < 0.5).astype(np.float32)
    cut = oc.nonzero(gpu, x, (2, 10), -1.0)          # output rank differs from the input's; capacity 20
    np.testing.assert_array_equal(cut.reshape(-1), np.flatnonzero(x.reshape(-1))[:20].astype(np.float32))
    z = np.array([0.0, -0.0, np.nan, 1e-45, 0.0], np.float32)
    np.testing.assert_array_equal(oc.nonzero(gpu, z, (5,), -1.0), np.array([2, 3, -1, -1, -1], np.float32))


def test_empty_tensors_are_no_ops(gpu, cpu):
    # an empty batch (or an empty tensor of any kind) launches nothing, writes nothing, raises nothing,
    # and leaves no error behind; the oracle agrees entry point by entry point
    got = oc.empty_tensor_behaviour(gpu)
    assert got == oc.empty_tensor_behaviour(cpu)
    assert set(got.values()) == {"untouched"}, got


# ---- fp16, channels-last -----------------------------------------------------------------

def conv_f16(gpu, x, w, b, pads, strides, group, activ, fmt, z=None, inplace=False):
    """x, w (and the residual z) in logical NCHW / KCRS order; returns logical NCHW.  inplace: the result buffer
    holds z and is passed as both Z and Y."""
    N, C, H, W = x.shape
    K, Cg, R, S = w.shape
    P, Q = oc.conv_out_hw(H, W, R, S, pads, strides)
    xin = x if fmt != _abi.NHWC else np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    win = w if fmt == _abi.NCHW else np.ascontiguousarray(w.transpose(0, 2, 3, 1))  # K,R,S,C
    X, Wt, B = gpu.put(xin), gpu.put(win), gpu.put(b)
    Y = gpu.empty((N * K * P * Q,), np.float16)
    gpu.ops.set_format(fmt)
    try:
        if z is None:
            gpu.ops.conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), pads, strides, activ,
                                    gpu.ptr(Y), group, _abi.F16)
        else:  # laid out like Y
            Z = gpu.put(z if fmt == _abi.NCHW else np.ascontiguousarray(z.transpose(0, 2, 3, 1)))
            if inplace:
                Y = Z
            gpu.ops.conv_bias_add_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), gpu.ptr(Z), pads, strides,
                                        activ, gpu.ptr(Y), group, _abi.F16)
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    y = gpu.get(Y)
    return y.reshape(N, K, P, Q) if fmt == _abi.NCHW else y.reshape(N, P, Q, K).transpose(0, 3, 1, 2)


F16_CASES = [
    # N, C, H, W, K, R, stride, pad
    (2, 64, 56, 56, 64, 3, 1, 1),      # fast path, K_out = 64 tile
    (2, 64, 56, 56, 256, 1, 1, 0),
    (2, 256, 28, 28, 128, 3, 2, 1),    # strided 3x3
    (3, 512, 7, 7, 512, 3, 1, 1),      # ragged pixel tile (147 pixels)
    (2, 256, 14, 14, 1000, 1, 1, 0),   # K_out not a multiple of the tile
    (1, 1024, 14, 14, 2048, 1, 2, 0),
    (2, 32, 9, 11, 40, 3, 1, 1),       # smallest C the fast path takes
    (2, 64, 9, 11, 40, 3, 1, 1),       # 64 x 128 tile, ragged in both directions
    (2, 64, 9, 11, 40, 1, 1, 0),       # one-step reduction (single LDS stage), ragged in both directions
    (1, 64, 12, 12, 72, 1, 2, 0),      # the same with stride 2 and two k_out tiles
    (2, 128, 9, 11, 40, 1, 1, 0),      # two, three and four steps taking turns in the one LDS stage
    (1, 192, 10, 7, 72, 1, 1, 0),
    (2, 256, 7, 7, 136, 1, 1, 0),
    (64, 2048, 1, 1, 1000, 1, 1, 0),   # few pixels (a fully connected layer): 16 filters x 32 pixels per workgroup
    (1, 512, 1, 1, 1000, 1, 1, 0),     # the same with one pixel
    (3, 320, 3, 5, 72, 1, 1, 0),       # 45 pixels, five chunks over four wavefronts, half a block of filters
    (1, 1088, 7, 7, 24, 1, 1, 0),      # 49 pixels, 17 chunks
    (2, 3, 32, 32, 64, 7, 2, 3),       # 3 channels: first-layer kernel (NCHW in, NHWC out), generic otherwise
    (2, 3, 45, 37, 64, 7, 2, 3),       # first-layer kernel, ragged tiles (23 x 19 output pixels)
    (1, 3, 224, 224, 64, 7, 2, 3),     # the ResNet first layer at full size
    (1, 20, 9, 9, 24, 3, 1, 1),        # generic path: C % 32 != 0
    # channels-last 1x1 layers over a multiple of 8 channels that is not one of 64: one wavefront per 32 pixels
    (2, 16, 20, 20, 96, 1, 1, 0),      # one 16-channel step
    (3, 24, 9, 11, 144, 1, 1, 0),      # half of the second step is past the channels; 297 pixels: a ragged last wavefront
    (2, 144, 7, 9, 24, 1, 1, 0),       # nine steps, fewer filters than a block
    (1, 160, 7, 7, 960, 1, 1, 0),      # 49 pixels: the filter blocks are dealt over the grid
    (5, 8, 3, 3, 8, 1, 1, 0),          # the smallest
    (1, 248, 6, 5, 40, 1, 1, 0),       # sixteen steps, the last one half empty
    (1, 200, 9, 9, 72, 1, 1, 0),
    (8, 24, 56, 56, 144, 1, 1, 0),     # a MobileNetV2 expansion layer
    # first layers other than the 7x7 one (N,C,H,W in, channels-last out): a thread per output pixel
    (2, 3, 33, 30, 32, 3, 2, 1),       # MobileNetV2's, on a ragged image
    (1, 3, 224, 224, 32, 3, 2, 1),     # ... at full size
    (2, 3, 20, 17, 64, 3, 1, 1),       # a VGG's
    (3, 1, 12, 12, 16, 3, 1, 0),       # one channel, no padding
    (2, 4, 9, 9, 24, 1, 1, 0),         # four channels, 1x1
    (1, 2, 10, 11, 48, 2, 2, 1),       # 2x2 filter
]


@pytest.mark.parametrize("case", F16_CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("fmt", [_abi.NHWC, _abi.NCHW_TO_NHWC, _abi.NCHW])
def test_conv_f16(gpu, cpu, case, fmt):
    N, C, H, W, K, R, st, pd = case
    r = rng(sum(case) + fmt)
    x = r.standard_normal((N, C, H, W)).astype(np.float16)
    w = (r.standard_normal((K, C, R, R)) * np.sqrt(2.0 / (C * R * R))).astype(np.float16)
    b = r.uniform(-0.1, 0.1, K).astype(np.float16)
    ref = oc.conv(cpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_RELU)          # fp16 storage, exact accumulate
    got = conv_f16(gpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_RELU, fmt)
    # fp32 accumulation then one rounding to fp16: within 1 fp16 ulp of the oracle
    np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3)
    if fmt == _abi.NHWC:
        ident = conv_f16(gpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_IDENTITY, fmt)
        refi = oc.conv(cpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_IDENTITY)
        np.testing.assert_allclose(ident.astype(np.float32), refi.astype(np.float32), rtol=2e-3, atol=2e-3)
    z = r.standard_normal(ref.shape).astype(np.float16)
    refz = oc.conv(cpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_RELU, z=z)
    gotz = conv_f16(gpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_RELU, fmt, z=z)
    np.testing.assert_allclose(gotz.astype(np.float32), refz.astype(np.float32), rtol=4e-3, atol=4e-3)
    if fmt != _abi.NCHW_TO_NHWC:  # written over the residual operand: the same bits
        np.testing.assert_array_equal(conv_f16(gpu, x, w, b, (pd, pd), (st, st), 1, _abi.ACT_RELU, fmt, z=z, inplace=True), gotz)


# N, C, H, W, K, R, S, stride, pad: one, two and three steps of 16 taps; every number of filters; images of less than 32 pixels, of
# no multiple of 32 and of several runs of 32 a wavefront; filters that are not square, windows past every border
@pytest.mark.parametrize("case", [(2, 3, 37, 53, 32, 3, 3, (2, 2), (1, 1)), (1, 4, 20, 19, 64, 3, 3, (1, 1), (2, 2)), (5, 3, 5, 5, 24, 3, 3, (1, 1), (1, 1)),
                                  (2, 1, 9, 40, 16, 1, 3, (1, 2), (0, 1)), (1, 2, 33, 9, 48, 3, 2, (3, 1), (2, 1)), (1, 4, 8, 8, 32, 2, 2, (2, 2), (0, 0)),
                                  (70, 3, 64, 96, 32, 3, 3, (2, 2), (1, 1)), (3, 3, 1, 1, 64, 3, 3, (1, 1), (1, 1))], ids=lambda c: "x".join(map(str, c[:7])))
@pytest.mark.parametrize("activ", [_abi.ACT_IDENTITY, _abi.ACT_RELU])
def test_conv_f16_first_layers(gpu, cpu, case, activ):
    """Against 64-bit sums: the fp32 additions, at most 2^-24 of the sum of magnitudes each, and one rounding to fp16 (two with a
    residual operand); infinities and NaN only where a window holds them."""
    import torch
    N, C, H, W, K, R, S, st, pd = case
    r = rng(N + H + W + K)
    x = r.standard_normal((N, C, H, W)).astype(np.float16)
    w = (r.standard_normal((K, C, R, S)) * np.sqrt(2.0 / (C * R * S))).astype(np.float16)
    b = r.uniform(-0.3, 0.3, K).astype(np.float16)
    conv64 = lambda t, f, v: torch.nn.functional.conv2d(*(torch.from_numpy(u).double() for u in (t, f, v)), stride=st, padding=pd).numpy()  # noqa: E731
    act = (lambda t: np.maximum(t, 0)) if activ == _abi.ACT_RELU else (lambda t: t)
    ref, magnitude = conv64(x, w, b), conv64(np.abs(x), np.abs(w), np.abs(b))
    exact = (C * R * S + 2) * 2.0 ** -24 * magnitude
    got = conv_f16(gpu, x, w, b, pd, st, 1, activ, _abi.NCHW_TO_NHWC).astype(np.float64)
    assert (np.abs(got - act(ref)) <= exact + 2.0 ** -11 * (np.abs(ref) + exact) + 2.0 ** -25).all()
    z = r.standard_normal(ref.shape).astype(np.float16)
    got = conv_f16(gpu, x, w, b, pd, st, 1, activ, _abi.NCHW_TO_NHWC, z=z)
    twice = exact + 2.0 ** -11 * (np.abs(ref) + exact) + 2.0 ** -25
    assert (np.abs(got - act(ref + z)) <= twice + 2.0 ** -11 * (np.abs(ref + z) + twice) + 2.0 ** -25).all()
    x[0, C - 1, H // 2, W // 3] = np.nan
    x[N - 1, 0, H - 1, W - 1] = -np.inf
    got, ref = conv_f16(gpu, x, w, b, pd, st, 1, _abi.ACT_IDENTITY, _abi.NCHW_TO_NHWC), oc.conv(cpu, x, w, b, pd, st, 1, _abi.ACT_IDENTITY)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    assert np.isfinite(got[np.isfinite(ref)]).all()


@pytest.mark.parametrize("case", [(2, 32, 14, 14, 32, 3, 1, 1, 32), (1, 96, 28, 28, 96, 3, 2, 1, 96), (2, 6, 7, 7, 12, 3, 1, 1, 6),
                                  (1, 16, 10, 10, 32, 3, 1, 1, 4), (2, 128, 9, 9, 128, 1, 1, 0, 2), (3, 144, 13, 9, 144, 3, 2, 1, 144),
                                  (1, 960, 7, 7, 960, 3, 1, 1, 960), (2, 24, 9, 9, 24, 5, 1, 2, 24), (1, 12, 6, 6, 12, 3, 1, 1, 12)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("fmt", [_abi.NHWC, _abi.NCHW])
def test_conv_f16_grouped_and_depthwise(gpu, cpu, case, fmt):
    """fp16 convolutions with groups (depthwise: the channels-last kernel of its own for channel counts that are
    multiples of eight, MobileNetV2's shapes among them, the generic kernel otherwise; depthwise with a channel
    multiplier; a few wide groups), with bias, ReLU and a residual operand, channels-last and N,C,H,W, against the
    oracle to the fp16 convolution tolerance."""
    N, C, H, W, K, R, st, pd, grp = case
    r = rng(sum(case) + fmt)
    x = r.standard_normal((N, C, H, W)).astype(np.float16)
    w = (r.standard_normal((K, C // grp, R, R)) * np.sqrt(2.0 / (C // grp * R * R))).astype(np.float16)
    b = r.uniform(-0.1, 0.1, K).astype(np.float16)
    ref = oc.conv(cpu, x, w, b, (pd, pd), (st, st), grp, _abi.ACT_RELU)
    got = conv_f16(gpu, x, w, b, (pd, pd), (st, st), grp, _abi.ACT_RELU, fmt)
    np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3)
    z = r.standard_normal(ref.shape).astype(np.float16)
    refz = oc.conv(cpu, x, w, b, (pd, pd), (st, st), grp, _abi.ACT_RELU, z=z)
    gotz = conv_f16(gpu, x, w, b, (pd, pd), (st, st), grp, _abi.ACT_RELU, fmt, z=z)
    np.testing.assert_allclose(gotz.astype(np.float32), refz.astype(np.float32), rtol=4e-3, atol=4e-3)
    np.testing.assert_array_equal(conv_f16(gpu, x, w, b, (pd, pd), (st, st), grp, _abi.ACT_RELU, fmt, z=z, inplace=True), gotz)


def stem_pool_f16(gpu, x, w, b, activ, fmt=_abi.NCHW_TO_NHWC, kernel=(3, 3), ppads=(1, 1, 1, 1), pstrides=(2, 2)):
    """The fused first layer through the C-ABI; x in N,C,H,W, w logical K,C,R,S; returns logical N,K,PP,QQ."""
    N, C, H, W = x.shape
    K = w.shape[0]
    P, Q = oc.conv_out_hw(H, W, 7, 7, (3, 3), (2, 2))
    PP, QQ = oc.conv_out_hw(P, Q, 3, 3, (1, 1), (2, 2))
    X, Wt, B = gpu.put(x), gpu.put(np.ascontiguousarray(w.transpose(0, 2, 3, 1))), gpu.put(b)
    Y = gpu.empty((N * K * PP * QQ,), np.float16)
    gpu.ops.set_format(fmt)
    try:
        gpu.ops.conv_bias_activ_max_pool(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (3, 3), (2, 2), activ, kernel,
                                         ppads, pstrides, gpu.ptr(Y), (N, K, PP, QQ))
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    return gpu.get(Y).reshape(N, PP, QQ, K).transpose(0, 3, 1, 2)


@pytest.mark.parametrize("case", [(2, 32, 32), (2, 45, 38), (3, 64, 80), (1, 224, 224), (5, 23, 62), (70, 16, 16), (1, 7, 2)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("activ", [_abi.ACT_RELU, _abi.ACT_IDENTITY])
def test_first_layer_with_its_max_pool_in_one_call(gpu, cpu, case, activ):
    """dnnrtConvBiasActivMaxPool against the two calls it replaces: the oracle's chain to the convolution's
    tolerance (one rounding to fp16 of an fp32 sum; the maximum adds none), and this library's own two calls
    bit for bit (same products in the same order, then an exact maximum).  Identity activation leaves negative
    values, so a padding of zeros instead of -inf would show; odd heights and widths that are not multiples of 28
    leave ragged strips and a last pooled row and column whose windows hang over the edge."""
    N, H, W = case
    r = rng(N + H + W + activ)
    x = r.standard_normal((N, 3, H, W)).astype(np.float16)
    w = (r.standard_normal((64, 3, 7, 7)) * np.sqrt(2.0 / 147)).astype(np.float16)
    b = r.uniform(-0.5, 0.1, 64).astype(np.float16)
    if case == (5, 23, 62):
        x[1, 2, 11, 30] = np.nan  # reaches a 4 x 4 block of convolution outputs of image 1, every channel
        x[3, 0, 5, 40] = np.inf   # infinities of both signs in one window's reach: inf - inf is a NaN as well,
        x[3, 1, 6, 41] = -np.inf  # and around it results of +inf and -inf
    got = stem_pool_f16(gpu, x, w, b, activ)
    conv_ref = oc.conv(cpu, x, w, b, (3, 3), (2, 2), 1, activ)
    ref = oc.pool(cpu, "max", conv_ref, (3, 3), (1, 1), (2, 2))
    assert got.shape == ref.shape
    np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3)
    if case == (5, 23, 62):
        assert np.isnan(got[1]).any() and np.isnan(got[3]).any() and not np.isnan(got[[0, 2, 4]]).any()
        assert (np.isnan(got) == np.isnan(ref)).all()
    # the two calls on the GPU, channels-last in between
    conv_gpu = conv_f16(gpu, x, w, b, (3, 3), (2, 2), 1, activ, _abi.NCHW_TO_NHWC)       # logical NCHW
    mid = gpu.put(np.ascontiguousarray(conv_gpu.transpose(0, 2, 3, 1)))
    P, Q = conv_gpu.shape[2:]
    PP, QQ = ref.shape[2:]
    Y2 = gpu.empty((N * 64 * PP * QQ,), np.float16)
    gpu.ops.set_format(_abi.NHWC)
    try:
        gpu.ops.maxpool(gpu.ptr(mid), (N, 64, P, Q), gpu.ptr(Y2), (N, 64, PP, QQ), (3, 3), (1, 1, 1, 1), (2, 2), _abi.F16)
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    two = gpu.get(Y2).reshape(N, PP, QQ, 64).transpose(0, 3, 1, 2)
    np.testing.assert_array_equal(got, two)


def test_first_layer_with_its_max_pool_refuses_other_shapes(gpu):
    r = rng(3)
    x = r.standard_normal((1, 3, 32, 32)).astype(np.float16)
    w = r.standard_normal((64, 3, 7, 7)).astype(np.float16)
    b = np.zeros(64, np.float16)
    for kw, word in ((dict(fmt=_abi.NHWC), "NCHW_TO_NHWC"), (dict(kernel=(2, 2)), "3x3"), (dict(pstrides=(1, 1)), "stride 2"),
                     (dict(ppads=(0, 0, 0, 0)), "pad 1")):
        with pytest.raises(RuntimeError, match=word):
            stem_pool_f16(gpu, x, w, b, _abi.ACT_RELU, **kw)
    with pytest.raises(RuntimeError, match="even width"):
        stem_pool_f16(gpu, r.standard_normal((1, 3, 32, 33)).astype(np.float16), w, b, _abi.ACT_RELU)
    with pytest.raises(RuntimeError, match="7x7"):
        w5 = r.standard_normal((64, 3, 5, 5)).astype(np.float16)
        X, Wt, B = gpu.put(x), gpu.put(np.ascontiguousarray(w5.transpose(0, 2, 3, 1))), gpu.put(b)
        Y = gpu.empty((64 * 8 * 8,), np.float16)
        gpu.ops.set_format(_abi.NCHW_TO_NHWC)
        try:
            gpu.ops.conv_bias_activ_max_pool(gpu.ptr(X), x.shape, gpu.ptr(Wt), w5.shape, gpu.ptr(B), (2, 2), (2, 2), _abi.ACT_RELU,
                                             (3, 3), (1, 1, 1, 1), (2, 2), gpu.ptr(Y), (1, 64, 8, 8))
        finally:
            gpu.ops.set_format(_abi.NCHW)


@pytest.mark.parametrize("case", [(1, 224, 224), (2, 64, 64), (3, 37, 51), (1, 9, 9), (2, 30, 61)], ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("crsk", [False, True])
@pytest.mark.parametrize("activ", [_abi.ACT_RELU, _abi.ACT_IDENTITY])
def test_first_layer_fp32_alone_and_with_its_max_pool(gpu, cpu, case, crsk, activ):
    """The fp32 N,C,H,W first layer (3 -> 64 channels, 7x7, stride 2, pad 3) through dnnrtConvBiasActiv and, with the
    3x3 stride-2 pooling behind it, through dnnrtConvBiasActivMaxPool, against the oracle's convolution and its chain:
    rtol 1e-4, atol 1e-5 as for every fp32 convolution (the maximum adds no rounding).  Both filter layouts; the
    benchmark's size, odd sizes with ragged tiles in both directions, an image smaller than one tile; identity
    activation leaves negative values, so a padding of zeros instead of -inf would show."""
    N, H, W = case
    r = rng(N + H + W + activ)
    x = r.standard_normal((N, 3, H, W)).astype(np.float32)
    w = (r.standard_normal((64, 3, 7, 7)) * np.sqrt(2.0 / 147)).astype(np.float32)
    b = r.uniform(-0.5, 0.1, 64).astype(np.float32)
    if case == (3, 37, 51):
        x[1, 2, 11, 30] = np.nan
        x[2, 0, 5, 40] = np.inf
        x[2, 1, 6, 41] = -np.inf
    conv_ref = oc.conv(cpu, x, w, b, (3, 3), (2, 2), 1, activ)
    ref = oc.pool(cpu, "max", conv_ref, (3, 3), (1, 1), (2, 2))
    lay = (lambda t: np.ascontiguousarray(t.transpose(1, 2, 3, 0))) if crsk else (lambda t: t)
    X, Wt, B = gpu.put(x), gpu.put(lay(w)), gpu.put(b)
    Yc, Yp = gpu.empty(conv_ref.shape, np.float32), gpu.empty(ref.shape, np.float32)
    gpu.ops.set_filter_layout(_abi.FILTER_CRSK if crsk else _abi.FILTER_KCRS)
    try:
        gpu.ops.conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (3, 3), (2, 2), activ, gpu.ptr(Yc))
        gpu.ops.conv_bias_activ_max_pool(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (3, 3), (2, 2), activ,
                                         (3, 3), (1, 1, 1, 1), (2, 2), gpu.ptr(Yp), ref.shape, dtype=_abi.F32)
        gpu.sync()
    finally:
        gpu.ops.set_filter_layout(_abi.FILTER_KCRS)
    got_c, got = gpu.get(Yc), gpu.get(Yp)
    finite = np.isfinite(conv_ref)
    assert (np.isnan(got_c) == np.isnan(conv_ref)).all() and (np.isnan(got) == np.isnan(ref)).all()
    np.testing.assert_allclose(got_c[finite], conv_ref[finite], rtol=1e-4, atol=1e-5)
    np.testing.assert_array_equal(got_c[~finite & ~np.isnan(conv_ref)], conv_ref[~finite & ~np.isnan(conv_ref)])
    np.testing.assert_allclose(got, ref, rtol=1e-4, atol=1e-5)
    if case == (3, 37, 51):
        assert np.isnan(got[1]).any() and np.isnan(got[2]).any() and not np.isnan(got[0]).any()
    # the pooled result is the exact maximum of this library's own convolution
    Y2 = gpu.empty(ref.shape, np.float32)
    gpu.ops.maxpool(gpu.ptr(Yc), conv_ref.shape, gpu.ptr(Y2), ref.shape, (3, 3), (1, 1, 1, 1), (2, 2), _abi.F32)
    gpu.sync()
    np.testing.assert_array_equal(got, gpu.get(Y2))


# batches of many tiles, where workgroups walk down columns of tiles: one walk a column and several, walks that end in a
# partial step, one-row and one-column edges, images of one step
@pytest.mark.parametrize("case", [(32, 224, 224), (9, 130, 97), (40, 21, 230), (130, 8, 8), (3, 300, 300), (2, 448, 448)], ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("pool", [False, True])
def test_first_layer_fp32_in_walks(gpu, case, pool):
    """Against 64-bit sums: 148 additions, each rounding by at most 2^-24 of the sum of magnitudes (a maximum adds none); a NaN
    reaches the windows that hold it and no others."""
    import torch
    N, H, W = case
    g = torch.Generator().manual_seed(H)
    x, w = torch.randn(N, 3, H, W, generator=g), torch.randn(64, 3, 7, 7, generator=g) * (2.0 / 147) ** 0.5
    b = torch.rand(64, generator=g) * 0.6 - 0.5
    x[N // 2, 1, H // 2, W // 3] = float("nan")
    X, Wt, B = gpu.put(x.numpy()), gpu.put(w.numpy()), gpu.put(b.numpy())
    P, Q = (H - 1) // 2 + 1, (W - 1) // 2 + 1
    shape = (N, 64, (P - 1) // 2 + 1, (Q - 1) // 2 + 1) if pool else (N, 64, P, Q)
    Y = gpu.empty(shape, np.float32)
    if pool:
        gpu.ops.conv_bias_activ_max_pool(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (3, 3), (2, 2), _abi.ACT_IDENTITY,
                                         (3, 3), (1, 1, 1, 1), (2, 2), gpu.ptr(Y), shape, dtype=_abi.F32)
    else:
        gpu.ops.conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (3, 3), (2, 2), _abi.ACT_IDENTITY, gpu.ptr(Y))
    gpu.sync()
    got = torch.from_numpy(gpu.get(Y))
    for n in sorted({0, N // 2, N - 1}):
        ref = torch.nn.functional.conv2d(x[n:n + 1].double(), w.double(), b.double(), stride=2, padding=3)
        bound = 148 * 2.0 ** -24 * torch.nn.functional.conv2d(x[n:n + 1].nan_to_num().abs().double(), w.abs().double(), b.abs().double(), stride=2, padding=3)
        if pool:
            nan = torch.nn.functional.max_pool2d(ref.isnan().float(), 3, 2, 1) > 0
            ref, bound = torch.nn.functional.max_pool2d(ref.nan_to_num(nan=-1e30), 3, 2, 1), torch.nn.functional.max_pool2d(bound, 3, 2, 1)
            ref[nan] = float("nan")
        assert (got[n].isnan() == ref[0].isnan()).all()
        ok = ~ref[0].isnan()
        assert ((got[n] - ref[0]).abs()[ok] <= bound[0][ok]).all()


def test_first_layer_fp32_with_its_max_pool_refuses_other_shapes(gpu):
    r = rng(4)
    x = r.standard_normal((1, 3, 32, 32)).astype(np.float32)
    b = np.zeros(64, np.float32)
    X, B = gpu.put(x), gpu.put(b)
    Y = gpu.empty((64 * 8 * 8,), np.float32)
    w5 = r.standard_normal((64, 3, 5, 5)).astype(np.float32)
    with pytest.raises(RuntimeError, match="7x7"):
        gpu.ops.conv_bias_activ_max_pool(gpu.ptr(X), x.shape, gpu.ptr(gpu.put(w5)), w5.shape, gpu.ptr(B), (2, 2), (2, 2), _abi.ACT_RELU,
                                         (3, 3), (1, 1, 1, 1), (2, 2), gpu.ptr(Y), (1, 64, 8, 8), dtype=_abi.F32)
    w7 = r.standard_normal((64, 3, 7, 7)).astype(np.float32)
    with pytest.raises(RuntimeError, match="ReLU or identity"):
        gpu.ops.conv_bias_activ_max_pool(gpu.ptr(X), x.shape, gpu.ptr(gpu.put(w7)), w7.shape, gpu.ptr(B), (3, 3), (2, 2), _abi.ACT_LEAKY_RELU,
                                         (3, 3), (1, 1, 1, 1), (2, 2), gpu.ptr(Y), (1, 64, 8, 8), dtype=_abi.F32)


def dual_conv_f16(gpu, x, w, b, x2, w2, b2, stride2, activ, algo=0):
    """dnnrtConvBiasAddConvBiasActiv through the C-ABI; tensors in logical NCHW / KCRS order; returns logical NCHW."""
    N, C, P, Q = x.shape
    K = w.shape[0]
    nhwc = lambda t: np.ascontiguousarray(t.transpose(0, 2, 3, 1))  # noqa: E731
    X, Wt, B, X2, Wt2, B2 = gpu.put(nhwc(x)), gpu.put(nhwc(w)), gpu.put(b), gpu.put(nhwc(x2)), gpu.put(nhwc(w2)), gpu.put(b2)
    Y = gpu.empty((N * K * P * Q,), np.float16)
    gpu.ops.set_format(_abi.NHWC)
    try:
        gpu.ops.conv_bias_add_conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (0, 0), (1, 1), gpu.ptr(X2), x2.shape,
                                              gpu.ptr(Wt2), w2.shape, gpu.ptr(B2), (0, 0), (stride2, stride2), activ, gpu.ptr(Y),
                                              algo=algo)
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    return gpu.get(Y).reshape(N, P, Q, K).transpose(0, 3, 1, 2)


@pytest.mark.parametrize("case", [(2, 9, 11, 64, 64, 72, 1), (3, 13, 13, 128, 256, 200, 2), (2, 14, 10, 192, 128, 256, 2), (8, 56, 56, 64, 64, 256, 1), (4, 56, 56, 128, 256, 512, 2), (3, 9, 13, 128, 256, 136, 2), (2, 10, 10, 128, 128, 72, 1), (2, 12, 12, 64, 256, 64, 2), (1, 9, 9, 192, 256, 40, 1),
                                  (1, 7, 7, 64, 128, 64, 1)], ids=lambda c: "x".join(map(str, c)))
def test_last_convolution_and_projection_shortcut_in_one_call(gpu, cpu, case):
    """dnnrtConvBiasAddConvBiasActiv against the two calls it replaces: the oracle's chain to the fp16 convolutions'
    tolerance.  N, H2, W2, C, C2, K, stride of the shortcut; ragged tiles in both directions.  64 + 64 and 128 + 256
    channels take the kernel that gives this library's own two calls bit for bit (each conv + bias rounded to fp16 on
    its own, the sum and ReLU in fp32); other multiples of 64 take one reduction over both convolutions' channels,
    rounded once, which is as close to the oracle as the two calls are but not their bits."""
    N, H2, W2, C, C2, K, st = case
    P, Q = (H2 - 1) // st + 1, (W2 - 1) // st + 1
    r = rng(sum(case))
    x = r.standard_normal((N, C, P, Q)).astype(np.float16)
    x2 = r.standard_normal((N, C2, H2, W2)).astype(np.float16)
    w = (r.standard_normal((K, C, 1, 1)) * np.sqrt(2.0 / C)).astype(np.float16)
    w2 = (r.standard_normal((K, C2, 1, 1)) * np.sqrt(2.0 / C2)).astype(np.float16)
    b, b2 = r.uniform(-0.2, 0.2, K).astype(np.float16), r.uniform(-0.2, 0.2, K).astype(np.float16)
    got = dual_conv_f16(gpu, x, w, b, x2, w2, b2, st, _abi.ACT_RELU)
    z_ref = oc.conv(cpu, x2, w2, b2, (0, 0), (st, st), 1, _abi.ACT_IDENTITY)
    ref = oc.conv(cpu, x, w, b, (0, 0), (1, 1), 1, _abi.ACT_RELU, z=z_ref)
    np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=4e-3, atol=4e-3)
    z_gpu = conv_f16(gpu, x2, w2, b2, (0, 0), (st, st), 1, _abi.ACT_IDENTITY, _abi.NHWC)
    two = conv_f16(gpu, x, w, b, (0, 0), (1, 1), 1, _abi.ACT_RELU, _abi.NHWC, z=z_gpu)
    if (C, C2) in ((64, 64), (128, 256)):
        np.testing.assert_array_equal(got, two)
    else:
        np.testing.assert_allclose(got.astype(np.float32), two.astype(np.float32), rtol=4e-3, atol=4e-3)
    if case[0] == 2 and C == 64:  # the oracle's own entry point is that chain
        X, Wt, B, X2, Wt2, B2 = cpu.put(x), cpu.put(w), cpu.put(b), cpu.put(x2), cpu.put(w2), cpu.put(b2)
        Y = cpu.empty(ref.shape, np.float16)
        cpu.ops.conv_bias_add_conv_bias_activ(cpu.ptr(X), x.shape, cpu.ptr(Wt), w.shape, cpu.ptr(B), (0, 0), (1, 1), cpu.ptr(X2), x2.shape,
                                              cpu.ptr(Wt2), w2.shape, cpu.ptr(B2), (0, 0), (st, st), _abi.ACT_RELU, cpu.ptr(Y))
        np.testing.assert_array_equal(cpu.get(Y), ref)


@pytest.mark.parametrize("case", [(64, 28, 28, 256, 512, 1024, 2), (64, 14, 14, 512, 1024, 2048, 2), (3, 13, 13, 128, 256, 200, 2),
                                  (2, 14, 10, 192, 128, 256, 2), (5, 9, 13, 64, 64, 136, 1)], ids=lambda c: "x".join(map(str, c)))
def test_shortcut_pair_as_one_reduction_every_variant(gpu, cpu, case):
    """The one-reduction form of dnnrtConvBiasAddConvBiasActiv on every tile variant it is compiled in, asked for
    through the call's `algo` operand (DNNRT_CONV_ALGO_BASE + id), ResNet-50's two long pairs at batch 64 among the
    cases and the short pairs too (which take this form only when asked): the oracle's chain to the fp16
    convolutions' tolerance."""
    N, H2, W2, C, C2, K, st = case
    P, Q = (H2 - 1) // st + 1, (W2 - 1) // st + 1
    r = rng(sum(case) + 1)
    x = r.standard_normal((N, C, P, Q)).astype(np.float16)
    x2 = r.standard_normal((N, C2, H2, W2)).astype(np.float16)
    w = (r.standard_normal((K, C, 1, 1)) * np.sqrt(2.0 / C)).astype(np.float16)
    w2 = (r.standard_normal((K, C2, 1, 1)) * np.sqrt(2.0 / C2)).astype(np.float16)
    b, b2 = r.uniform(-0.2, 0.2, K).astype(np.float16), r.uniform(-0.2, 0.2, K).astype(np.float16)
    z_ref = oc.conv(cpu, x2, w2, b2, (0, 0), (st, st), 1, _abi.ACT_IDENTITY)
    ref = oc.conv(cpu, x, w, b, (0, 0), (1, 1), 1, _abi.ACT_RELU, z=z_ref).astype(np.float32)
    for vid in (33, 37, 39, 61, 64, 66):
        got = dual_conv_f16(gpu, x, w, b, x2, w2, b2, st, _abi.ACT_RELU, algo=_abi.CONV_ALGO_BASE + vid)
        np.testing.assert_allclose(got.astype(np.float32), ref, rtol=4e-3, atol=4e-3, err_msg=f"variant {vid}")


@pytest.mark.parametrize("case", [(1, 56, 56, 64, 64, 256, 1), (1, 56, 56, 128, 256, 512, 2), (1, 28, 28, 256, 512, 1024, 2),
                                  (1, 14, 14, 512, 1024, 2048, 2), (2, 9, 11, 24, 40, 72, 1), (16, 28, 28, 128, 256, 512, 2)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("crsk", [False, True])
def test_last_convolution_and_projection_shortcut_fp32(gpu, cpu, case, crsk):
    """The same call on fp32 N,C,H,W tensors with both filter layouts: ResNet-50's four shortcut pairs at batch 1 (one
    launch of the small 1x1 kernel, the second reduction appended to the first: one rounding of the whole sum where the
    chain has three), an odd-sized pair and a batch-16 pair (the two convolutions one after the other through Y: the
    chain's bits).  Against the oracle's chain: rtol 1e-4, atol 1e-5 as for every fp32 convolution."""
    N, H2, W2, C, C2, K, st = case
    P, Q = (H2 - 1) // st + 1, (W2 - 1) // st + 1
    r = rng(sum(case))
    x = r.standard_normal((N, C, P, Q)).astype(np.float32)
    x2 = r.standard_normal((N, C2, H2, W2)).astype(np.float32)
    w = (r.standard_normal((K, C, 1, 1)) * np.sqrt(2.0 / C)).astype(np.float32)
    w2 = (r.standard_normal((K, C2, 1, 1)) * np.sqrt(2.0 / C2)).astype(np.float32)
    b, b2 = r.uniform(-0.2, 0.2, K).astype(np.float32), r.uniform(-0.2, 0.2, K).astype(np.float32)
    z_ref = oc.conv(cpu, x2, w2, b2, (0, 0), (st, st), 1, _abi.ACT_IDENTITY)
    ref = oc.conv(cpu, x, w, b, (0, 0), (1, 1), 1, _abi.ACT_RELU, z=z_ref)
    lay = (lambda t: np.ascontiguousarray(t.transpose(1, 2, 3, 0))) if crsk else (lambda t: t)
    X, Wt, B, X2, Wt2, B2 = gpu.put(x), gpu.put(lay(w)), gpu.put(b), gpu.put(x2), gpu.put(lay(w2)), gpu.put(b2)
    Y = gpu.empty(ref.shape, np.float32)
    gpu.ops.set_filter_layout(_abi.FILTER_CRSK if crsk else _abi.FILTER_KCRS)
    try:
        for _ in range(2):  # twice: the split reduction's counters must be back at zero
            gpu.ops.conv_bias_add_conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (0, 0), (1, 1), gpu.ptr(X2), x2.shape,
                                                  gpu.ptr(Wt2), w2.shape, gpu.ptr(B2), (0, 0), (st, st), _abi.ACT_RELU, gpu.ptr(Y), dtype=_abi.F32)
            gpu.sync()
            np.testing.assert_allclose(gpu.get(Y), ref, rtol=1e-4, atol=1e-5)
    finally:
        gpu.ops.set_filter_layout(_abi.FILTER_KCRS)


def test_last_convolution_and_projection_shortcut_with_other_convolutions(gpu, cpu):
    """Shapes the one-kernel forms do not take run as the two convolutions through Y and give the chain's bits: a 3x3
    closing convolution in fp16 channels-last."""
    r = rng(11)
    x = r.standard_normal((2, 64, 9, 9)).astype(np.float16)
    x2 = r.standard_normal((2, 128, 9, 9)).astype(np.float16)
    w = (r.standard_normal((72, 64, 3, 3)) * 0.06).astype(np.float16)
    w2 = (r.standard_normal((72, 128, 1, 1)) * 0.1).astype(np.float16)
    b, b2 = r.uniform(-0.2, 0.2, 72).astype(np.float16), r.uniform(-0.2, 0.2, 72).astype(np.float16)
    nhwc = lambda t: np.ascontiguousarray(t.transpose(0, 2, 3, 1))  # noqa: E731
    X, Wt, B, X2, Wt2, B2 = gpu.put(nhwc(x)), gpu.put(nhwc(w)), gpu.put(b), gpu.put(nhwc(x2)), gpu.put(nhwc(w2)), gpu.put(b2)
    Y = gpu.empty((2 * 72 * 9 * 9,), np.float16)
    gpu.ops.set_format(_abi.NHWC)
    try:
        gpu.ops.conv_bias_add_conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (1, 1), (1, 1), gpu.ptr(X2), x2.shape,
                                              gpu.ptr(Wt2), w2.shape, gpu.ptr(B2), (0, 0), (1, 1), _abi.ACT_RELU, gpu.ptr(Y))
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    got = gpu.get(Y).reshape(2, 9, 9, 72).transpose(0, 3, 1, 2)
    z_gpu = conv_f16(gpu, x2, w2, b2, (0, 0), (1, 1), 1, _abi.ACT_IDENTITY, _abi.NHWC)
    two = conv_f16(gpu, x, w, b, (1, 1), (1, 1), 1, _abi.ACT_RELU, _abi.NHWC, z=z_gpu)
    np.testing.assert_array_equal(got, two)
    z_ref = oc.conv(cpu, x2, w2, b2, (0, 0), (1, 1), 1, _abi.ACT_IDENTITY)
    ref = oc.conv(cpu, x, w, b, (1, 1), (1, 1), 1, _abi.ACT_RELU, z=z_ref)
    np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=4e-3, atol=4e-3)


def test_last_convolution_and_projection_shortcut_refuses_other_shapes(gpu):
    r = rng(4)
    x = r.standard_normal((1, 64, 8, 8)).astype(np.float16)
    w = r.standard_normal((64, 64, 1, 1)).astype(np.float16)
    b = np.zeros(64, np.float16)
    X, Wt, B = gpu.put(x), gpu.put(w), gpu.put(b)
    Y = gpu.empty((64 * 64,), np.float16)
    gpu.ops.set_format(_abi.NHWC)
    try:
        with pytest.raises(RuntimeError, match="give"):  # the two convolutions must land on the same tensor
            gpu.ops.conv_bias_add_conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (0, 0), (1, 1), gpu.ptr(X), (1, 64, 4, 16),
                                                  gpu.ptr(Wt), w.shape, gpu.ptr(B), (0, 0), (1, 1), _abi.ACT_RELU, gpu.ptr(Y))
        with pytest.raises(RuntimeError, match="dtype"):
            gpu.ops.conv_bias_add_conv_bias_activ(gpu.ptr(X), x.shape, gpu.ptr(Wt), w.shape, gpu.ptr(B), (0, 0), (1, 1), gpu.ptr(X), x.shape,
                                                  gpu.ptr(Wt), w.shape, gpu.ptr(B), (0, 0), (1, 1), _abi.ACT_RELU, gpu.ptr(Y), dtype=_abi.I64)
    finally:
        gpu.ops.set_format(_abi.NCHW)


# Problems of the size ResNet-50 has at batch 64: the dispatcher picks its large tiles (128 x 128 and up,
# four or eight wavefronts) only when a launch has hundreds of tiles, so these are the only cases that reach
# them.  N, C, H, W, K, R, stride, pad
F16_BATCH64_CASES = [
    (64, 128, 28, 28, 128, 3, 1, 1),   # 392 tiles of 128 x 128, padded taps
    (32, 128, 28, 28, 128, 3, 1, 1),   # 196 tiles: about one per CU
    (64, 512, 28, 28, 128, 1, 1, 0),   # 1x1, no taps to mask, eight steps
    (64, 256, 14, 14, 256, 3, 1, 1),   # 14 x 14: 196 tiles
    (64, 128, 56, 56, 128, 3, 2, 1),   # strided 3x3
    (64, 256, 56, 56, 512, 1, 2, 0),   # strided 1x1 (downsample branch)
    (64, 64, 56, 56, 64, 3, 1, 1),     # K_out = 64: 64-filter tiles
    (61, 128, 28, 28, 136, 3, 1, 1),   # ragged in pixels (47824 = 373.6 x 128) and in filters
    (64, 512, 7, 7, 512, 3, 1, 1),     # 7 x 7: few, deep tiles
    (64, 1024, 14, 14, 256, 1, 1, 0),  # sixteen steps
    (64, 2048, 7, 7, 512, 1, 1, 0),    # 7 x 7, 1x1: 64-row tiles on eight wavefronts
    (64, 512, 14, 14, 512, 3, 2, 1),   # the same, strided 3x3
]


def f16_problem(case, seed):
    N, C, H, W, K, R, st, pd = case
    r = rng(seed)
    x = r.standard_normal((N, C, H, W), dtype=np.float32).astype(np.float16)
    w = (r.standard_normal((K, C, R, R), dtype=np.float32) * np.sqrt(2.0 / (C * R * R))).astype(np.float16)
    b = r.uniform(-0.1, 0.1, K).astype(np.float16)
    return x, w, b, (pd, pd), (st, st)


@pytest.mark.parametrize("case", F16_BATCH64_CASES, ids=lambda c: "x".join(map(str, c)))
def test_conv_f16_at_batch_64_sizes(gpu, cpu, case):
    x, w, b, pads, strides = f16_problem(case, sum(case))
    ref = oc.conv(cpu, x, w, b, pads, strides, 1, _abi.ACT_RELU)
    got = conv_f16(gpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, _abi.NHWC)
    np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3)
    z = rng(1 + sum(case)).standard_normal(ref.shape, dtype=np.float32).astype(np.float16)
    refz = oc.conv(cpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, z=z)
    gotz = conv_f16(gpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, _abi.NHWC, z=z)
    np.testing.assert_allclose(gotz.astype(np.float32), refz.astype(np.float32), rtol=4e-3, atol=4e-3)
    np.testing.assert_array_equal(conv_f16(gpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, _abi.NHWC, z=z, inplace=True), gotz)


def test_every_compiled_f16_conv_variant(gpu, cpu):
    """Each variant dnnrtListConvTiles names, forced with dnnrtSetConvTile, on a padded 3x3 problem, a 1x1
    problem over 128 channels and one over 512, and two 3x3 problems on small images whose runs of pixels cross
    image boundaries (one to three per tile), all ragged in both directions: it either matches the
    oracle or refuses the problem loudly (the single-stage variants take reductions of up to four steps)."""
    tiles = gpu.ops.conv_tiles()
    assert tiles and 0 not in tiles
    cases = [(3, 128, 19, 23, 200, 3, 1, 1), (5, 128, 19, 23, 200, 1, 1, 0), (5, 512, 9, 13, 136, 1, 2, 0),
             (11, 192, 14, 14, 136, 3, 1, 1), (23, 128, 7, 7, 72, 3, 1, 1), (5, 64, 13, 20, 72, 3, 1, 1), (2, 64, 56, 56, 64, 3, 1, 1)]
    ran = {t: 0 for t in tiles}
    for case in cases:
        x, w, b, pads, strides = f16_problem(case, 5 + sum(case))
        z = rng(6).standard_normal((case[0], case[4]) + oc.conv_out_hw(case[2], case[3], case[5], case[5], pads, strides),
                                   dtype=np.float32).astype(np.float16)
        ref = oc.conv(cpu, x, w, b, pads, strides, 1, _abi.ACT_RELU)
        refz = oc.conv(cpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, z=z)
        for t in tiles:
            gpu.ops.set_conv_tile(t)
            try:
                got = conv_f16(gpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, _abi.NHWC)
                try:
                    gotz = conv_f16(gpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, _abi.NHWC, z=z)
                    np.testing.assert_array_equal(conv_f16(gpu, x, w, b, pads, strides, 1, _abi.ACT_RELU, _abi.NHWC, z=z, inplace=True), gotz,
                                                  err_msg=f"variant {t} on {case} written over its residual operand")
                except RuntimeError as e:  # a variant without the residual operand says so
                    assert "residual" in str(e), str(e)
                    gotz = None
            except RuntimeError as e:
                assert "tile" in str(e) or "variant" in str(e), str(e)
                continue
            finally:
                gpu.ops.set_conv_tile(0)
            ran[t] += 1
            np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=2e-3,
                                       err_msg=f"variant {t} on {case}")
            if gotz is not None:
                np.testing.assert_allclose(gotz.astype(np.float32), refz.astype(np.float32), rtol=4e-3, atol=4e-3,
                                           err_msg=f"variant {t} on {case} with a residual")
    assert all(ran.values()), f"variants that ran no case: {[t for t, n in ran.items() if not n]}"
    with pytest.raises(RuntimeError):
        gpu.ops.set_conv_tile(9999)


def test_f16_channels_last_ops(gpu, cpu):
    r = rng(77)
    x = r.standard_normal((2, 64, 28, 28)).astype(np.float16)
    xl = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    gpu.ops.set_format(_abi.NHWC)
    try:
        X = gpu.put(xl)
        Y = gpu.empty((2 * 64 * 14 * 14,), np.float16)
        gpu.ops.maxpool(gpu.ptr(X), x.shape, gpu.ptr(Y), (2, 64, 14, 14), (3, 3), (1, 1, 1, 1), (2, 2), _abi.F16)
        G = gpu.empty((2 * 64,), np.float16)
        gpu.ops.reduce_mean(gpu.ptr(X), x.shape, gpu.ptr(G), (2, 64, 1, 1), _abi.F16)
        bias = r.standard_normal((1, 64, 1, 1)).astype(np.float16)
        Bv = gpu.put(bias.reshape(64))
        O = gpu.empty(xl.shape, np.float16)
        gpu.ops.tensor_op(_abi.OP_ADD, gpu.ptr(X), x.shape, gpu.ptr(Bv), (1, 64, 1, 1), gpu.ptr(O), 1.0, _abi.F16)
        gpu.sync()
    finally:
        gpu.ops.set_format(_abi.NCHW)
    np.testing.assert_array_equal(gpu.get(Y).reshape(2, 14, 14, 64).transpose(0, 3, 1, 2),
                                  oc.pool(cpu, "max", x, (3, 3), (1, 1), (2, 2)))
    np.testing.assert_allclose(gpu.get(G).reshape(2, 64, 1, 1).astype(np.float32),
                               oc.reduce_mean(cpu, x, (2, 64, 1, 1)).astype(np.float32), rtol=2e-3, atol=1e-3)
    np.testing.assert_array_equal(gpu.get(O).transpose(0, 3, 1, 2), oc.tensor_op(cpu, _abi.OP_ADD, x, bias))


@pytest.mark.parametrize("C", [64, 12])          # 16-byte vector kernel / scalar kernel
@pytest.mark.parametrize("kind", ["max", "avg"])
def test_pooling_f16_channels_last(gpu, cpu, C, kind):
    r = rng(79 + C)
    x = r.standard_normal((3, C, 15, 13)).astype(np.float16)
    x[1, 3, 4, 5] = np.nan                        # NaN must reach every window that sees it
    for kernel, pads, strides in [((3, 3), (1, 1), (2, 2)), ((2, 2), (0, 0), (2, 2)), ((3, 2), (1, 0), (1, 2))]:
        P, Q = oc.conv_out_hw(15, 13, kernel[0], kernel[1], pads, strides)
        gpu.ops.set_format(_abi.NHWC)
        try:
            X = gpu.put(np.ascontiguousarray(x.transpose(0, 2, 3, 1)))
            Y = gpu.empty((3 * C * P * Q,), np.float16)
            fn = gpu.ops.maxpool if kind == "max" else gpu.ops.avgpool
            fn(gpu.ptr(X), x.shape, gpu.ptr(Y), (3, C, P, Q), kernel, [pads[0], pads[1], pads[0], pads[1]], strides, _abi.F16)
            gpu.sync()
        finally:
            gpu.ops.set_format(_abi.NCHW)
        got = gpu.get(Y).reshape(3, P, Q, C).transpose(0, 3, 1, 2)
        ref = oc.pool(cpu, kind, x, kernel, pads, strides)
        if kind == "max":
            np.testing.assert_array_equal(got, ref)
        else:
            np.testing.assert_allclose(got.astype(np.float32), ref.astype(np.float32), rtol=2e-3, atol=1e-3)


def test_matmul2d_f16(gpu, cpu):
    r = rng(78)
    for M, K, N in [(64, 2048, 1000), (2, 64, 8), (130, 96, 72)]:
        a = r.standard_normal((M, K)).astype(np.float16)
        b = (r.standard_normal((N, K)) / np.sqrt(K)).astype(np.float16)
        np.testing.assert_allclose(oc.matmul2d(gpu, a, b, transB=1).astype(np.float32),
                                   oc.matmul2d(cpu, a, b, transB=1).astype(np.float32), rtol=2e-3, atol=2e-3)
        # C as one row with beta 1 (a Gemm's bias): the convolution kernel's bias; the oracle runs product, then add
        row = r.standard_normal(N).astype(np.float16)
        np.testing.assert_allclose(oc.matmul2d_row(gpu, a, b, row, transB=1).astype(np.float32),
                                   oc.matmul2d_row(cpu, a, b, row, transB=1).astype(np.float32), rtol=2e-3, atol=4e-3)
    # every other form on the generic fp16 kernel: the four operand layouts, alpha and beta with a row or a matrix C
    # (the matrix updated in place), ragged tiles
    for M, K, N in [(130, 96, 72), (5, 7, 3), (64, 200, 65)]:
        for tA in (0, 1):
            for tB in (0, 1):
                a = r.standard_normal((K, M) if tA else (M, K)).astype(np.float16)
                b = (r.standard_normal((N, K) if tB else (K, N)) / np.sqrt(K)).astype(np.float16)
                c = r.standard_normal((M, N)).astype(np.float16)
                row = r.standard_normal(N).astype(np.float16)
                for kw in (dict(), dict(alpha=0.5), dict(c=c, alpha=1.5, beta=0.5), dict(c=c, beta=1.0)):
                    np.testing.assert_allclose(oc.matmul2d(gpu, a, b, transA=tA, transB=tB, **kw).astype(np.float32),
                                               oc.matmul2d(cpu, a, b, transA=tA, transB=tB, **kw).astype(np.float32), rtol=4e-3, atol=6e-3)
                if not tA:
                    np.testing.assert_allclose(oc.matmul2d_row(gpu, a, b, row, beta=0.5, transB=tB).astype(np.float32),
                                               oc.matmul2d_row(cpu, a, b, row, beta=0.5, transB=tB).astype(np.float32), rtol=4e-3, atol=6e-3)


class ExecBlock(C.Structure):
    _fields_ = ([(n, C.c_void_p) for n in ("x", "w1", "b1", "wd", "bd", "w3", "b3", "z", "y")] +
                [(n, C.c_int64) for n in ("n", "cin", "h", "w", "ch", "r", "s", "stride", "pad_h", "pad_w", "p", "q", "cout", "act1", "actd", "act")] +
                [(n, C.c_float) for n in ("coef1", "coefd", "coef")] + [(n, C.c_int32) for n in ("expand", "dtype", "format", "filter_layout")])


@pytest.mark.parametrize("n,cin,h,w,ch,cout,stride,expand,residual", [
    (1, 8, 5, 7, 48, 8, 1, True, False),       # less than one tile, channels short of every block
    (2, 16, 33, 17, 96, 24, 2, True, False),   # one step of input channels, stride 2, ragged tiles
    (1, 24, 28, 29, 144, 24, 1, True, True),   # half a step, half a group of channels, residual
    (3, 64, 14, 14, 384, 64, 1, True, True),
    (1, 96, 7, 9, 576, 160, 2, True, False),   # most steps, five blocks of output channels
    (2, 40, 11, 10, 200, 328, 1, True, False),  # output channels over two workgroups
    (1, 32, 30, 31, 32, 16, 1, False, False),  # no expansion
    (1, 24, 13, 12, 24, 24, 2, False, False),
])
def test_inverted_residual_block_fp16(n, cin, h, w, ch, cout, stride, expand, residual):
    """The block call of the executor against fp32 arithmetic on the same operands, rounded to fp16 where the three
    separate calls round."""
    import torch
    import torch.nn.functional as F
    g = torch.Generator().manual_seed(n * 1000 + cin)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x = rnd(n, cin, h, w).half()
    w1, b1 = (rnd(ch, cin) * (2 / cin) ** 0.5).half(), rnd(ch).half() * 0.5
    wd, bd = (rnd(ch, 1, 3, 3) * 0.4).half(), rnd(ch).half() * 0.5
    w3, b3 = (rnd(cout, ch) * (1 / ch) ** 0.5).half(), rnd(cout).half() * 0.5
    r16 = lambda t: t.half().float()  # noqa: E731
    t = x.float()
    if expand:
        t = r16(F.conv2d(t, w1.float()[:, :, None, None], b1.float()).clamp(0, 6))
    t = r16(F.conv2d(t, wd.float(), bd.float(), stride, 1, groups=ch).clamp(0, 6))
    want = F.conv2d(t, w3.float()[:, :, None, None], b3.float())
    p, q = want.shape[2:]
    z = rnd(n, cout, p, q).half() if residual else None
    want = r16(r16(want) + z.float()) if residual else r16(want)

    lib = C.CDLL(_abi.RUNTIME_PATH)
    handle = C.c_void_p()
    assert lib.dnnrtCreate(C.byref(handle)) == 0
    lib.dnnrtExecBlockFilter.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_int64]

    def blocked(m):
        out = torch.empty_like(m)
        lib.dnnrtExecBlockFilter(out.data_ptr(), m.contiguous().data_ptr(), m.shape[0], m.shape[1])
        return out.cuda()
    keep = dict(x=x.permute(0, 2, 3, 1).contiguous().cuda(), w1=blocked(w1) if expand else None, b1=b1.cuda() if expand else None,
                wd=wd.cuda(), bd=bd.cuda(), w3=blocked(w3), b3=b3.cuda(), z=None if z is None else z.permute(0, 2, 3, 1).contiguous().cuda(),
                y=torch.full((n, p, q, cout), float("nan"), dtype=torch.half, device="cuda"))
    k = ExecBlock(n=n, cin=cin, h=h, w=w, ch=ch, r=3, s=3, stride=stride, pad_h=1, pad_w=1, p=p, q=q, cout=cout, act1=3, actd=3, act=5,
                  coef1=6.0, coefd=6.0, expand=int(expand), dtype=_abi.F16, format=1, **{m: v.data_ptr() for m, v in keep.items() if v is not None})
    torch.cuda.synchronize()
    lib.dnnrtLastError.restype = C.c_char_p
    assert lib.dnnrtExecRunBlock(handle, C.byref(k)) == 0, lib.dnnrtLastError()
    torch.cuda.synchronize()
    got = keep["y"].permute(0, 3, 1, 2).float().cpu()
    lib.dnnrtDestroy(handle)
    np.testing.assert_allclose(got.numpy(), want.numpy(), rtol=4e-3, atol=8e-3)


@pytest.mark.parametrize("n,cin,h,w,ch,cout,stride,expand,residual", [
    (1, 160, 7, 7, 960, 160, 1, True, True),     # ten steps of input channels, parts of the hidden ones
    (40, 136, 7, 6, 840, 160, 1, True, False),   # a last step and a last group that are not full
    (2, 160, 7, 7, 960, 320, 1, True, False),    # output channels over two workgroups, each with parts
    (1, 96, 14, 13, 576, 96, 1, True, True),
    (1, 32, 9, 11, 200, 24, 2, True, False),     # seven groups in parts of unequal size
    (3, 192, 8, 8, 192, 16, 1, False, False),    # parts without an expansion
])
def test_inverted_residual_block_fp16_in_parts(n, cin, h, w, ch, cout, stride, expand, residual):
    """The hidden channels cut over workgroups."""
    test_inverted_residual_block_fp16(n, cin, h, w, ch, cout, stride, expand, residual)


@pytest.mark.parametrize("n,cin,h,w,ch,cout,stride,expand,residual", [
    (64, 24, 20, 21, 144, 24, 1, True, True),    # whole channels: every number of steps of input channels, both strides
    (64, 24, 30, 31, 144, 24, 2, True, False),
    (1, 40, 7, 7, 240, 72, 2, True, False),
    (48, 88, 14, 13, 528, 96, 1, True, False),
    (24, 88, 30, 31, 528, 96, 2, True, False),
    (2, 120, 7, 6, 240, 328, 1, True, False),
    (2, 120, 7, 6, 240, 328, 2, True, False),
    (1, 16, 7, 9, 960, 24, 1, True, False),      # ... and in parts
    (1, 16, 7, 9, 960, 24, 2, True, False),
    (1, 64, 7, 7, 384, 64, 2, True, False),
    (1, 136, 7, 7, 272, 104, 2, True, False),
    (2, 192, 7, 7, 192, 16, 2, False, False),
])
def test_inverted_residual_block_fp16_kernels(n, cin, h, w, ch, cout, stride, expand, residual):
    """With the cases of the two tests above, each of the kernels."""
    test_inverted_residual_block_fp16(n, cin, h, w, ch, cout, stride, expand, residual)


@pytest.mark.parametrize("n,cin,h,w,ch,cout,stride,pads,expand,residual,acts", [
    (1, 8, 5, 7, 16, 8, 1, (1, 1), True, False, (3, 3, 5)),      # less than a tile, one group of hidden channels
    (1, 16, 33, 17, 96, 24, 2, (1, 1), True, False, (3, 3, 5)),  # ragged tiles, half a block of output channels
    (1, 24, 28, 29, 144, 24, 1, (1, 1), True, True, (3, 3, 3)),  # the hidden channels over workgroups, residual
    (16, 32, 30, 31, 192, 32, 1, (2, 0), True, True, (1, 3, 1)),  # many tiles
    (1, 64, 14, 14, 384, 64, 1, (1, 1), True, True, (3, 3, 5)),
    (3, 40, 11, 10, 208, 72, 2, (0, 2), True, False, (5, 1, 5)),  # a last chunk of one step in four
    (24, 96, 13, 14, 288, 96, 1, (1, 1), True, False, (3, 3, 5)),
    (1, 96, 7, 9, 576, 160, 2, (1, 1), True, False, (3, 3, 5)),
    (1, 160, 7, 7, 960, 328, 1, (1, 1), True, False, (3, 3, 5)),  # output channels over three workgroups, the last with one block
    (40, 160, 7, 6, 480, 160, 1, (1, 1), True, True, (3, 3, 5)),
    (2, 120, 9, 2, 112, 16, 1, (1, 2), True, False, (3, 3, 5)),  # an image narrower than a square's window
    (1, 32, 30, 31, 32, 16, 1, (1, 1), False, False, (0, 3, 5)),  # no expansion
    (5, 48, 13, 12, 48, 24, 2, (1, 1), False, False, (0, 1, 5)),
])
def test_inverted_residual_block_fp32(n, cin, h, w, ch, cout, stride, pads, expand, residual, acts):
    """The fp32 block call against 64 bits: every result within the bound that its three sums' lengths and magnitudes give, and
    the same bits in a second call (the parts' counters are back at zero)."""
    import torch
    import torch.nn.functional as F
    g = torch.Generator().manual_seed(n * 1000 + cin + h)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, w1, b1 = rnd(n, cin, h, w), rnd(ch, cin) * (2 / cin) ** 0.5, rnd(ch) * 0.5
    wd, bd, w3, b3 = rnd(ch, 1, 3, 3) * 0.4, rnd(ch) * 0.5, rnd(cout, ch) * (1 / ch) ** 0.5, rnd(cout) * 0.5
    act = lambda t, mode: t if mode == 5 else t.clamp(0, 6) if mode == 3 else t.clamp(min=0)  # noqa: E731
    u, d = 2.0 ** -24, lambda t: t.double()  # noqa: E731
    t, err = d(x), torch.zeros_like(d(x))
    if expand:
        k = d(w1)[:, :, None, None]
        err = (cin + 2) * u * (F.conv2d(t.abs(), k.abs()) + d(b1).abs()[:, None, None])
        t = act(F.conv2d(t, k, d(b1)), acts[0])
    k, mag = d(wd), t.abs()
    err = F.conv2d(err, k.abs(), None, stride, pads, groups=ch) + 11 * u * (F.conv2d(mag, k.abs(), None, stride, pads, groups=ch) + d(bd).abs()[:, None, None])
    t = act(F.conv2d(t, k, d(bd), stride, pads, groups=ch), acts[1])
    k, mag = d(w3)[:, :, None, None], t.abs()
    err = F.conv2d(err, k.abs()) + (ch + 4) * u * (F.conv2d(mag, k.abs()) + d(b3).abs()[:, None, None])
    want = F.conv2d(t, k, d(b3))
    p, q = want.shape[2:]
    z = rnd(n, cout, p, q) if residual else None
    if residual:
        want, err = want + d(z), err + 2 * u * (want.abs() + d(z).abs())
    want = act(want, acts[2])

    lib = C.CDLL(_abi.RUNTIME_PATH)
    handle = C.c_void_p()
    assert lib.dnnrtCreate(C.byref(handle)) == 0
    lib.dnnrtExecBlockFilterF32.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_int64]

    def blocked(m):
        out, crsk = torch.empty_like(m), m.t().contiguous()
        lib.dnnrtExecBlockFilterF32(out.data_ptr(), crsk.data_ptr(), m.shape[0], m.shape[1])
        return out.cuda()
    keep = dict(x=x.cuda(), w1=blocked(w1) if expand else None, b1=b1.cuda() if expand else None, wd=wd.reshape(ch, 9).t().contiguous().cuda(), bd=bd.cuda(),
                w3=blocked(w3), b3=b3.cuda(), z=None if z is None else z.cuda(), y=torch.full((n, cout, p, q), float("nan"), device="cuda"))
    k = ExecBlock(n=n, cin=cin, h=h, w=w, ch=ch, r=3, s=3, stride=stride, pad_h=pads[0], pad_w=pads[1], p=p, q=q, cout=cout, act1=acts[0], actd=acts[1],
                  act=acts[2], coef1=6.0, coefd=6.0, coef=6.0, expand=int(expand), dtype=_abi.F32, format=_abi.NCHW, **{m: v.data_ptr() for m, v in keep.items() if v is not None})
    torch.cuda.synchronize()
    lib.dnnrtLastError.restype = C.c_char_p
    got = []
    for _ in range(2):
        assert lib.dnnrtExecRunBlock(handle, C.byref(k)) == 0, lib.dnnrtLastError()
        torch.cuda.synchronize()
        got.append(keep["y"].cpu())
        keep["y"].fill_(float("nan"))
        torch.cuda.synchronize()
    assert torch.equal(*got)
    worst = ((got[0].double() - want).abs() / err).max()
    assert worst <= 1, worst
    for bad in (dict(cin=cin + 4), dict(ch=ch + 8), dict(cout=cout + 4), dict(format=_abi.NHWC), dict(q=q + 1), dict(pad_h=3), dict(actd=6)):  # not run: refused
        other = ExecBlock.from_buffer_copy(k)
        for name, value in bad.items():
            setattr(other, name, value)
        assert not lib.dnnrtExecBlockApplies(handle, C.byref(other)) and lib.dnnrtExecRunBlock(handle, C.byref(other)) != 0, bad
    lib.dnnrtDestroy(handle)


@pytest.mark.parametrize("n,cin,h,w,ch,cout,stride,pads,expand,residual,acts", [
    # tiles of 32 pixels with 40 to 160 input channels: four and eight wavefronts, whole channels and parts
    (48, 40, 14, 13, 240, 72, 1, (1, 1), True, False, (3, 3, 5)),
    (8, 64, 14, 13, 384, 64, 1, (1, 1), True, True, (3, 3, 5)),
    (12, 40, 20, 21, 240, 72, 1, (1, 1), True, False, (3, 3, 1)),
    (12, 64, 14, 13, 384, 96, 1, (1, 1), True, False, (3, 3, 5)),
    (48, 96, 20, 21, 576, 96, 2, (1, 1), True, False, (3, 3, 5)),
    (24, 96, 14, 13, 576, 96, 2, (1, 1), True, False, (3, 3, 5)),
    (6, 40, 56, 57, 240, 72, 2, (1, 1), True, False, (3, 3, 5)),
    (16, 64, 20, 21, 384, 64, 2, (1, 1), True, True, (3, 3, 5)),
    (48, 8, 14, 13, 48, 160, 1, (1, 1), True, False, (3, 3, 5)),  # two steps of 40: the others are read and not used
    (6, 96, 14, 13, 576, 160, 1, (1, 1), True, False, (3, 3, 5)),
    (12, 120, 14, 13, 240, 328, 1, (1, 1), True, False, (3, 3, 5)),
    (16, 160, 7, 7, 960, 160, 1, (1, 1), True, True, (3, 3, 5)),
    (32, 8, 20, 21, 48, 160, 2, (1, 1), True, False, (3, 3, 5)),
    (24, 96, 14, 13, 576, 160, 2, (1, 1), True, False, (3, 3, 5)),
    # tiles of 16 pixels, eight wavefronts
    (12, 40, 14, 13, 240, 72, 1, (1, 1), True, False, (3, 3, 5)),
    (6, 64, 14, 13, 384, 64, 1, (1, 1), True, True, (3, 3, 5)),
    (12, 40, 28, 28, 240, 72, 2, (1, 1), True, False, (3, 3, 5)),
    (8, 96, 14, 13, 576, 96, 2, (1, 1), True, False, (3, 3, 5)),
    (6, 120, 14, 13, 240, 328, 1, (1, 1), True, False, (3, 3, 5)),
    (8, 160, 7, 7, 960, 160, 1, (1, 1), True, False, (3, 3, 5)),
    (12, 120, 14, 13, 240, 328, 2, (1, 1), True, False, (3, 3, 5)),
    (6, 120, 14, 13, 240, 328, 2, (1, 1), True, False, (3, 3, 5)),
    # four, whole channels
    (6, 40, 28, 28, 240, 72, 1, (1, 1), True, False, (3, 3, 5)),
    (24, 40, 28, 28, 240, 72, 2, (1, 1), True, False, (3, 3, 5)),
    (2, 8, 7, 7, 48, 160, 1, (1, 1), True, False, (3, 3, 5)),
    (2, 8, 7, 7, 48, 160, 2, (1, 1), True, False, (3, 3, 5)),
    (1, 24, 7, 7, 144, 24, 2, (1, 1), True, False, (3, 3, 5)),
    (3, 32, 9, 8, 32, 16, 2, (1, 1), False, False, (0, 3, 5)),
])
def test_inverted_residual_block_fp32_kernels(n, cin, h, w, ch, cout, stride, pads, expand, residual, acts):
    """With the cases above, each of the kernels in each of the ways that the planner launches it."""
    test_inverted_residual_block_fp32(n, cin, h, w, ch, cout, stride, pads, expand, residual, acts)


@pytest.mark.parametrize("case", [
    # N, C, H, W, K, pad, residual, activation: sizes at which the launcher picks the tiles of conv_f32_winograd.hip
    (22, 64, 56, 56, 64, 1, False, _abi.ACT_RELU),          # 539 tiles: 27 left over, in parts of four stages of four channels
    (6, 48, 75, 77, 100, 1, True, _abi.ACT_LEAKY_RELU),     # odd image, filters off the 64 grid
    (3, 512, 19, 19, 486, 1, False, _abi.ACT_IDENTITY),     # filter rows off the 16-byte grid
    (4, 128, 64, 63, 128, 0, True, _abi.ACT_RELU),          # no padding
    (1, 256, 50, 51, 256, 2, False, _abi.ACT_CLIPPED_RELU),
    (2, 512, 28, 28, 256, 1, True, _abi.ACT_RELU),
])
def test_conv_3x3_by_minimal_filtering(gpu, case):
    """Against 64-bit sums: no further from them than a chain of 9 C fp32 additions, whose relative error in the 2-norm is about
    2^-25 sqrt(9 C) / 2.4 for independent products, and the transforms' few roundings beside it."""
    import torch
    N, Cc, H, W, K, pad, residual, activ = case
    r = rng(N * 100 + Cc)
    x = np.maximum(r.standard_normal((N, Cc, H, W)), 0).astype(np.float32)
    w = (r.standard_normal((K, Cc, 3, 3)) * np.sqrt(2.0 / (9 * Cc))).astype(np.float32)
    b = r.uniform(-0.5, 0.5, K).astype(np.float32)
    ref = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), torch.from_numpy(b).double(), padding=pad).numpy()
    z = r.standard_normal(ref.shape).astype(np.float32) if residual else None
    if residual:
        ref = ref + z
    coef = {_abi.ACT_LEAKY_RELU: 0.1, _abi.ACT_CLIPPED_RELU: 1.5}.get(activ)
    if activ == _abi.ACT_LEAKY_RELU:
        ref = np.where(ref < 0, 0.1 * ref, ref)
    elif activ != _abi.ACT_IDENTITY:
        ref = np.clip(ref, 0, 1.5 if activ == _abi.ACT_CLIPPED_RELU else None)
    bound = 2.0 ** -25 * (np.sqrt(9 * Cc) / 2.4 + 4)
    for _ in range(2):  # twice: the split reduction's counters must be back at zero
        got = oc.conv(gpu, x, w, b, (pad, pad), (1, 1), 1, activ, crsk=True, z=z, coef=coef, inplace=residual)
        assert np.linalg.norm(got - ref) <= bound * np.linalg.norm(ref)
        np.testing.assert_allclose(got, ref, rtol=RTOL, atol=ATOL)
    direct = oc.conv(gpu, x, w, b, (pad, pad), (1, 1), 1, activ, crsk=True, z=z, coef=coef, inplace=residual, algo=_abi.CONV_ALGO_DIRECT)
    assert (got != direct).any()  # the kernel under test is the one that ran
    np.testing.assert_allclose(direct, ref, rtol=RTOL, atol=ATOL)


def _minimal_filtering_magnitudes(x, w, pad):
    """F(2x2, 3x3) with every value and every coefficient replaced by its magnitude, in 64 bits."""
    import torch
    G = torch.tensor([[1, 0, 0], [.5, .5, .5], [.5, .5, .5], [0, 0, 1]], dtype=torch.float64)
    B = torch.tensor([[1, 0, 1, 0], [0, 1, 1, 0], [0, 1, 1, 0], [0, 1, 0, 1]], dtype=torch.float64)
    A = torch.tensor([[1, 1, 1, 0], [0, 1, 1, 1]], dtype=torch.float64)
    N, Cc, H, W = x.shape
    K, P, Q = w.shape[0], H + 2 * pad - 2, W + 2 * pad - 2
    th, tw = (P + 1) // 2, (Q + 1) // 2
    d = torch.zeros((N, Cc, 2 * th + 2, 2 * tw + 2), dtype=torch.float64)
    d[:, :, pad:pad + H, pad:pad + W] = torch.from_numpy(np.abs(x)).double()[:, :, :2 * th + 2 - pad, :2 * tw + 2 - pad]
    V = torch.matmul(torch.matmul(B, d.unfold(2, 4, 2).unfold(3, 4, 2)), B.T).permute(4, 5, 1, 0, 2, 3).reshape(4, 4, Cc, -1)
    U = torch.matmul(torch.matmul(G, torch.from_numpy(np.abs(w)).double()), G.T)
    M = torch.stack([torch.stack([U[:, :, i, j] @ V[i, j] for j in range(4)], -1) for i in range(4)], -2)  # [K][tiles][4][4]
    Y = torch.matmul(torch.matmul(A, M), A.T).reshape(K, N, th, tw, 2, 2).permute(1, 0, 2, 4, 3, 5).reshape(N, K, 2 * th, 2 * tw)
    return Y[:, :, :P, :Q].numpy()


@pytest.mark.parametrize("values", ["dense", "sparse", "pruned", "both", "uneven"])
@pytest.mark.parametrize("case", [(3, 512, 19, 19, 486, 1), (2, 256, 56, 55, 256, 1), (4, 128, 64, 63, 128, 0)], ids=["512", "256", "128"])
def test_conv_3x3_of_sparse_and_uneven_values(gpu, case, values):
    """What the two ways of a 3x3 convolution promise for any values.  Direct sums: each of the 9 C + 1 additions rounds by at
    most 2^-24 of the sum of magnitudes.  Minimal filtering: a patch value has passed two roundings and a filter value
    four when they are multiplied, C products are added, four more additions and up to sixteen parts lead back, and one
    adds the bias: C + 27 roundings of the magnitudes' own minimal filtering, which know the patch and not the window.  With
    values that differ by orders of magnitude within a patch the first bound does not hold for the second way."""
    import torch
    N, Cc, H, W, K, pad = case
    r = rng(Cc)
    x = np.maximum(r.standard_normal((N, Cc, H, W)), 0)
    w = r.standard_normal((K, Cc, 3, 3)) * np.sqrt(2.0 / (9 * Cc))
    b = r.uniform(-0.01, 0.01, K).astype(np.float32)
    if values in ("sparse", "both"):
        x = np.abs(r.standard_normal(x.shape)) * (r.random(x.shape) < 0.05)
    if values in ("pruned", "both"):
        w *= r.random(w.shape) < 0.1
    if values == "uneven":  # the centre tap alone, pixels over eight decades
        x = np.abs(r.standard_normal(x.shape)) * 10.0 ** r.uniform(-4, 4, (N, 1, H, W))
        w *= np.pad(np.ones((1, 1)), 1)
    x, w = x.astype(np.float32), w.astype(np.float32)
    conv64 = lambda t, f, v: torch.nn.functional.conv2d(*(torch.from_numpy(u).double() for u in (t, f, v)), padding=pad).numpy()  # noqa: E731
    ref, magnitude = conv64(x, w, b), conv64(np.abs(x), np.abs(w), np.abs(b))
    default, direct = (oc.conv(gpu, x, w, b, (pad, pad), (1, 1), 1, _abi.ACT_IDENTITY, crsk=True, algo=a) for a in (1, _abi.CONV_ALGO_DIRECT))
    assert (np.abs(direct - ref) <= (9 * Cc + 1) * 2.0 ** -24 * magnitude).all()
    bound = (Cc + 27) * 2.0 ** -24 * (_minimal_filtering_magnitudes(x, w, pad) + np.abs(b)[:, None, None])
    assert (np.abs(default - ref) <= bound).all()
    assert (default != direct).any()
    if values == "uneven":
        assert (np.abs(default - ref) > (9 * Cc + 1) * 2.0 ** -24 * magnitude).any()
    error = [np.linalg.norm(v - ref) for v in (default, direct)]
    # measured: dense 0.7 to 0.8, sparse 1.1 to 1.3, pruned 1.4 to 1.6, both 2.1 to 2.4, uneven 1.3 to 1.5
    assert error[0] <= {"dense": 1.0, "sparse": 1.6, "pruned": 2.0, "both": 3.0, "uneven": 2.0}[values] * error[1]


@pytest.mark.parametrize("crsk", [False, True])
@pytest.mark.parametrize("geometry", [(2, 62, 64, 128, 1), (1, 14, 13, 40, 2)], ids=["many-tiles", "split"])
@pytest.mark.parametrize("Cc", [1, 2, 3, 5, 6, 9, 17, 24, 33, 41, 48, 57, 64, 131])
def test_conv_3x3_small_for_every_length_of_a_wavefronts_slice(gpu, geometry, Cc, crsk):
    """One to eight and more iterations of two channels a wavefront, the last with one channel or two, wavefronts without any:
    every ending of the 3x3 small kernel's ring of loads.  Bound: each of the 9 C + 1 additions rounds by at most 2^-24
    of the sum of magnitudes."""
    import torch
    N, H, W, K, st = geometry
    r = rng(Cc)
    x = r.standard_normal((N, Cc, H, W)).astype(np.float32)
    w = (r.standard_normal((K, Cc, 3, 3)) * np.sqrt(2.0 / (9 * Cc))).astype(np.float32)
    b = r.uniform(-0.5, 0.5, K).astype(np.float32)
    conv64 = lambda t, f, v: torch.nn.functional.conv2d(*(torch.from_numpy(u).double() for u in (t, f, v)), stride=st, padding=1).numpy()  # noqa: E731
    ref, magnitude = conv64(x, w, b), conv64(np.abs(x), np.abs(w), np.abs(b))
    for _ in range(2):  # twice: the split reduction's counters must be back at zero
        got = oc.conv(gpu, x, w, b, (1, 1), (st, st), 1, _abi.ACT_IDENTITY, crsk=crsk)
        assert (np.abs(got - ref) <= (9 * Cc + 1) * 2.0 ** -24 * magnitude).all()


# N, C, H, W, K, filter side, stride, pad, groups: on either side of the line between the kernels that know one image size, stride 1 and one
# group, and those that take any; one image and several, tiles that end within an image, slices that end the reduction early
@pytest.mark.parametrize("case", [(1, 40, 9, 13, 36, 1, 1, 0, 1), (3, 40, 9, 13, 36, 1, 1, 0, 1), (2, 72, 7, 5, 68, 1, 2, 0, 1), (2, 64, 6, 11, 48, 1, 1, 0, 2), (1, 256, 14, 14, 64, 1, 1, 0, 1),
                                  (1, 12, 9, 13, 36, 3, 1, 1, 1), (3, 12, 9, 13, 36, 3, 1, 1, 1), (2, 12, 9, 13, 36, 3, 1, 0, 1), (2, 12, 8, 13, 36, 3, 1, 2, 1),
                                  (1, 24, 9, 10, 40, 3, 2, 1, 1), (2, 16, 6, 11, 48, 3, 1, 1, 2), (1, 96, 14, 14, 64, 3, 1, 1, 1)], ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("crsk", [False, True])
def test_conv_f32_small_of_one_image_size_and_others(gpu, case, crsk):
    """Bound: each of the C R S + 2 additions rounds by at most 2^-24 of the sum of magnitudes."""
    import torch
    N, Cc, H, W, K, R, st, pad, g = case
    r = rng(sum(case))
    x = r.standard_normal((N, Cc, H, W)).astype(np.float32)
    w = (r.standard_normal((K, Cc // g, R, R)) * np.sqrt(2.0 / (R * R * Cc))).astype(np.float32)
    b = r.uniform(-0.5, 0.5, K).astype(np.float32)
    conv64 = lambda t, f, v: torch.nn.functional.conv2d(*(torch.from_numpy(u).double() for u in (t, f, v)), stride=st, padding=pad, groups=g).numpy()  # noqa: E731
    ref, magnitude = conv64(x, w, b), conv64(np.abs(x), np.abs(w), np.abs(b))
    z = r.standard_normal(ref.shape).astype(np.float32)
    for _ in range(2):  # twice: the split reduction's counters must be back at zero
        got = oc.conv(gpu, x, w, b, (pad, pad), (st, st), g, _abi.ACT_RELU, crsk=crsk, z=z)
        assert (np.abs(got - np.maximum(ref + z, 0)) <= (Cc // g * R * R + 2) * 2.0 ** -24 * (magnitude + np.abs(z))).all()


# N, C, H, W, K, pad: patches cut by every border, fewer channels than wavefronts and odd numbers of them, every number of filters
@pytest.mark.parametrize("case", [(1, 1, 1, 1, 1, 1), (2, 2, 17, 15, 2, 1), (1, 3, 16, 33, 3, 0), (2, 7, 20, 18, 4, 2), (1, 64, 90, 117, 3, 1), (3, 13, 5, 70, 1, 1)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("crsk", [False, True])
def test_conv_f32_3x3_with_at_most_four_filters(gpu, cpu, case, crsk):
    """Bound: each of the 9 C + 2 additions rounds by at most 2^-24 of the sum of magnitudes; a NaN stays in its windows."""
    import torch
    N, Cc, H, W, K, pad = case
    r = rng(sum(case))
    x = r.standard_normal((N, Cc, H, W)).astype(np.float32)
    w = (r.standard_normal((K, Cc, 3, 3)) * np.sqrt(2.0 / (9 * Cc))).astype(np.float32)
    b = r.uniform(-0.5, 0.5, K).astype(np.float32)
    conv64 = lambda t, f, v: torch.nn.functional.conv2d(*(torch.from_numpy(u).double() for u in (t, f, v)), padding=pad).numpy()  # noqa: E731
    ref, magnitude = conv64(x, w, b), conv64(np.abs(x), np.abs(w), np.abs(b))
    z = r.standard_normal(ref.shape).astype(np.float32)
    got = oc.conv(gpu, x, w, b, (pad, pad), (1, 1), 1, _abi.ACT_RELU, crsk=crsk, z=z, inplace=True)
    assert (np.abs(got - np.maximum(ref + z, 0)) <= (9 * Cc + 2) * 2.0 ** -24 * (magnitude + np.abs(z))).all()
    x[N - 1, Cc - 1, H // 2, W // 2] = np.nan
    got, ref = oc.conv(gpu, x, w, b, (pad, pad), (1, 1), 1, _abi.ACT_IDENTITY, crsk=crsk), oc.conv(cpu, x, w, b, (pad, pad), (1, 1), 1, _abi.ACT_IDENTITY)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))


def test_conv_3x3_by_minimal_filtering_keeps_infinities_in_their_place(gpu, cpu):
    """The transforms take differences within a 4x4 patch: an infinity, a NaN and values whose differences leave fp32's range
    must reach the results that use them and no others, as they do tap by tap."""
    r = rng(9)
    x = r.standard_normal((6, 48, 75, 77)).astype(np.float32)
    w = (r.standard_normal((100, 48, 3, 3)) * 0.1).astype(np.float32)
    b = r.uniform(-0.5, 0.5, 100).astype(np.float32)
    plain = [oc.conv(gpu, x, w, b, (1, 1), (1, 1), 1, _abi.ACT_IDENTITY, crsk=True, algo=a) for a in (1, _abi.CONV_ALGO_DIRECT)]
    assert (plain[0] != plain[1]).any()  # the kernel under test is the one that ran
    x[0, 3, 10, 20] = np.inf
    x[1, 5, 0, 0] = -np.inf
    x[2, 7, 74, 76] = np.nan
    x[3, 9, 30, 31], x[3, 9, 30, 33] = 3e38, -3e38
    w[5, 11, 1, 1] = np.inf
    ref = oc.conv(cpu, x, w, b, (1, 1), (1, 1), 1, _abi.ACT_IDENTITY)
    got = oc.conv(gpu, x, w, b, (1, 1), (1, 1), 1, _abi.ACT_IDENTITY, crsk=True)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(ref))
    ok = np.isfinite(ref)
    ok[3] = False  # its values of 3e38 are summed in another order, and so rounded differently
    np.testing.assert_allclose(got[ok], ref[ok], rtol=RTOL, atol=ATOL)
    far = np.isfinite(ref[3]) & (np.abs(ref[3]) > 1e30)
    np.testing.assert_allclose(got[3][far], ref[3][far], rtol=RTOL)


@pytest.mark.parametrize("case", [(7, 64, 56, 56, 64), (22, 64, 56, 56, 64), (3, 512, 19, 19, 486), (2, 512, 28, 28, 256)], ids=["whole", "rest-split", "odd-rows", "split"])
def test_conv_3x3_by_minimal_filtering_recomputes_only_what_is_not_finite(gpu, case):
    """A NaN or an infinity reaches the results whose windows hold it, and of the finite results only those of the same 2x2
    tiles may change a bit; with a whole image of NaN, the other images keep theirs."""
    import torch
    N, Cc, H, W, K = case
    r = rng(Cc)
    x = np.maximum(r.standard_normal((N, Cc, H, W)), 0).astype(np.float32)
    w = (r.standard_normal((K, Cc, 3, 3)) * np.sqrt(2.0 / (9 * Cc))).astype(np.float32)
    w[2, 0] = w[2, Cc - 1] = 0
    b = r.uniform(-0.5, 0.5, K).astype(np.float32)
    run = lambda t, f=w: oc.conv(gpu, t, f, b, (1, 1), (1, 1), 1, _abi.ACT_IDENTITY, crsk=True)  # noqa: E731
    conv64 = lambda t, f=w: torch.nn.functional.conv2d(*(torch.from_numpy(u).double() for u in (t, f, b)), padding=1).numpy()  # noqa: E731
    plain = run(x)
    assert (plain != oc.conv(gpu, x, w, b, (1, 1), (1, 1), 1, _abi.ACT_IDENTITY, crsk=True, algo=_abi.CONV_ALGO_DIRECT)).any()
    for value in (np.nan, np.inf):
        y = x.copy()
        y[1, Cc - 1, 10, 7] = value
        y[0, 0, 0, 0] = value
        got, ref = run(y), conv64(y)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
        np.testing.assert_array_equal(np.isposinf(got), np.isposinf(ref))
        np.testing.assert_array_equal(np.isneginf(got), np.isneginf(ref))
        tiles = np.zeros((N, 1, H, W), bool)
        tiles[1, :, 8:12, 6:10] = True  # the tiles whose patches hold row 10, column 7
        tiles[0, :, 0:2, 0:2] = True
        tiles = np.broadcast_to(tiles, plain.shape)
        np.testing.assert_array_equal(got[~tiles], plain[~tiles])
        ok = np.isfinite(ref)
        np.testing.assert_allclose(got[ok], ref[ok], rtol=RTOL, atol=ATOL)
    y = x.copy()
    y[1] = np.nan
    got = run(y)
    assert np.isnan(got[1]).all()
    np.testing.assert_array_equal(np.delete(got, 1, 0), np.delete(plain, 1, 0))
    f = w.copy()
    f[3, 5, 1, 1] = np.nan
    got = run(x, f)
    assert np.isnan(got[:, 3]).all()
    np.testing.assert_array_equal(np.delete(got, 3, 1), np.delete(plain, 3, 1))
