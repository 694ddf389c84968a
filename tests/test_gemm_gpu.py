"""Prefill dequant-GEMM (yule_hip_quantized_gemm, Q4_0 / Q4_K / Q5_K / Q6_K / Q8_0 / Q8_K) on
the MFMA units: each row
of Y must equal the quantized matvec of the same row of X to the matvec bar
(max|y - y_ref| <= 1e-3 * ||y_ref||_2 / sqrt(N), y_ref the f64 dot of the
bit-exact dequantized weights with the bf16 row converted exactly to f32)."""
import sys

import numpy as np
import pytest

import oracle
from refgen import tolerance_bar
from yule_amd import DType, synth
from yule_amd.backend import YuleGpuError

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bf16_bits(x: np.ndarray) -> np.ndarray:
    """f32 -> bf16 (round to nearest even) as uint16."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def bf16_to_f32(b: np.ndarray) -> np.ndarray:
    return (b.astype(np.uint32) << 16).view(np.float32)


# f32 X: 2-norm error of a row's results.  The kernels' own figures are 1.3e-7
# to 1.7e-6; left out on the CPU, the low half of X makes it 2.3e-4, the low
# halves of the min term's columns 8e-5 (sums) and 4e-4 (mins), the third bf16
# part of the one-launch kernel 1.0e-5.
F32_REL = 4e-6


def rel_error(got, ref):
    """2-norm of the difference over 2-norm of the result, in f64."""
    return float(np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref))


def run_gemm(hip, dt, w, xb, M, N, K):
    hw, hx, hy = hip.upload(w), hip.upload(xb), hip.allocate(4 * M * N)
    hip.quantized_gemm(hw, hx, hy, M, N, K, dt)
    y = hip.download(hy, (M, N))
    for h in (hw, hx, hy):
        hip.free(h)
    return y


@pytest.mark.parametrize("dt", [DType.Q4_K, DType.Q6_K, DType.Q8_0, DType.Q4_0, DType.Q5_K, DType.Q8_K],
                         ids=lambda d: d.name)
@pytest.mark.parametrize("M,N,K", [(1, 128, 256), (7, 300, 512), (64, 256, 1024), (130, 129, 2048), (65, 200, 5632)])
def test_gemm_rows_match_oracle(hip, dt, M, N, K):
    say(f"[gemm] {dt.name} M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 50 + M, N, K)
    xb = bf16_bits(synth.gauss(60 + K, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in range(M):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"


@pytest.mark.parametrize("M", [64, 512])
@pytest.mark.parametrize("N,K", [(14336, 4096), (4096, 14336)])
def test_gemm_config_shapes(hip, N, K, M):
    """BASELINE configs[3] shapes at M = 64 and 512, sampled rows vs the
    oracle; every seventh row against the GPU matvec of the same row."""
    dt = DType.Q4_K
    say(f"[gemm] Q4_K {N}x{K} M={M}")
    w = synth.gen_quant(dt, 70, N, K)
    xb = bf16_bits(synth.gauss(71, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in (0, 17, 63, M - 1):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
    hw, hx, hy = hip.upload(w), hip.allocate(4 * K), hip.allocate(4 * N)
    for m in range(0, M, 7):
        hip.copy_to_device(xf[m], hx)
        hip.quantized_matmul(hw, hx, hy, N, K, dt)
        mv = hip.download(hy, N)
        assert np.max(np.abs(y[m] - mv)) <= 2 * tolerance_bar(mv), f"row {m} vs matvec"
    for h in (hw, hx, hy):
        hip.free(h)


@pytest.mark.parametrize("dt,M,N,K", [(DType.Q4_K, 1024, 300, 1024), (DType.Q4_K, 1100, 513, 512),
                                      (DType.Q6_K, 512, 260, 768), (DType.Q6_K, 1030, 129, 256),
                                      (DType.Q8_0, 1024, 300, 1024), (DType.Q4_0, 1100, 513, 512),
                                      (DType.Q5_K, 1024, 300, 1024), (DType.Q8_K, 1030, 129, 512)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_gemm_wide_tiles(hip, dt, M, N, K):
    """M large enough for the 128 x 256 tiles (eight waves), ragged N and M:
    sampled rows vs the oracle, every row vs the GPU matvec of that row."""
    say(f"[gemm] wide tiles {dt.name} M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 90 + M, N, K)
    xb = bf16_bits(synth.gauss(91 + K, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in (0, 1, 127, 128, 255, M // 2, M - 1):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
    hw, hx, hy = hip.upload(w), hip.allocate(4 * K), hip.allocate(4 * N)
    for m in range(M):
        hip.copy_to_device(xf[m], hx)
        hip.quantized_matmul(hw, hx, hy, N, K, dt)
        mv = hip.download(hy, N)
        assert np.max(np.abs(y[m] - mv)) <= 2 * tolerance_bar(mv), f"row {m} vs matvec"
    for h in (hw, hx, hy):
        hip.free(h)


@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (13, 77, 2304), (16, 200, 4096), (5, 33, 8448), (16, 4096, 4096),
                                   (17, 200, 4096)])
def test_gemm_few_rows_q8_0(hip, M, N, K):
    """Q8_0, M <= 16: the one-launch kernel (one unit for one wave, nine units
    and 33 over 16 waves, a ragged last tile), bf16 and f32 X, every row vs the
    oracle; f32 X spread over 60 powers of two and a row near the top of the
    range, whose outputs are finite; M = 17 is the tile kernel's."""
    dt = DType.Q8_0
    say(f"[gemm] few rows Q8_0 M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 130 + M, N, K)
    xb = bf16_bits(synth.gauss(131 + K, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    xf = bf16_to_f32(xb).reshape(M, K)
    x32 = synth.gauss(132 + K, (M, K)) * np.exp2(np.arange(M, dtype=np.float32) * 4 - 30)[:, None].astype(np.float32)
    if M == 13:
        x32[12] *= np.float32(2.0 ** 102)   # quants times it pass the f32 range, the scaled outputs do not
    y32 = run_gemm_f32(hip, dt, w, x32, M, N, K)
    for m in range(M):
        for got, x in ((y, xf), (y32, x32)):
            ref = oracle.qmv_f64(int(dt), w, x[m], N, K)
            assert np.max(np.abs(ref)) < 3e38 and np.max(np.abs(got[m] - ref)) <= tolerance_bar(ref), f"row {m}"
            assert N < 30 or rel_error(got[m], ref) <= F32_REL, f"row {m}"   # (bf16 X is exact here)


@pytest.mark.parametrize("M,N,K", [(3, 40, 5632), (3, 4096, 14080), (3, 4097, 5632), (3, 4097, 5888), (3, 8193, 3584),
                                   (3, 8193, 3840), (8, 16384, 2816), (3, 16385, 256), (8, 100, 14080), (9, 100, 12032), (9, 100, 12544),
                                   (3, 100, 14592), (9, 100, 7168), (9, 100, 9216), (9, 4097, 4608), (3, 100, 6144)])
@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "f32"])
def test_gemm_few_rows_q8_0_line(hip, M, N, K, f32):
    """Either side of the line between the one-launch kernel and the tiles (one,
    two, three, four and five rounds of workgroups; up to 55 units over 16
    waves; more than eight rows; a width of whole 2048s)."""
    dt = DType.Q8_0
    say(f"[gemm] few rows Q8_0 {N}x{K} {'f32' if f32 else 'bf16'} X")
    w, x = synth.gen_quant(dt, 160, N, K), synth.gauss(161 + K, (M, K))
    if f32:
        got = run_gemm_f32(hip, dt, w, x, M, N, K)
    else:
        xb = bf16_bits(x)
        got, x = run_gemm(hip, dt, w, xb, M, N, K), bf16_to_f32(xb).reshape(M, K)
    for m in range(M):
        assert rel_error(got[m], oracle.qmv_f64(int(dt), w, np.ascontiguousarray(x[m]), N, K)) <= F32_REL, f"row {m}"


@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "f32"])
def test_gemm_few_rows_q8_0_small_rows(hip, f32):
    """The one-launch kernel on rows far below 1: as exact as ordinary ones down
    to the subnormals (f32 sums of 2304 terms: well under 4e-6), alone, beside
    ordinary rows, a zero row, a row whose 256-column units differ, and weight
    rows of zeros."""
    N, K, dt = 96, 2304, DType.Q8_0
    say(f"[gemm] few rows Q8_0, small rows, {'f32' if f32 else 'bf16'} X")
    w = synth.gen_quant(dt, 150, N, K)
    w.reshape(N, -1)[[17, 90]] = 0
    scale = np.float32(2.0) ** np.array([-118, -122, -100, -64, 0, -63, -125, -90, 0], np.float32)
    x = synth.gauss(151, (9, K)) * scale[:, None]
    x[8, 256:] *= np.float32(2.0 ** -120)      # one ordinary unit, eight small ones
    x[7, :] = 0
    if f32:
        got = run_gemm_f32(hip, dt, w, x, 9, N, K)
    else:
        xb = bf16_bits(x)
        got, x = run_gemm(hip, dt, w, xb, 9, N, K), bf16_to_f32(xb).reshape(9, K)
    for m in range(9):
        ref = oracle.qmv_f64(int(dt), w, np.ascontiguousarray(x[m]), N, K).astype(np.float64)
        if m == 7:
            assert not np.any(got[m])
        else:
            # results next to the smallest normal f32 carry its spacing, 2^-149
            assert rel_error(got[m], ref) <= F32_REL + 2.0 ** -148 * np.sqrt(N) / np.linalg.norm(ref), f"row {m}"


@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "f32"])
def test_gemm_few_rows_q8_0_non_finite(hip, f32):
    """The one-launch kernel on infinite and NaN scales and X: rows of X of any
    magnitude and zero rows give what the sums in f64 give (an infinity may be
    NaN where its block has quants of both signs or zero)."""
    N, K, dt = 32, 768, DType.Q8_0
    say(f"[gemm] few rows Q8_0, non-finite, {'f32' if f32 else 'bf16'} X")
    w = synth.gen_quant(dt, 175, N, K)
    d = w.reshape(N, K // 32, 34)[:, :, :2].view(np.float16)
    d[3, 2], d[5, 9], d[7, 20] = np.inf, np.nan, -np.inf
    x = bf16_to_f32(bf16_bits(synth.gauss(176, (5, K)))) * np.array([1, 2.0 ** -110, 0, 1, 2.0 ** -110], np.float32)[:, None]
    x[3, 300], x[4, 300] = np.inf, np.nan
    got = run_gemm_f32(hip, dt, w, x, 5, N, K) if f32 else run_gemm(hip, dt, w, bf16_bits(x), 5, N, K)
    bad = np.zeros((5, N), bool)
    bad[:, [3, 5, 7]] = True
    bad[3:] = True
    assert np.array_equal(~np.isfinite(got), bad)
    assert np.all(np.isnan(got[:, 5])) and np.all(np.isnan(got[2, [3, 7]]))


@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "f32"])
def test_gemm_few_rows_q8_0_large_partial_sums(hip, f32):
    """The one-launch kernel where a wave's partial sum passes the f32 range and
    the result does not: the second 256 columns' weights repeat the first's,
    their X is the first's times -127/128 (an f32 sum's error then counts 255
    times)."""
    N, K, dt = 64, 512, DType.Q8_0
    say(f"[gemm] few rows Q8_0, large partial sums, {'f32' if f32 else 'bf16'} X")
    w = synth.gen_quant(dt, 170, N, K, 8.0).reshape(N, 2, -1)
    w[:, 1] = w[:, 0]
    x = bf16_to_f32(bf16_bits(synth.gauss(171, (2, 256)))) * np.float32(2.0 ** 123)
    x = np.concatenate([x, x * np.float32(-127 / 128)], axis=1)
    if f32:
        got = run_gemm_f32(hip, dt, w, x, 2, N, K)
    else:
        xb = bf16_bits(x)
        got, x = run_gemm(hip, dt, w, xb, 2, N, K), bf16_to_f32(xb).reshape(2, K)
    d = w.reshape(N, K // 32, 34)[:, :, :2].copy().view(np.float16).astype(np.float64)
    wf = (d * w.reshape(N, K // 32, 34)[:, :, 2:].view(np.int8)).reshape(N, K)
    for m in range(2):
        part, ref = wf[:, :256] @ x[m, :256].astype(np.float64), wf @ x[m].astype(np.float64)
        assert np.max(np.abs(part)) > 2.0 ** 128 > 2 * np.max(np.abs(ref))
        assert rel_error(got[m], ref) <= 255 * F32_REL, f"row {m}"


@pytest.mark.parametrize("M,N,K", [(1, 77, 1024), (5, 300, 3072), (16, 64, 2048), (17, 129, 1024),
                                   (32, 200, 3072), (32, 1000, 2048), (8, 4096, 5120), (3, 2000, 14336),
                                   (33, 1000, 2048)])
def test_gemm_few_rows(hip, M, N, K):
    """Q4_K, M <= 32 and K / 256 a multiple of 4: the streaming kernel for
    few X rows (one or two 16-row X tiles; ragged N and M; K splits of one,
    two, five and fourteen super-block groups), every row vs the oracle;
    M = 33 is the tile kernel's again."""
    dt = DType.Q4_K
    say(f"[gemm] few rows Q4_K M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 110 + M, N, K)
    xb = bf16_bits(synth.gauss(111 + K, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in range(M):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"


@pytest.mark.parametrize("N,K", [(14336, 4096), (4096, 14336)])
def test_gemm_config_shapes_m2048(hip, N, K):
    """BASELINE configs[3] at M=2048, on the 256 x 256 tiles (128 x 64 per
    wave, accumulators rescaled per super-block): 14336x4096 is 448 tiles,
    4096x14336 128 tiles in two K splits.  Rows at tile edges and in the
    last tiles vs the oracle, and a repeat call bit-identical."""
    dt, M = DType.Q4_K, 2048
    say(f"[gemm] Q4_K {N}x{K} M={M}")
    w = synth.gen_quant(dt, 72, N, K)
    xb = bf16_bits(synth.gauss(73, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    assert np.array_equal(y, run_gemm(hip, dt, w, xb, M, N, K)), "second call differs"
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in (0, 255, 256, 1663, 1664, 1800, 2047):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"


# Shapes whose tile count passes a whole round of resident workgroups (256
# CUs: one 128 x 256 tile or two 128 x 128 tiles per CU) by at most half a
# round: the last tiles then run as two K halves added into zeroed y.  The
# last two cases take the 64-row tiles (M <= 64) with lm_head-like widths.
@pytest.mark.parametrize("dt,M,N,K", [(DType.Q4_K, 1024, 8348, 512), (DType.Q4_K, 1100, 7673, 768),
                                      (DType.Q5_K, 1024, 8348, 512), (DType.Q6_K, 512, 16590, 512),
                                      (DType.Q8_0, 512, 16512, 512), (DType.Q4_0, 1024, 8348, 512),
                                      (DType.Q8_K, 1024, 8348, 512), (DType.Q4_K, 40, 66000, 512),
                                      (DType.Q6_K, 64, 65800, 768)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_gemm_tail_halves(hip, dt, M, N, K):
    """The last m tiles (where the split tail tiles lie) vs the oracle, every
    row vs the GPU matvec, and a second call bit-identical to the first."""
    say(f"[gemm] tail halves {dt.name} M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 70 + M, N, K)
    xb = bf16_bits(synth.gauss(71 + K, (M, K)))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    assert np.array_equal(y, run_gemm(hip, dt, w, xb, M, N, K)), "second call differs"
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in sorted({0, max(M - 129, 0), max(M - 128, 0), max(M - 65, 0), M - 2, M - 1}):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
    hw, hx, hy = hip.upload(w), hip.allocate(4 * K), hip.allocate(4 * N)
    for m in range(M):
        hip.copy_to_device(xf[m], hx)
        hip.quantized_matmul(hw, hx, hy, N, K, dt)
        mv = hip.download(hy, N)
        assert np.max(np.abs(y[m] - mv)) <= 2 * tolerance_bar(mv), f"row {m} vs matvec"
    for h in (hw, hx, hy):
        hip.free(h)


ALL_GEMM = [DType.Q4_K, DType.Q6_K, DType.Q8_0, DType.Q4_0, DType.Q5_K, DType.Q8_K]


def range_rows(K: int) -> np.ndarray:
    """Rows that leave f16's range or precision unscaled: magnitudes 1e5 and
    1e36, 1e-7 and 1e-30, a row of 2100s (sub-block sums of 67200 > 65504),
    a row of small values holding two 3e38 elements, zeros, and N(0,1)."""
    g = np.random.default_rng(K)
    n = lambda: g.standard_normal(K)
    big = 1e-3 * n()
    big[[5, K - 7]] = 3e38
    rows = [1e5 * n(), 1e36 * n(), 1e-7 * n(), 1e-30 * n(), np.full(K, 2100.0), big, np.zeros(K), n()]
    return np.array(rows, np.float32)


@pytest.mark.parametrize("dt", ALL_GEMM, ids=lambda d: d.name)
@pytest.mark.parametrize("M", [8, 136])
def test_gemm_bf16_full_range(hip, dt, M):
    """Any finite bf16 row: each row against the oracle's f64 dot of the same
    bf16-valued row (the per-row power-of-two scale is exact)."""
    N, K = 160, 1024
    say(f"[gemm] bf16 range rows {dt.name} M={M}")
    w = synth.gen_quant(dt, 95, N, K)
    base = range_rows(K)
    xb = bf16_bits(np.concatenate([base] * (M // len(base)) + [base[:M % len(base)]]))
    y = run_gemm(hip, dt, w, xb, M, N, K)
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in range(M):
        ref = oracle.qmv_f64(int(dt), w, xf[m], N, K)
        if not np.any(xf[m]):
            assert np.all(y[m] == 0.0), f"row {m}"
            continue
        assert np.all(np.isfinite(y[m])), f"row {m}"
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"


def run_gemm_f32(hip, dt, w, x, M, N, K):
    hw, hx, hy = hip.upload(w), hip.upload(np.ascontiguousarray(x, np.float32)), hip.allocate(4 * M * N)
    hip.quantized_gemm_f32(hw, hx, hy, M, N, K, dt)
    y = hip.download(hy, (M, N))
    for h in (hw, hx, hy):
        hip.free(h)
    return y


@pytest.mark.parametrize("dt", ALL_GEMM, ids=lambda d: d.name)
@pytest.mark.parametrize("M,N,K", [(1, 128, 256), (7, 300, 512), (128, 2560, 2048), (128, 2048, 5632),
                                   (130, 129, 2048), (1024, 300, 1024)])
def test_gemm_f32_rows_match_oracle(hip, dt, M, N, K):
    """f32 X (hi + lo on the matrix cores): rows against the oracle's f64 dot
    of the same f32 row, and against the GPU's f32 matvec of that row."""
    say(f"[gemm f32] {dt.name} M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 110 + M, N, K)
    x = synth.gauss(111 + K, (M, K))
    y = run_gemm_f32(hip, dt, w, x, M, N, K)
    rows = sorted({0, M // 2, M - 1} | set(range(0, M, max(1, M // 8))))
    for m in rows:
        ref = oracle.qmv_f64(int(dt), w, x[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
    hw, hx, hy = hip.upload(w), hip.allocate(4 * K), hip.allocate(4 * N)
    for m in rows:
        hip.copy_to_device(x[m], hx)
        hip.quantized_matmul(hw, hx, hy, N, K, dt)
        mv = hip.download(hy, N)
        assert np.max(np.abs(y[m] - mv)) <= tolerance_bar(mv), f"row {m} vs matvec"
    for h in (hw, hx, hy):
        hip.free(h)


@pytest.mark.parametrize("dt", [DType.Q4_K, DType.Q6_K, DType.Q8_0], ids=lambda d: d.name)
def test_gemm_f32_full_range_and_repeat(hip, dt):
    """f32 rows of any magnitude, and a second call bit-identical (the lo
    product adds into Y in a fixed order: split-K at M = 16, whole tiles at
    M = 1024 where the bf16 call would split its tail tiles)."""
    K = 1024
    say(f"[gemm f32] range rows and repeat {dt.name}")
    w = synth.gen_quant(dt, 120, 160, K)
    x = range_rows(K)
    y = run_gemm_f32(hip, dt, w, x, len(x), 160, K)
    for m in range(len(x)):
        ref = oracle.qmv_f64(int(dt), w, x[m], 160, K)
        if not np.any(x[m]):
            assert np.all(y[m] == 0.0)
            continue
        assert np.all(np.isfinite(y[m])) and np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
    for M, N, KK in ((16, 4096, 4096), (1024, 8348, 512)):
        w2 = synth.gen_quant(dt, 121, N, KK)
        x2 = synth.gauss(122, (M, KK))
        a = run_gemm_f32(hip, dt, w2, x2, M, N, KK)
        assert np.array_equal(a, run_gemm_f32(hip, dt, w2, x2, M, N, KK)), f"M={M}: second call differs"
        ref = oracle.qmv_f64(int(dt), w2, x2[M - 1], N, KK)
        assert np.max(np.abs(a[M - 1] - ref)) <= tolerance_bar(ref)


def test_gemm_operand_tiles(hip):
    """The operand-tile path at the edges of its tiles, all formats, bf16 and
    f32 X (tests/gemm_tiled_check.py, in a child process because the switch
    that sends small products there is read once per process)."""
    import os
    import subprocess
    from pathlib import Path
    say("[gemm] operand tiles")
    r = subprocess.run([sys.executable, str(Path(__file__).with_name("gemm_tiled_check.py"))],
                       env=dict(os.environ, YULE_GEMM_TILED_MIN="1"), capture_output=True, text=True, timeout=110)
    out = r.stdout.strip().splitlines()
    assert r.returncode == 0 and out and out[-1].startswith("ok"), r.stdout[-2000:] + r.stderr[-4000:]
    say(f"[gemm] {out[-1]}")


# Q6_K with bf16 X, 129..511 rows: shapes on either side of the line between
# 128- and 256-wide tiles (few tiles, 16, 32 to 64, by cost, one round unsplit)
@pytest.mark.parametrize("M,N,K", [(132, 612, 3328), (490, 1247, 1280), (129, 2048, 2048), (129, 2048, 1792), (200, 4100, 1024),
                                   (300, 1536, 4096), (129, 2817, 14336), (140, 14336, 1024), (511, 7000, 2048)])
def test_gemm_q6k_tile_widths(hip, M, N, K):
    say(f"[gemm] Q6_K bf16 M={M} N={N} K={K}")
    w = synth.gen_quant(DType.Q6_K, 180, N, K)
    xb = bf16_bits(synth.gauss(181 + M, (M, K)))
    y, xf = run_gemm(hip, DType.Q6_K, w, xb, M, N, K), bf16_to_f32(xb).reshape(M, K)
    for m in (0, 127, 128, M - 1):
        ref = oracle.qmv_f64(int(DType.Q6_K), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"


# Q6_K on either side of the operand tiles' line: bf16 X by tiles, columns of
# tiles and rows; f32 X below 512 rows by whole tiles and columns of them
@pytest.mark.parametrize("M,N,K,f32", [(768, 2048, 8192, False), (768, 2305, 8192, False), (1290, 1100, 11520, False),
                                       (1270, 1100, 11520, False), (257, 2048, 2816, True), (256, 2048, 4096, True),
                                       (300, 512, 14336, True)])
def test_gemm_q6k_operand_tile_line(hip, M, N, K, f32):
    say(f"[gemm] Q6_K {'f32' if f32 else 'bf16'} X M={M} N={N} K={K}")
    w, x = synth.gen_quant(DType.Q6_K, 190, N, K), synth.gauss(191 + M, (M, K))
    if f32:
        y = run_gemm_f32(hip, DType.Q6_K, w, x, M, N, K)
    else:
        xb = bf16_bits(x)
        y, x = run_gemm(hip, DType.Q6_K, w, xb, M, N, K), bf16_to_f32(xb).reshape(M, K)
    for m in (0, 128, M - 1):
        ref = oracle.qmv_f64(int(DType.Q6_K), w, np.ascontiguousarray(x[m]), N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
        assert not f32 or rel_error(y[m], ref) <= F32_REL, f"row {m}"


# Q6_K: partials of the 256-wide tiles' K splits that do and do not fit the
# static workspace (then the 128-wide tiles serve the call)
@pytest.mark.parametrize("M", [130, 384, 511])
def test_gemm_noalloc_q6k_partials(hip, M):
    N = K = 4096
    say(f"[gemm noalloc] Q6_K M={M}")
    w = synth.gen_quant(DType.Q6_K, 140, N, K)
    xb = bf16_bits(synth.gauss(141, (M, K)))
    hw, hx, hy = hip.upload(w), hip.upload(xb), hip.allocate(4 * M * N)
    hip.quantized_gemm_noalloc(hw, hx, hy, M, N, K, DType.Q6_K)
    y = hip.download(hy, (M, N))
    xf = bf16_to_f32(xb).reshape(M, K)
    for m in (0, M - 1):
        ref = oracle.qmv_f64(int(DType.Q6_K), w, xf[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
    for h in (hw, hx, hy):
        hip.free(h)


# products that the size rule itself sends to the operand tiles, one K split
# and several, and the first row count on either side of the line
@pytest.mark.parametrize("dt,M,N,K", [(DType.Q6_K, 129, 3900, 3072), (DType.Q6_K, 128, 3900, 3072),
                                      (DType.Q8_0, 300, 5000, 2048), (DType.Q4_K, 700, 11264, 2048),
                                      (DType.Q5_K, 699, 11264, 2048), (DType.Q4_0, 200, 4096, 4096)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_gemm_f32_many_rows(hip, dt, M, N, K):
    say(f"[gemm f32] many rows {dt.name} M={M} N={N} K={K}")
    w = synth.gen_quant(dt, 130 + M, N, K)
    x = synth.gauss(131 + K, (M, K))
    y = run_gemm_f32(hip, dt, w, x, M, N, K)
    for m in (0, M // 2, M - 1):
        ref = oracle.qmv_f64(int(dt), w, x[m], N, K)
        assert np.max(np.abs(y[m] - ref)) <= tolerance_bar(ref), f"row {m}"
        assert rel_error(y[m], ref) <= F32_REL, f"row {m}"


def test_gemm_errors(hip):
    w = synth.gen_quant(DType.Q4_K, 1, 16, 256)
    hw, hx, hy = hip.upload(w), hip.allocate(2 * 256 * 4), hip.allocate(4 * 16 * 4)
    with pytest.raises(YuleGpuError):
        hip.quantized_gemm(hw, hx, hy, 4, 16, 256, DType.F16)       # not on the MFMA path
    with pytest.raises(YuleGpuError):
        hip.quantized_gemm(hw, hx, hy, 5, 16, 256, DType.Q4_K)      # x too small
    with pytest.raises(YuleGpuError):
        hip.quantized_gemm(hw, hx, hx, 1, 16, 256, DType.Q4_K)      # x aliases y
    with pytest.raises(YuleGpuError):
        hip.quantized_gemm(hw, hx, hw, 1, 16, 256, DType.Q4_K)      # weights alias y
    with pytest.raises(YuleGpuError):
        hip.quantized_gemm(hw, hw, hy, 1, 16, 256, DType.Q4_K)      # weights alias x
    for h in (hw, hx, hy):
        hip.free(h)
