"""Child-process check for tests/test_gemm_gpu.py: every product through the
operand-tile path (YULE_GEMM_TILED_MIN=1, read once per process, set by the
parent), at the edges of its tiles: one row and ragged rows, row counts of W
around 32 and 256, one super-block, extra-k padding, K splits; rows of X taken
four to a workgroup, of every 32-row tile; the tail tiles of one pass
and of several over a wide W (that the shapes have them is checked in
tests/test_gemm_plan.py); super-blocks whose d is zero (at the start, inside and at the end of a row), rows of any magnitude,
and repeats bit for bit.  Rows against the oracle's f64 dot.  Prints "ok <max
err / bar>" or raises."""
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
sys.path[:0] = [str(ROOT), str(ROOT / "tests")]

import numpy as np  # noqa: E402

import oracle  # noqa: E402
from refgen import tolerance_bar  # noqa: E402
from test_gemm_gpu import F32_REL, ALL_GEMM, bf16_bits, bf16_to_f32, range_rows, rel_error, run_gemm, run_gemm_f32  # noqa: E402
from yule_amd import DType, GEOMETRY, synth  # noqa: E402
from yule_amd.backend import HipBackend  # noqa: E402

D_AT = {DType.Q4_K: (0, 2), DType.Q5_K: (0, 2), DType.Q6_K: (208, 210), DType.Q8_K: (0, 4), DType.Q8_0: (0, 2),
        DType.Q4_0: (0, 2)}
SHAPES = [(1, 1, 256), (3, 31, 512), (33, 300, 2816), (129, 257, 1024), (130, 513, 2304)]
WIDE = [(DType.Q6_K, 130, 67000, 512), (DType.Q4_K, 2, 134000, 512), (DType.Q4_K, 2, 9300, 14336),
        (DType.Q6_K, 130, 67000, 1024), (DType.Q4_K, 130, 67000, 1024), (DType.Q4_K, 130, 153000, 1536)]
MANY_ROWS = (1030, 96, 512)   # four rows of X a workgroup


def weights(dt, seed, n, k):
    """Quantized rows, some super-blocks (or blocks) of which have d = 0."""
    w = synth.gen_quant(dt, seed, n, k)
    bs, bb = GEOMETRY[dt]
    b = w.reshape(n, k // bs, bb)
    lo, hi = D_AT[dt]
    for row in range(0, n, 3):
        b[row, [0, (k // bs) // 2, -1][row // 3 % 3], lo:hi] = 0
    if n > 4:
        b[4, :, lo:hi] = 0
    return w


def check(hip, dt, m, n, k, f32, x, rel=True):
    """rel: the 2-norm bar too, with f32 X and where results do not cancel to
    much less than their terms (few of them, or rows of one value)."""
    w = weights(dt, 7 * m + n, n, k)
    if f32:
        run, xs, xf = run_gemm_f32, x, x
    else:
        run, xs = run_gemm, bf16_bits(x)
        xf = bf16_to_f32(xs).reshape(m, k)
    y = run(hip, dt, w, xs, m, n, k)
    assert np.array_equal(y, run(hip, dt, w, xs, m, n, k)), "second call differs"
    worst = 0.0
    big = n * k > 1 << 25
    for i in range(m) if m > 1000 else sorted({0, 1 % m, m // 2, m - 1} | set(range(0 if big else min(m, 8)))):
        ref = oracle.qmv_f64(int(dt), w, np.ascontiguousarray(xf[i], np.float32), n, k)
        if not np.any(xf[i]):
            assert np.all(y[i] == 0.0), f"row {i}"
            continue
        assert np.all(np.isfinite(y[i])), f"row {i}"
        worst = max(worst, float(np.max(np.abs(y[i] - ref))) / tolerance_bar(ref))
        if f32 and rel and n >= 30:
            worst = max(worst, rel_error(y[i], ref) / F32_REL)
        if big:   # the last tiles by themselves
            cols = slice(n - 3000, n)
            worst = max(worst, float(np.max(np.abs(y[i, cols] - ref[cols]))) / tolerance_bar(ref[cols]))
            if f32:
                worst = max(worst, rel_error(y[i, cols], ref[cols]) / F32_REL)
    assert worst <= 1.0, f"{dt.name} m={m} n={n} k={k} f32={f32}: {worst:.3g} of the bar"
    return worst


def main():
    worst = 0.0
    with HipBackend(0) as hip:
        for f32 in (False, True):
            for dt in ALL_GEMM if f32 else [DType.Q6_K]:   # (the other formats have no tiles for bf16 X)
                for m, n, k in SHAPES:
                    worst = max(worst, check(hip, dt, m, n, k, f32, synth.gauss(m + k, (m, k))))
                worst = max(worst, check(hip, dt, 8, 160, 1024, f32, range_rows(1024), rel=False))
                worst = max(worst, check(hip, dt, *MANY_ROWS, f32, synth.gauss(5, MANY_ROWS[::2])))
                print(f"# {dt.name} f32={f32} {worst:.3f}", flush=True)
            for dt, m, n, k in WIDE if f32 else [c for c in WIDE if c[0] == DType.Q6_K]:
                worst = max(worst, check(hip, dt, m, n, k, f32, synth.gauss(m + k, (m, k))))
                print(f"# wide {dt.name} {n}x{k} f32={f32} {worst:.3f}", flush=True)
    print(f"ok {worst:.3f}", flush=True)


if __name__ == "__main__":
    main()
