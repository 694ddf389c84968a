"""Child-process check for tests/test_runner_gpu.py: the batched prompt pass
with every projection through the operand tiles (YULE_GEMM_TILED_MIN=1, read
once per process, set by the parent): RMSNorm and SwiGLU on the way into the X
tiles, a pending split-K reduction there with and without adding into the
residual rows, the output and down products added into them by the epilogue,
and matrices of one format stacked (Q/K/V, gate|up) or, in mixed formats, one
by one.  A prompt of a few rows, one of ragged tiles, and one long enough for
four rows of X a workgroup; logits vs the oracle after each, and of decode
steps that read the rows' K and V.  Prints "ok <max err / bar>" or raises."""
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
sys.path[:0] = [str(ROOT), str(ROOT / "tests")]

import numpy as np  # noqa: E402

import oracle  # noqa: E402
from refgen import tolerance_bar  # noqa: E402
from yule_amd import synth  # noqa: E402
from yule_amd.backend import HipBackend, HipRunner  # noqa: E402
from yule_amd.model import LlamaConfig, SyntheticModel  # noqa: E402

# K splits need four super-blocks: dim 512 and ff 1024 split the down product
# (left, added, to the next layer's norm), dim 1024 and ff 512 the output
# product (left to the gate|up norm) and gate|up (left to the SwiGLU)
SHAPES = [(512, 1024), (1024, 512), (1024, 1024)]
SCHEMES = ["Q4_K_M", "Q6_K", "Q8_0", "Q5_K", "Q4_0"]
PIECES = (5, 67)


def check(hip, cfg, scheme, pieces):
    m = SyntheticModel.generate(cfg, seed=51, scheme=scheme)
    toks, at, worst = synth.uniform_tokens(52, sum(pieces) + 3, cfg.vocab), 0, 0.0
    run, ref = HipRunner(hip, m), oracle.Runner(m, n_threads=8)
    for n in pieces + (1, 1, 1):
        got = run.decode_step(int(toks[at])) if n == 1 else run.prefill_batched(toks[at:at + n])
        for t in toks[at:at + n]:
            want = ref.forward(int(t))
        at += n
        worst = max(worst, float(np.max(np.abs(got - want))) / tolerance_bar(want))
    run.close()
    assert worst <= 1.0, f"{cfg} {scheme} {pieces}: {worst:.3g} of the bar"
    print(f"# {cfg.dim}/{cfg.ff_dim} {scheme} {pieces} {worst:.3f}", flush=True)
    return worst


def main():
    worst = 0.0
    with HipBackend(0) as hip:
        for dim, ff in SHAPES:
            for scheme in SCHEMES:
                cfg = LlamaConfig(n_layers=3, dim=dim, n_heads=dim // 64, n_kv_heads=4, ff_dim=ff, vocab=512, max_seq=96)
                worst = max(worst, check(hip, cfg, scheme, PIECES))
        for scheme in ("Q4_K_M", "Q6_K"):
            cfg = LlamaConfig(n_layers=2, dim=512, n_heads=8, n_kv_heads=4, ff_dim=1024, vocab=512, max_seq=1100)
            worst = max(worst, check(hip, cfg, scheme, (1030,)))
    print(f"ok {worst:.3f}", flush=True)


if __name__ == "__main__":
    main()
