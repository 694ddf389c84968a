"""Device memory is returned: backends, their workspace, buffers and runners
created and destroyed repeatedly leave the free device memory where it was
(hipMemGetInfo, read through the HIP runtime the library itself links)."""
import ctypes as C
import sys

import numpy as np
import pytest

import oracle
from refgen import tolerance_bar
from yule_amd import DType, synth
from yule_amd.backend import HipBackend, HipRunner, YuleGpuError
from yule_amd.model import TINY_TEST, LlamaConfig, SyntheticModel

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def free_bytes() -> int:
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def cycle(model):
    be = HipBackend(0)
    w = be.upload(synth.gen_quant(DType.Q4_K, 5, 512, 1024))
    xb = (synth.gauss(6, (300, 1024)).view(np.uint32) >> 16).astype(np.uint16)
    hx, hy = be.upload(xb), be.allocate(4 * 300 * 512)
    be.quantized_gemm(w, hx, hy, 300, 512, 1024, DType.Q4_K)        # grows the backend workspace
    be.gqa_decode_attn(be.allocate(4 * 8 * 64), be.upload(np.zeros((600, 2 * 64), np.float32)),
                       be.upload(np.zeros((600, 2 * 64), np.float32)), be.allocate(4 * 8 * 64), 8, 2, 64, 600)
    run = HipRunner(be, model)
    run.generate_greedy(synth.uniform_tokens(3, 4, model.cfg.vocab), 4)
    run.close()
    be.synchronize()
    be.close()                                                      # frees buffers and workspace


def test_no_device_memory_growth():
    print("[resources] backend / runner create-destroy cycles", flush=True)
    sys.stdout.flush()
    model = SyntheticModel.generate(TINY_TEST, seed=2)
    cycle(model)                     # first cycle: runtime and code-object setup
    base = free_bytes()
    for _ in range(5):
        cycle(model)
    drift = base - free_bytes()
    assert drift < 16 << 20, f"free device memory fell by {drift} bytes over 5 cycles"


def test_gemm_without_room_for_operand_tiles(hip, monkeypatch):
    """Where the operand tiles' workspace cannot be had, the plan that needs
    least serves the call: a limit on allocations, then a capture, under which
    the workspace cannot grow (replays against the eager result).  Below that
    plan's needs too, the call is refused and the backend goes on."""
    M, N, K, dt = 300, 2048, 5632, DType.Q6_K   # 59 MB as operand tiles, 19 MB without
    say("[resources] gemm f32 Q6_K under a workspace limit, then captured")
    w, x = synth.gen_quant(dt, 5, N, K), synth.gauss(6, (M, K))
    monkeypatch.setenv("YULE_WORKSPACE_LIMIT_MB", "8")
    with HipBackend(0) as be:
        hw, hx, hy = be.upload(w), be.upload(x), be.allocate(4 * M * N)
        with pytest.raises(YuleGpuError, match="LIMIT"):
            be.quantized_gemm_f32(hw, hx, hy, M, N, K, dt)
        monkeypatch.setenv("YULE_WORKSPACE_LIMIT_MB", "24")
        be.quantized_gemm_f32(hw, hx, hy, M, N, K, dt)
        small = be.download(hy, (M, N))
        monkeypatch.delenv("YULE_WORKSPACE_LIMIT_MB")
        be.capture_begin()
        try:
            be.quantized_gemm_f32(hw, hx, hy, M, N, K, dt)
        finally:
            be.capture_end()
        for _ in range(2):
            be.copy_to_device(np.full(M * N, np.nan, np.float32), hy)
            be.capture_replay()
            assert np.array_equal(be.download(hy, (M, N)), small)
        be.quantized_gemm_f32(hw, hx, hy, M, N, K, dt)   # with room: the operand tiles
        y = be.download(hy, (M, N))
    for m in (0, M - 1):
        ref = oracle.qmv_f64(int(dt), w, x[m], N, K)
        for got in (small, y):
            assert np.max(np.abs(got[m] - ref)) <= tolerance_bar(ref)


def test_prefill_without_room_for_operand_tiles(hip, monkeypatch):
    """The runner's batched prompt pass (95 MB of workspace for the operand
    tiles of the down products, 38 MB without) under a limit between the two,
    and refused below both."""
    say("[resources] prefill_batched under a workspace limit")
    m = SyntheticModel.generate(LlamaConfig(n_layers=1, dim=2048, n_heads=32, n_kv_heads=4, ff_dim=5632, vocab=256,
                                            max_seq=256), seed=7, scheme="Q4_K_M")
    toks = synth.uniform_tokens(8, 200, 256)
    got = []
    for limit in ("4", "48", "0"):
        monkeypatch.setenv("YULE_WORKSPACE_LIMIT_MB", limit)
        run = HipRunner(hip, m)
        try:
            if limit == "4":
                with pytest.raises(YuleGpuError, match="LIMIT"):
                    run.prefill_batched(toks)
            else:
                got.append(run.prefill_batched(toks))
        finally:
            run.close()
    assert np.max(np.abs(got[0] - got[1])) <= tolerance_bar(got[1])


def test_error_is_reported_once(hip):
    """A failed allocation is the failed call's error, not the next launch's."""
    say("[resources] failed allocation, then a launch")
    a = hip.upload(np.ones(8, np.float32))
    with pytest.raises(YuleGpuError):
        hip.allocate(1 << 60)
    hip.add(a, a, a, 8)
    assert np.array_equal(hip.download(a, 8), np.full(8, 2.0, np.float32))
    hip.free(a)
