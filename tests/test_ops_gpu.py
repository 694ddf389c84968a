"""The non-matvec ComputeBackend methods on the GPU, read like the
reference's CpuBackend tests (yule-gpu/src/cpu.rs:597-1157): known answers
from those tests (tests/golden/reference_kats.json) plus float64 numpy
references on seeded inputs."""
import math
import sys

import numpy as np
import pytest

import oracle
from refgen import kats
from yule_amd import synth
from yule_amd.backend import YuleGpuError

pytestmark = pytest.mark.gpu
K = kats()


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def f32(a):
    return np.asarray(a, dtype=np.float32)


def close(a, b, tol):
    return np.max(np.abs(np.asarray(a, np.float64) - np.asarray(b, np.float64))) <= tol


def test_allocate_zeroed_and_copies(hip):
    say("[ops] allocate / copies")
    h = hip.allocate(64)
    assert np.all(hip.download(h, 16) == 0)                        # cpu.rs:157 zero-initialised
    src, dst = hip.upload(f32([1, 2, 3, 4])), hip.allocate(16)
    hip.copy_buffer(src, dst, 16)
    assert list(hip.download(dst, 4)) == [1, 2, 3, 4]
    cache = hip.allocate(4 * 4 * 4)                                 # KV-cache write pattern (cpu.rs:805-857)
    hip.copy_buffer_offset(src, cache, 0, 2 * 16, 16)
    got = hip.download(cache, 16)
    assert list(got[8:12]) == [1, 2, 3, 4] and np.all(got[:8] == 0) and np.all(got[12:] == 0)
    with pytest.raises(YuleGpuError):
        hip.copy_buffer_offset(src, cache, 0, 60, 16)              # past the end of dst
    with pytest.raises(YuleGpuError):
        hip.copy_to_device(np.zeros(32, np.float32), src)          # larger than the buffer
    for b in (h, src, dst, cache):
        hip.free(b)
    hip.free(h)                                                     # unknown handles are ignored (cpu.rs free)


def test_rms_norm_softmax_elementwise(hip):
    say("[ops] rms_norm / softmax / silu / mul / add / silu_mul")
    n = 2048
    x, w, b = synth.gauss(1, n), synth.gauss(2, n), synth.gauss(3, n)
    hx, hw, hb, ho = hip.upload(x), hip.upload(w), hip.upload(b), hip.allocate(4 * n)
    xd, wd, bd = x.astype(np.float64), w.astype(np.float64), b.astype(np.float64)
    hip.rms_norm(hx, hw, ho, n, 1e-5)
    assert close(hip.download(ho, n), xd / np.sqrt(np.mean(xd * xd) + 1e-5) * wd, 1e-5)
    hip.softmax(hx, ho, n)
    e = np.exp(xd - xd.max())
    assert close(hip.download(ho, n), e / e.sum(), 1e-7)
    hip.silu(hx, ho, n)
    assert close(hip.download(ho, n), xd / (1 + np.exp(-xd)), 1e-6)
    hip.element_mul(hx, hb, ho, n)
    assert close(hip.download(ho, n), xd * bd, 1e-6)
    hip.add(hx, hb, ho, n)
    assert close(hip.download(ho, n), xd + bd, 1e-6)
    hip.silu_mul(hx, hb, ho, n)
    assert close(hip.download(ho, n), xd / (1 + np.exp(-xd)) * bd, 1e-5)
    for h in (hx, hw, hb, ho):
        hip.free(h)


def test_rope_kats_and_table(hip):
    say("[ops] rope")
    k0 = K["rope_pos0"]
    q, k = hip.upload(f32(k0["q"])), hip.upload(f32(k0["k"]))
    hip.rope(q, k, 0, 4, 10000.0, 1, 1)
    assert close(hip.download(q, 4), k0["expect_q"], 1e-5) and close(hip.download(k, 4), k0["expect_k"], 1e-5)
    hip.copy_to_device(f32(K["rope_pos5"]["q"]), q)
    hip.rope(q, k, 5, 4, 10000.0, 1, 1)
    got = hip.download(q, 4)
    assert abs(got[0] - math.cos(5.0)) < 1e-4 and abs(got[1] - math.sin(5.0)) < 1e-4
    # many heads, many positions vs the oracle's RopeTable (model_runner.rs:77-100)
    hd, nq, nk, pos = 64, 32, 4, 300
    qv, kv = synth.gauss(4, nq * hd), synth.gauss(5, nk * hd)
    hq, hk = hip.upload(qv), hip.upload(kv)
    hip.rope(hq, hk, pos, hd, 10000.0, nq, nk)
    c, s = oracle.rope_table(pos + 1, hd, 10000.0)
    c, s = c[pos * 32:(pos + 1) * 32], s[pos * 32:(pos + 1) * 32]

    def rot(v):
        v = v.reshape(-1, hd).astype(np.float64)
        o = v.copy()
        o[:, 0::2] = v[:, 0::2] * c - v[:, 1::2] * s
        o[:, 1::2] = v[:, 0::2] * s + v[:, 1::2] * c
        return o.reshape(-1)
    # device trig vs host libm: both round the same f32 formula; 1e-4 absolute on |x| ~ 3
    assert close(hip.download(hq, nq * hd), rot(qv), 1e-4) and close(hip.download(hk, nk * hd), rot(kv), 1e-4)
    for h in (q, k, hq, hk):
        hip.free(h)


def test_matmul_f32(hip):
    say("[ops] matmul")
    m, n, k = 3, 70, 129
    a, b = synth.gauss(6, (m, k)), synth.gauss(7, (k, n))
    ha, hb, hc = hip.upload(a), hip.upload(b), hip.allocate(4 * m * n)
    hip.matmul(ha, hb, hc, m, n, k)
    assert close(hip.download(hc, (m, n)), a.astype(np.float64) @ b.astype(np.float64), 1e-4)
    for h in (ha, hb, hc):
        hip.free(h)


def test_attn_score_value_kats(hip):
    say("[ops] attn_score / attn_value")
    a = K["attn_score"]
    q, kc, vc = hip.upload(f32(a["q"])), hip.upload(f32(a["k_cache"])), hip.upload(f32(a["v_cache"]))
    sc, out = hip.allocate(4 * 3), hip.allocate(4 * 8)
    hip.attn_score(q, kc, sc, 2, 3, 0, 0, 4)
    s = hip.download(sc, 3)
    assert close(s * math.sqrt(2), a["expect_scores_times_sqrt2"], 1e-5)
    hip.softmax(sc, sc, 3)
    hip.attn_value(sc, vc, out, 2, 3, 0, 4, 0)
    p = hip.download(sc, 3).astype(np.float64)
    V = np.array(a["v_cache"]).reshape(3, 4)[:, :2]
    assert close(hip.download(out, 2), p @ V, 1e-4)
    for h in (q, kc, vc, sc, out):
        hip.free(h)


@pytest.mark.parametrize("hd,nh,nkv,seq", [(2, 2, 1, 2), (64, 32, 4, 384), (128, 32, 8, 1000), (64, 8, 8, 1),
                                          (256, 8, 2, 200), (64, 32, 4, 600), (80, 8, 2, 77), (32, 4, 4, 33),
                                          (16, 8, 2, 100), (8, 4, 1, 50), (4, 4, 2, 300), (48, 8, 2, 200),
                                          (4, 32, 2, 1500), (16, 32, 2, 3000), (96, 32, 2, 1100)])
def test_gqa_decode_attn(hip, hd, nh, nkv, seq):
    say(f"[ops] gqa_decode_attn hd={hd} heads={nh}/{nkv} seq={seq}")
    if hd == 2:
        g = K["gqa_2to1"]
        q, kc, vc = f32(g["q"]), f32(g["k_cache"]), f32(g["v_cache"])
        with pytest.raises(YuleGpuError):           # head_dim must be a multiple of 4 here
            hip.gqa_decode_attn(hip.upload(q), hip.upload(kc), hip.upload(vc), hip.allocate(16), 2, 1, 2, 2)
        return
    run_gqa_case(hip, hd, nh, nkv, seq)


def gqa_ref(q, kc, vc, nh, nkv, hd):
    want = np.zeros(nh * hd)
    for h in range(nh):
        kv = h // (nh // nkv)
        Kh = kc[:, kv * hd:(kv + 1) * hd].astype(np.float64)
        s = Kh @ q[h * hd:(h + 1) * hd] / math.sqrt(hd)
        p = np.exp(s - s.max())
        p /= p.sum()
        want[h * hd:(h + 1) * hd] = p @ vc[:, kv * hd:(kv + 1) * hd]
    return want


def run_gqa_case(hip, hd, nh, nkv, seq, tol=1e-5):
    q, kc, vc = synth.gauss(8, nh * hd), synth.gauss(9, (seq, nkv * hd)), synth.gauss(10, (seq, nkv * hd))
    hq, hk, hv, ho = hip.upload(q), hip.upload(kc), hip.upload(vc), hip.allocate(4 * nh * hd)
    hip.gqa_decode_attn(hq, hk, hv, ho, nh, nkv, hd, seq)
    got = hip.download(ho, nh * hd)
    for h in (hq, hk, hv, ho):
        hip.free(h)
    want = gqa_ref(q, kc, vc, nh, nkv, hd)
    err = np.max(np.abs(got - want))
    assert err <= tol, f"max error {err:.3g}"


@pytest.mark.parametrize("hd,nh,nkv,seq", [(hd, nh, nkv, seq) for hd, nh, nkv in ((64, 4, 4), (128, 20, 2))
                                          for seq in (1, 16, 17, 128, 257, 511, 512)])
def test_gqa_decode_attn_per_head(hip, hd, nh, nkv, seq):
    """The one-workgroup-per-head kernel at the ends of a wave's positions and
    of its rounds; more than 8 heads per KV head, which never run split-KV,
    stay on it at 512."""
    say(f"[ops] per-head gqa_decode_attn hd={hd} heads={nh}/{nkv} seq={seq}")
    run_gqa_case(hip, hd, nh, nkv, seq)


@pytest.mark.parametrize("hd,nh,nkv,seq", [(64, 8, 2, 1), (64, 8, 2, 65), (64, 32, 4, 384), (128, 32, 8, 1000),
                                          (80, 8, 2, 77), (32, 4, 4, 33), (64, 24, 8, 300), (64, 40, 8, 500),
                                          (256, 16, 2, 129), (128, 56, 8, 257), (64, 4, 4, 700)])
def test_gqa_decode_attn_split_forced(hip, hd, nh, nkv, seq, monkeypatch):
    """The split-KV path (per-chunk max / sum / partial output, then the
    combine) at every group size 1..8 and every chunk length, forced on
    short sequences."""
    say(f"[ops] split gqa_decode_attn hd={hd} heads={nh}/{nkv} seq={seq}")
    monkeypatch.setenv("YULE_ATTN_SPLIT_MIN", "1")
    run_gqa_case(hip, hd, nh, nkv, seq)


@pytest.mark.parametrize("hd,nh,nkv,seq", [(64, 32, 4, 5000), (128, 32, 8, 9000), (64, 32, 4, 20000),
                                          (128, 64, 8, 17000)])
def test_gqa_decode_attn_long(hip, hd, nh, nkv, seq):
    """Long contexts: split-KV by default from 512 positions; above 16384
    (the one-workgroup-per-head kernel's LDS limit) it is the only path."""
    say(f"[ops] long gqa_decode_attn hd={hd} heads={nh}/{nkv} seq={seq}")
    run_gqa_case(hip, hd, nh, nkv, seq)


@pytest.mark.parametrize("hd,nh,nkv,seq", [(64, 8, 8, 20481), (128, 8, 8, 12097), (128, 16, 2, 82001),
                                          (64, 48, 16, 7937), (128, 32, 32, 2033)])
def test_gqa_decode_attn_chunk_lengths(hip, hd, nh, nkv, seq):
    """Split-KV chunks with a short last one (one key, or part of a 16-key
    sub-tile): the tile kernel's of 320, 256 and 256 positions (first, third
    and fourth case), the vector kernel's of 128."""
    say(f"[ops] gqa_decode_attn chunks hd={hd} heads={nh}/{nkv} seq={seq}")
    run_gqa_case(hip, hd, nh, nkv, seq)


@pytest.mark.parametrize("hd,nh,nkv,seq", [(64, 32, 32, 513), (64, 32, 32, 3327), (64, 32, 32, 3328), (128, 8, 8, 15359), (128, 8, 8, 16129),
                                          (64, 16, 16, 1536), (64, 16, 16, 1537), (80, 4, 4, 1536), (256, 2, 2, 1537)])
def test_gqa_decode_attn_one_query_head(hip, hd, nh, nkv, seq):
    """One query head per KV head: the vector kernel up to a length that goes by
    the heads, the tile kernel from there on; 24 and 25
    chunks, either side of the end of the combine's walk."""
    say(f"[ops] one query head per KV head, hd={hd} heads={nh}/{nkv} seq={seq}")
    run_gqa_case(hip, hd, nh, nkv, seq)


@pytest.mark.parametrize("hd,nh,nkv,seq", [(128, 16, 8, 12097), (64, 32, 8, 20481), (128, 24, 12, 12033), (64, 12, 4, 16385)])
def test_gqa_decode_attn_row_lengths(hip, hd, nh, nkv, seq):
    """The tile kernel's chunks by the length of a cache row: 192 and 320
    positions for 4096 and 2048 bytes, 256 and 128 for others, each with a
    short last chunk."""
    say(f"[ops] gqa_decode_attn rows of {4 * nkv * hd} bytes, seq={seq}")
    run_gqa_case(hip, hd, nh, nkv, seq)


def test_gqa_decode_attn_limits(hip):
    """More than 8 query heads per KV head: the per-head kernel up to 16384
    positions, refused above; above 262144 positions refused for any shape."""
    say("[ops] gqa_decode_attn limits")
    run_gqa_case(hip, 64, 32, 2, 2000)
    h = hip.allocate(4 * 64 * 32)
    with pytest.raises(YuleGpuError, match="8 query heads"):
        hip.gqa_decode_attn(h, h, h, h, 32, 2, 64, 16385)
    with pytest.raises(YuleGpuError, match="262144"):
        hip.gqa_decode_attn(h, h, h, h, 32, 4, 64, 262145)
    with pytest.raises(YuleGpuError, match="131072"):   # per-head kernel's cache row width
        hip.gqa_decode_attn(h, h, h, h, 513, 513, 256, 10)
    hip.free(h)


def test_argmax_kats(hip):
    say("[ops] argmax")
    out = hip.allocate(4)
    for vals, want in ((K["argmax"]["values"], K["argmax"]["expect"]), ([1.0, 3.0, 3.0, 2.0], 2),
                       ([5.0] * 3000, 2999)):
        h = hip.upload(f32(vals))
        hip.argmax(h, len(vals), out)
        assert int(hip.download(out, 1, np.uint32)[0]) == want
        hip.free(h)
    v = synth.gauss(11, 32000)
    h = hip.upload(v)
    hip.argmax(h, 32000, out)
    assert int(hip.download(out, 1, np.uint32)[0]) == oracle.argmax(v)
    hip.free(h)
    # ties between infinities: argmax_ct's sign test keeps the first (inf - inf
    # is a negative NaN on x86), equal finite maxima go to the last; the oracle
    # runs the reference's scan
    inf = np.inf
    cases = [[inf, 1.0, inf], [-inf] * 5, [1.0, inf, 2.0, inf], [-inf, 3.0, 3.0], [2.0, -inf],
             [-inf, -inf, 0.5, -inf], [inf] * 4000]
    big = np.full(5000, -inf, np.float32)
    big[[17, 2500, 4999]] = inf
    cases.append(big)
    for vals in cases:
        a = f32(vals)
        want = oracle.argmax(a)
        h = hip.upload(a)
        hip.argmax(h, len(a), out)
        assert int(hip.download(out, 1, np.uint32)[0]) == want, vals
        hip.free(h)
    hip.free(out)


@pytest.mark.parametrize("pattern", [0, 1, 2])
@pytest.mark.parametrize("loads", [1, 2, 4, 8])
def test_read_probe_variants_read_every_word_once(hip, pattern, loads):
    """Each read-probe variant covers every word exactly once, at ragged
    sizes and grids that leave lanes, runs and chunks partly empty."""
    say(f"[ops] read_probe_variant pattern {pattern}, {loads} loads in flight")
    for n_bytes, n_wg in ((16, 1), (16, 64), (4096, 3), (1_000_016, 2048), (33_030_144, 1024)):
        data = np.random.default_rng(n_bytes + loads).integers(0, 2**32, n_bytes // 4, dtype=np.uint32)
        src, part = hip.upload(data), hip.allocate(4 * n_wg)
        hip.read_probe_variant(src, n_bytes, part, n_wg, pattern, loads)
        got = np.bitwise_xor.reduce(hip.download(part, n_wg, np.uint32))
        assert int(got) == int(np.bitwise_xor.reduce(data)), (n_bytes, n_wg)
        hip.free(src)
        hip.free(part)
    src, part = hip.allocate(64), hip.allocate(4)
    with pytest.raises(YuleGpuError):
        hip.read_probe_variant(src, 64, part, 1, 3, loads)    # no such pattern
    with pytest.raises(YuleGpuError):
        hip.read_probe_variant(src, 64, part, 1, pattern, 3)  # loads not a power of two up to 8
    hip.free(src)
    hip.free(part)


@pytest.mark.parametrize("n_bytes,n_wg", [(16, 1), (16, 64), (4096, 3), (1_000_016, 2048), (33_030_144, 2048)])
def test_read_probe_reads_every_word_once(hip, n_bytes, n_wg):
    """The roofline probe: the XOR of its per-workgroup partials equals the
    XOR of every 32-bit word of the range (each word read exactly once)."""
    say(f"[ops] read_probe {n_bytes} B over {n_wg} workgroups")
    rng = np.random.default_rng(n_bytes)
    data = rng.integers(0, 2**32, n_bytes // 4, dtype=np.uint32)
    src, part = hip.upload(data), hip.allocate(4 * n_wg)
    hip.read_probe(src, n_bytes, part, n_wg)
    got = np.bitwise_xor.reduce(hip.download(part, n_wg, np.uint32))
    assert int(got) == int(np.bitwise_xor.reduce(data))
    with pytest.raises(YuleGpuError):
        hip.read_probe(src, n_bytes + 16, part, n_wg)          # past the buffer
    with pytest.raises(YuleGpuError):
        hip.read_probe(src, n_bytes - 4 if n_bytes > 16 else 8, part, n_wg)   # not a multiple of 16
    with pytest.raises(YuleGpuError):
        hip.read_probe(src, n_bytes, part, n_wg + 1)           # partials too small
    hip.free(src)
    hip.free(part)


# positions around the 16-position and 1024-thread steps, head sizes around the
# 16-dim slices, offsets and strides that are and are not multiples of 4
@pytest.mark.parametrize("hd, seq, n_kv, shift", [(64, 1, 4, 0), (64, 777, 4, 0), (128, 1024, 2, 0), (80, 257, 3, 0),
                                                  (20, 65, 2, 0), (7, 63, 3, 0), (64, 1025, 2, 1), (66, 300, 1, 0)])
def test_attn_score_value_shapes(hip, hd, seq, n_kv, shift):
    say(f"[ops] attn_score / attn_value hd={hd} seq={seq} kv={n_kv} shift={shift}")
    kvs = n_kv * hd + shift
    q, kc, vc = synth.gauss(31, 2 * hd), synth.gauss(32, (seq, kvs)), synth.gauss(33, (seq, kvs))
    off = (n_kv - 1) * hd + shift
    hq, hk, hv, hs, ho = hip.upload(q), hip.upload(kc), hip.upload(vc), hip.allocate(4 * seq), hip.allocate(4 * (hd + 3))
    hip.attn_score(hq, hk, hs, hd, seq, hd, off, kvs)
    s = hip.download(hs, seq)
    q64, k64, v64 = q[hd:].astype(np.float64), kc[:, off:off + hd].astype(np.float64), vc[:, off:off + hd].astype(np.float64)
    # f32 sums of n terms: error at most n * 2^-24 of the sum of magnitudes
    assert np.all(np.abs(s - k64 @ q64 / math.sqrt(hd)) <= (hd + 4) * 2.0 ** -24 * (np.abs(k64) @ np.abs(q64)) / math.sqrt(hd))
    hip.softmax(hs, hs, seq)
    p = hip.download(hs, seq)
    e = np.exp(s.astype(np.float64) - s.max())
    # exp of a rounded difference, relative: |difference| * 2^-24 plus expf's 2 ulp, the sum's and the product's rounding
    assert close(p / (e / e.sum()), 1.0, (np.ptp(s) + seq / 256 + 16) * 2.0 ** -23)
    hip.attn_value(hs, hv, ho, hd, seq, off, kvs, 3)
    p64 = p.astype(np.float64)
    assert np.all(np.abs(hip.download(ho, hd + 3)[3:] - p64 @ v64) <= (seq + 4) * 2.0 ** -24 * (p64 @ np.abs(v64)))
    for b in (hq, hk, hv, hs, ho):
        hip.free(b)


@pytest.mark.parametrize("n", [1, 1024, 1025, 8192, 8193])
def test_softmax_sizes(hip, n):
    say(f"[ops] softmax n={n}")
    x = synth.gauss(34, n, 3.0)
    hx = hip.upload(x)
    hip.softmax(hx, hx, n)
    e = np.exp(x.astype(np.float64) - x.max())
    assert close(hip.download(hx, n) / (e / e.sum()), 1.0, (np.ptp(x) + n / 256 + 16) * 2.0 ** -23)
    hip.free(hx)


@pytest.mark.parametrize("n", [8192, 8193, 8195, 10240, 32001, 128256, 1 << 20])
def test_argmax_many_workgroups(hip, n):
    say(f"[ops] argmax n={n}")
    v = synth.gauss(35, n)
    hv, out = hip.allocate(4 * n), hip.allocate(4)
    last = v.copy()
    last[-1] = last[1] = 9.0            # equal maxima: the last one
    inf = v.copy()
    inf[n // 2] = inf[n - 2] = np.inf   # equal infinities: the first one
    for a in (v, last, inf, np.full(n, -np.inf, np.float32), np.full(n, -1.0, np.float32), v):
        hip.copy_to_device(a, hv)
        hip.argmax(hv, n, out)
        assert int(hip.download(out, 1, np.uint32)[0]) == oracle.argmax(a)
    hip.free(hv)
    hip.free(out)
