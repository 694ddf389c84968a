// prefill.hip — the runner's batched prompt pass: the operations of a decode
// step applied to P prompt rows at once, so that each projection runs as one
// matrix-core GEMM (gemm.hip, f32 X) instead of P matvecs.  Yule prefills token
// by token (yule-infer/src/model_runner.rs:1075-1081); every row here computes
// exactly what that step computes for its token, to f32 rounding, and writes
// the same KV-cache rows:
//   embedding rows -> per layer [RMSNorm rows] [Q, K, V GEMMs] [RoPE + cache
//   rows] [causal attention] [O GEMM] [residual] [RMSNorm rows] [gate, up
//   GEMMs] [SwiGLU] [down GEMM] [residual].
#include "attn_tile.h"
#include "blocks.h"
#include "internal.h"
#include "qmv_common.h"

namespace yule {

// ---- embedding rows: out[p] = dequantized row tokens[p] of the table
// (the token lookup of model_runner.rs:543-560, gpu_runner.rs:309-343)
__global__ void embed_rows_kernel(uint32_t dtype, uint32_t bs, uint32_t bb, const uint8_t *__restrict__ table,
                                  const uint32_t *__restrict__ tokens, uint32_t vocab, float *__restrict__ out,
                                  uint32_t dim) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, p = blockIdx.y;
    if (i >= dim) return;
    uint32_t t = tokens[p];
    t = t < vocab ? t : vocab - 1;   // host-checked tokens are in range; the clamp keeps reads in the table
    const uint8_t *row = table + (size_t)t * (dim / bs) * bb;
    out[(size_t)p * dim + i] = dequant_one(dtype, row + (i / bs) * bb, i % bs);
}

int launch_embed_rows_batch(hipStream_t s, uint32_t dtype, const uint8_t *table, const uint32_t *tokens,
                            uint32_t vocab, float *out, uint32_t dim, uint32_t n) {
    uint32_t bs, bb;
    if (!quant_geometry(dtype, &bs, &bb)) return set_error(YULE_ERR_UNSUPPORTED, "embedding: unsupported dtype");
    hipLaunchKernelGGL(embed_rows_kernel, dim3((dim + 255) / 256, n), dim3(256), 0, s, dtype, bs, bb, table, tokens,
                       vocab, out, dim);
    return check_launch("embedding rows");
}

// ---- RoPE of row p's q (in place) and k with the table row of position
// pos0 + p, and k, v into cache row pos0 + p (model_runner.rs:277-293,
// 654-669; the same arithmetic as the decode step's Q/K/V epilogue).  Rows
// of q are ldq floats apart, rows of k and v ldkv (separate buffers: qd and
// kvd; one [q | k | v] buffer: qd + 2 kvd for all three).
__global__ void rope_rows_kernel(float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
                                 float *__restrict__ kc, float *__restrict__ vc, const float *__restrict__ cos_t,
                                 const float *__restrict__ sin_t, uint32_t pos0, uint32_t qd, uint32_t kvd,
                                 uint32_t hd, uint32_t ldq, uint32_t ldkv) {
    const uint32_t p = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x, half = hd / 2;
    const uint32_t pos = pos0 + p, nqp = qd / 2, nkp = kvd / 2;
    if (j < nqp) {   // rotation pair j of q
        const uint32_t i = j % half;
        const float c = cos_t[(size_t)pos * half + i], sn = sin_t[(size_t)pos * half + i];
        float *qr = q + (size_t)p * ldq + 2 * j;
        const float x0 = qr[0], x1 = qr[1];
        qr[0] = x0 * c - x1 * sn;
        qr[1] = x0 * sn + x1 * c;
    } else if (j < nqp + nkp) {   // pair j - nqp of k, and the matching v values
        const uint32_t jk = j - nqp, i = jk % half;
        const float c = cos_t[(size_t)pos * half + i], sn = sin_t[(size_t)pos * half + i];
        const float *kr = k + (size_t)p * ldkv + 2 * jk;
        const float x0 = kr[0], x1 = kr[1];
        float *krow = kc + (size_t)pos * kvd + 2 * jk, *vrow = vc + (size_t)pos * kvd + 2 * jk;
        krow[0] = x0 * c - x1 * sn;
        krow[1] = x0 * sn + x1 * c;
        const float *vr = v + (size_t)p * ldkv + 2 * jk;
        vrow[0] = vr[0];
        vrow[1] = vr[1];
    }
}

int launch_rope_rows(hipStream_t s, float *q, const float *k, const float *v, float *kc, float *vc, const float *cos_t,
                     const float *sin_t, uint32_t pos0, uint32_t n, uint32_t qd, uint32_t kvd, uint32_t hd, uint32_t ldq,
                     uint32_t ldkv) {
    const uint32_t pairs = (qd + kvd) / 2;
    hipLaunchKernelGGL(rope_rows_kernel, dim3((pairs + 255) / 256, n), dim3(256), 0, s, q, k, v, kc, vc, cos_t, sin_t,
                       pos0, qd, kvd, hd, ldq, ldkv);
    return check_launch("rope rows");
}

// ---- causal GQA attention of prompt rows p (positions pos0 + p) over cache
// rows 0..pos0 + p (model_runner.rs:679-758) on the f32 matrix instructions:
// a wave owns a unit of 16 query rows of one head and walks the keys in
// sub-tiles of 16 with an online softmax (attn_tile.h).
//
// Half bound by the f32 matrix rate for long prompts: 1531 rows of 32 heads of
// 64 dims need 9.8 GFLOP of it, 62 us at the nominal 157 TFLOP/s; in a prompt
// pass the launch takes 138 us (127 at best) with the matrix units 47% busy, the
// softmax between two products in series with them.
//
// A workgroup of NW waves owns one unit (head, query tile; the last, longest
// tiles first).  Its waves take the keys' sub-tiles in turn, with operands
// straight from the cache and one sub-tile in flight ahead, and their (m, l,
// O) meet in LDS at the end.  Measured against it:
// K and V tiles of 64 keys staged through LDS for four units (184 us against
// 118 at 1531 rows of 32 heads of 64 dims: two barriers a tile and the causal
// imbalance of the units), and two units per wave sharing the operand
// registers (132 us: the cache reads are not the bound, the registers cost
// waves).  One workgroup per row with vector FMAs took 653 us.
// A key past a query's position has weight 0 there, but its V row is still
// multiplied: an infinite or NaN V row makes the up to 15 rows before it in
// its tile NaN too, besides those from it on.  Nothing that can be read sees
// the difference: only the last row's logits leave the pass, and that row, as
// every later position, has the non-finite V row among its own keys.
template <uint32_t HD, uint32_t NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(HD <= 128 ? 2 : 1))) void attn_prefill_kernel(
    const float *__restrict__ q, const float *__restrict__ kc, const float *__restrict__ vc, float *__restrict__ out,
    uint32_t pos0, uint32_t n, uint32_t qd, uint32_t ldq, uint32_t group, uint32_t n_kv) {
    using T = AttnTile<HD>;
    constexpr uint32_t OS = HD + 4;
    __shared__ __align__(16) float os[NW * 16 * OS];
    __shared__ float ms[NW][16], ls[NW][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, c = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t h = blockIdx.x, kvh = h / group, q0 = 16 * (gridDim.y - 1u - blockIdx.y), rows = pos0 + n;
    const uint32_t p = q0 + c, qpos = pos0 + p, keys = pos0 + (q0 + 16 < n ? q0 + 16 : n);
    T st;
    st.init(q + (size_t)(p < n ? p : n - 1u) * ldq + (size_t)h * HD, g);
    const size_t kvs = (size_t)n_kv * HD;
    const float *kb = kc + (size_t)kvh * HD, *vb = vc + (size_t)kvh * HD;
    float4 kr[T::NS];
    float vr[4][T::NG][T::VW];
    auto row = [&](uint32_t k) { return (size_t)(k < rows ? k : rows - 1u) * kvs; };   // rows past the end are masked
    auto load_k = [&](uint32_t k0) {
#pragma unroll
        for (uint32_t s = 0; s < T::NS; s++)
            kr[s] = *reinterpret_cast<const float4 *>(kb + row(k0 + c) + 16 * s + 4 * g);
    };
    auto load_v = [&](uint32_t k0) {
#pragma unroll
        for (uint32_t r = 0; r < 4; r++)
#pragma unroll
            for (uint32_t G = 0; G < T::NG; G++) {
                const float *vp = vb + row(k0 + 4 * g + r) + 16 * T::VW * G + T::VW * c;
#pragma unroll
                for (uint32_t t = 0; t < T::VW; t++) vr[r][G][t] = vp[t];
            }
    };
    uint32_t k0 = 16 * wave;
    if (k0 < keys) {
        load_k(k0);
        load_v(k0);
    }
    for (; k0 < keys; k0 += 16 * NW) {
        f4v sc[2] = {f4v{0, 0, 0, 0}, f4v{0, 0, 0, 0}};
#pragma unroll
        for (uint32_t s = 0; s < T::NS; s++) st.score(sc[s & 1u], kr[s], s);
        const bool more = k0 + 16 * NW < keys;
        if (more) load_k(k0 + 16 * NW);
        sc[0] += sc[1];
        st.softmax(sc[0], k0, g, qpos, k0 + 16 > pos0 + q0 + 1);
#pragma unroll
        for (uint32_t r = 0; r < 4; r++)
#pragma unroll
            for (uint32_t G = 0; G < T::NG; G++) st.value(sc[0][r], vr[r][G], G);
        if (more) load_v(k0 + 16 * NW);
    }
    float l = st.l;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    st.store(os + (wave * 16 + c) * OS, g);
    if (g == 0) {
        ms[wave][c] = st.m;
        ls[wave][c] = l;
    }
    __syncthreads();
    // out = sum_w 2^(m_w - M) O_w / sum_w 2^(m_w - M) l_w (wave 0 always has key 0: M is its queries' maximum)
    for (uint32_t i = tid; i < 16 * (HD / 4); i += 64 * NW) {
        const uint32_t qi = i / (HD / 4), d = 4 * (i % (HD / 4));
        if (q0 + qi >= n) continue;
        float M = ms[0][qi];
#pragma unroll
        for (uint32_t w = 1; w < NW; w++) M = fmaxf(M, ms[w][qi]);
        float L = 0.f;
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (uint32_t w = 0; w < NW; w++) {
            const float f = __builtin_amdgcn_exp2f(ms[w][qi] - M);
            const float4 o = *reinterpret_cast<const float4 *>(os + (w * 16 + qi) * OS + d);
            L += f * ls[w][qi];
            a.x += f * o.x; a.y += f * o.y; a.z += f * o.z; a.w += f * o.w;
        }
        const float inv = 1.0f / L;
        *reinterpret_cast<float4 *>(out + (size_t)(q0 + qi) * qd + (size_t)h * HD + d) =
            make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
    }
}

bool attn_prefill_supported(uint32_t hd) { return hd == 32 || hd == 64 || hd == 128 || hd == 256; }

template <uint32_t HD, uint32_t NW>
static void launch_attn_prefill_nw(hipStream_t s, const float *q, const float *kc, const float *vc, float *out,
                                   uint32_t pos0, uint32_t n, uint32_t n_heads, uint32_t n_kv, uint32_t ldq) {
    hipLaunchKernelGGL((attn_prefill_kernel<HD, NW>), dim3(n_heads, (n + 15) / 16), dim3(64 * NW), 0, s, q, kc, vc, out,
                       pos0, n, n_heads * HD, ldq, n_heads / n_kv, n_kv);
}

template <uint32_t HD>
static void launch_attn_prefill_hd(hipStream_t s, const float *q, const float *kc, const float *vc, float *out,
                                   uint32_t pos0, uint32_t n, uint32_t n_heads, uint32_t n_kv, uint32_t ldq) {
    // Eight waves a workgroup for few units over many keys (64 dims, 64 rows
    // after 1000: 17.4 us against 19.2 with four), four otherwise (1531 rows
    // 112.6 against 115.0; 128 dims, 1531 rows: 224 against 248).
    if constexpr (HD <= 64) {
        if (n_heads * ((n + 15) / 16) <= 2u * (uint32_t)device_cus() && pos0 + n > 256)
            return launch_attn_prefill_nw<HD, 8>(s, q, kc, vc, out, pos0, n, n_heads, n_kv, ldq);
    }
    launch_attn_prefill_nw<HD, 4>(s, q, kc, vc, out, pos0, n, n_heads, n_kv, ldq);
}

int launch_attn_prefill(hipStream_t s, const float *q, const float *kc, const float *vc, float *out, uint32_t pos0,
                        uint32_t n, uint32_t n_heads, uint32_t n_kv, uint32_t hd, uint32_t ldq) {
    switch (hd) {
    case 32: launch_attn_prefill_hd<32>(s, q, kc, vc, out, pos0, n, n_heads, n_kv, ldq); break;
    case 64: launch_attn_prefill_hd<64>(s, q, kc, vc, out, pos0, n, n_heads, n_kv, ldq); break;
    case 128: launch_attn_prefill_hd<128>(s, q, kc, vc, out, pos0, n, n_heads, n_kv, ldq); break;
    case 256: launch_attn_prefill_hd<256>(s, q, kc, vc, out, pos0, n, n_heads, n_kv, ldq); break;
    default: return set_error(YULE_ERR_UNSUPPORTED, "prefill attention: head size");
    }
    return check_launch("prefill attention");
}

}  // namespace yule
