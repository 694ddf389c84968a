// attn_tile.h — attention of 16 queries against sub-tiles of 16 keys on the f32
// matrix instructions, one wave (prefill.hip: 16 rows of a head; ops.hip: the
// query heads of one KV head).
//
// Scores are formed transposed, S^T = K Q^T (16x16x4 f32 MFMA: operand A row
// and operand B column = lane % 16, k = lane / 16; result column = lane % 16,
// row = 4 (lane / 16) + r), so a lane holds the scores of one query (lane %
// 16) for keys 4 (lane / 16) + r: the softmax reduces in the lane and across
// two lane swaps, and result register r is already the B operand of O^T =
// V^T P^T, whose k index lane / 16 stands for key 4 (lane / 16) + r.  Row i of
// V^T's tile (G, t) is dim 64 G + VW i + t, so that one load of VW floats
// of a V row is the A operand of VW tiles and a lane's outputs are
// consecutive.  Everything stays in f32: no operand is split or rounded.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace yule {

typedef float f4v __attribute__((ext_vector_type(4)));

template <uint32_t HD>
struct AttnTile {
    static constexpr uint32_t NS = HD / 16;              // 16-dim steps of a K row
    static constexpr uint32_t VW = HD >= 64 ? 4 : 2;     // V floats per lane and key
    static constexpr uint32_t NG = HD / (16 * VW);       // such groups per row
    float4 q[NS];       // dims 16 s + 4 g + e of query lane % 16
    f4v o[NG][VW];      // O^T, unnormalised
    float m, l;         // running maximum (of the query), this lane's share of the sum

    __device__ __forceinline__ void init(const float *qrow, uint32_t g) {
#pragma unroll
        for (uint32_t s = 0; s < NS; s++) q[s] = *reinterpret_cast<const float4 *>(qrow + 16 * s + 4 * g);
#pragma unroll
        for (uint32_t G = 0; G < NG; G++)
#pragma unroll
            for (uint32_t t = 0; t < VW; t++) o[G][t] = f4v{0, 0, 0, 0};
        m = -INFINITY;
        l = 0.f;
    }
    // scores of one 16-key sub-tile += K . q over step s
    __device__ __forceinline__ void score(f4v &sc, const float4 &k, uint32_t s) const {
        sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k.x, q[s].x, sc, 0, 0, 0);
        sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k.y, q[s].y, sc, 0, 0, 0);
        sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k.z, q[s].z, sc, 0, 0, 0);
        sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k.w, q[s].w, sc, 0, 0, 0);
    }
    // a sub-tile's raw scores into probabilities (against the new running
    // maximum), with the running sum and outputs rescaled where the maximum
    // moved; key0 + 4 g + r is the key of sc[r], keys past qpos are masked
    // (only looked at with `diagonal`).  Probabilities are 2^(sc c - m), c =
    // log2(e) / sqrt(HD), m the maximum of sc c: the product and the difference
    // round once, in the fused multiply-add.
    __device__ __forceinline__ void softmax(f4v &sc, uint32_t key0, uint32_t g, uint32_t qpos, bool diagonal) {
        constexpr float c = (float)(1.44269504088896340736 / (HD == 32    ? 5.65685424949238019521
                                                              : HD == 64  ? 8.0
                                                              : HD == 128 ? 11.3137084989847603904
                                                                          : 16.0));
        if (diagonal) {
#pragma unroll
            for (uint32_t r = 0; r < 4; r++)
                if (key0 + 4 * g + r > qpos) sc[r] = -INFINITY;
        }
        float cm = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
        cm = fmaxf(cm, __shfl_xor(cm, 16, 64));
        cm = fmaxf(cm, __shfl_xor(cm, 32, 64)) * c;
        if (__ballot(cm > m)) {   // some query's maximum moved
            const float mn = fmaxf(m, cm);
            // (m = -inf: nothing was added yet, and the factor multiplies zeros)
            const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (uint32_t G = 0; G < NG; G++)
#pragma unroll
                for (uint32_t t = 0; t < VW; t++) o[G][t] *= alpha;
        }
        // (sub-tiles wholly past a query leave its maximum at -inf: nothing is added)
        const float mb = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
            sc[r] = __builtin_amdgcn_exp2f(fmaf(sc[r], c, -mb));
            l += sc[r];
        }
    }
    // outputs += p x V of keys 4 g + r: v = VW floats of that key's row, group G
    __device__ __forceinline__ void value(float p, const float *v, uint32_t G) {
#pragma unroll
        for (uint32_t t = 0; t < VW; t++) o[G][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t], p, o[G][t], 0, 0, 0);
    }
    // this lane's outputs, by (G, r): dims 16 VW G + VW (4 g + r) + 0..VW-1
    __device__ __forceinline__ void store(float *row, uint32_t g) const {
#pragma unroll
        for (uint32_t G = 0; G < NG; G++)
#pragma unroll
            for (uint32_t r = 0; r < 4; r++)
#pragma unroll
                for (uint32_t t = 0; t < VW; t++) row[16 * VW * G + VW * (4 * g + r) + t] = o[G][t][r];
    }
};

}  // namespace yule
