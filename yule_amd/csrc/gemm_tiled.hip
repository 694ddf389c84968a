// gemm_tiled.hip — prefill GEMM for many rows of X: the weights are expanded
// once per call into exact f16 integers, laid out as matrix-core operand tiles
// (gemm_tiled.h), and the product then runs as a plain f16 GEMM whose operands
// go from memory straight into LDS.  gemm.hip's kernels, which expand a weight
// tile in every workgroup that multiplies it, serve fewer rows.
//
// Exactness as in gemm.hip: the operand is the integer part of a weight, every
// scale is applied in f32.
//  * f32 X: Q4_K, Q5_K: q (<= 31), d * sc per 32 weights; the min term is an extra k
//    range (sums of x against -(dmin * mn), both split hi + lo).
//  * Q8_0, Q4_0, Q8_K: q, q - 8 and q, d per 32 weights.
//  * Q6_K with f32 X: q - 32, d * sc per 16 weights: one k-step of the MFMA.
//  * bf16 X, Q6_K only: sc * (q - 32), rounded to even above 2048 as in gemm.hip, d
//    per super-block (the finer scales would leave one operand bound by their
//    FMAs; the other formats' kernels in gemm.hip are as fast).
// Each scale's products are summed from zero and added times the scale; with d per
// super-block the accumulators are kept in units of the current super-block's
// d (acc *= unit / d_new at its start).  f32 X is two operands (hi, lo)
// against the same weight tile in the same pass.  Error against 64 bits
// (2-norm, f32 X): Q4_K 1000 x 4096 x 4096 1.7e-6 in gemm.hip, 4.0e-7 here
// (no rescaled accumulators); Q6_K 300 x 2048 x 5632 1.6e-7, 1.3e-7.
#include <type_traits>

#include "gemm_tiled.h"
#include "qmv_common.h"

namespace yule {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t pk_mul(uint32_t pair, h2_t s) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, pair) * s);
}
// two bytes (bits 0-7, 16-23, upper bits clear) as f16 u - bias, exact
__device__ __forceinline__ uint32_t pair_f16(uint32_t v, float bias) {
    const _Float16 b = (_Float16)(1024.0f + bias);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, v | 0x64006400u) - h2_t{b, b});
}
constexpr uint32_t kTiledBm = 128, kTiledBn = 256;   // workgroup tile

struct Mats {
    const uint8_t *w[3];
    uint32_t s1, s2;
};

template <uint32_t DT>
constexpr uint32_t block_bytes() {
    return DT == YULE_DTYPE_Q4_K ? 144 : DT == YULE_DTYPE_Q5_K ? 176 : DT == YULE_DTYPE_Q6_K ? 210
         : DT == YULE_DTYPE_Q8_K ? 292 : DT == YULE_DTYPE_Q8_0 ? 34 : 18;
}

// ---------------------------------------------------------------- weight tiles
// One workgroup per 32 weight rows (of the pass's rows r_lo..r_lo + n) and
// super-block, super-blocks fastest (consecutive in memory).  The rows' raw
// bytes are loaded row by row into LDS (read straight by the threads that
// expand them, each lane on a row of its own, the loads took the address
// unit 64 cycles apiece and three quarters of the launch); then thread t
// expands row t % 32, weights 32 (t / 32).. + 31, and 32 lanes store 512
// consecutive bytes.
// scale: [k / GRAN][np] f32: d * sc or d, or (GRAN 256) the rescale factor
// unit / d_new of the super-block and, in rows bpr.., the units themselves.
template <uint32_t DT, uint32_t GRAN>
__global__ __launch_bounds__(256) void tile_weights_kernel(const Mats mt, uint32_t r_lo, uint32_t n, uint32_t np,
                                                           uint32_t bpr, uint32_t ext, uint8_t *__restrict__ wt,
                                                           uint8_t *__restrict__ we, float *__restrict__ scale) {
    constexpr uint32_t BB = block_bytes<DT>();
    constexpr bool B32 = DT == YULE_DTYPE_Q8_0 || DT == YULE_DTYPE_Q4_0, Q5 = DT == YULE_DTYPE_Q5_K;
    constexpr uint32_t SBB = B32 ? 8 * BB : BB;          // bytes of a row's super-block
    constexpr bool ODD = SBB % 4 != 0;                   // then a row may start 2 bytes into a dword
    constexpr uint32_t W = (SBB + (ODD ? 2 : 0) + 3) / 4, WS = W | 1u;   // its dword window (at most 4 bytes past it)
    __shared__ uint32_t raw[32 * WS];
    const uint32_t tid = threadIdx.x, r = tid & 31u, part = tid >> 5, sb = blockIdx.x, rb = blockIdx.y;
    const uint32_t rr = 32 * rb + r;
    auto row_at = [&](uint32_t i) {   // super-block sb of the tile's row i (rows past the end repeat the last one)
        const uint32_t row = r_lo + (32 * rb + i < n ? 32 * rb + i : n - 1u);
        return (row >= mt.s2 ? mt.w[2] : row >= mt.s1 ? mt.w[1] : mt.w[0]) +
               ((size_t)(row - (row >= mt.s2 ? mt.s2 : row >= mt.s1 ? mt.s1 : 0u)) * bpr + sb) * SBB;
    };
#pragma unroll
    for (uint32_t i = 0; i < (32 * W + 255) / 256; i++) {
        const uint32_t at = tid + 256 * i, row = at / W, w = at % W;
        if (32 * W % 256 == 0 || row < 32) {
            const uint8_t *p = row_at(row);
            raw[row * WS + w] = reinterpret_cast<const uint32_t *>(p - (ODD ? reinterpret_cast<uintptr_t>(p) & 2u : 0u))[w];
        }
    }
    const uint8_t *own = row_at(r);
    const uint32_t mis = ODD ? (uint32_t)(reinterpret_cast<uintptr_t>(own) & 2u) : 0u;
    // GRAN 256 (Q6_K): the last non-zero d before this super-block's
    float prev = 1.f;
    if (GRAN == 256 && part == 0 && sb) {
        uint32_t back = 1;
        do prev = f16_bits(*reinterpret_cast<const uint16_t *>(own - (size_t)back * SBB + 208));
        while (prev == 0.f && ++back <= sb);
        if (prev == 0.f) prev = 1.f;
    }
    __syncthreads();
    const uint32_t *lr = raw + r * WS;
    auto dword = [&](uint32_t o) {   // bytes o..o + 3 of the super-block (o even)
        if constexpr (!ODD && !B32) return lr[o / 4];
        const uint32_t a = o + mis;
        const uint32_t lo = lr[a / 4];
        return (a & 2u) ? (lr[a / 4 + 1 < W ? a / 4 + 1 : a / 4] << 16) | (lo >> 16) : lo;
    };
    uint32_t o[16];   // 32 f16 weights in the {0, 2, 1, 3} order
    if constexpr (DT == YULE_DTYPE_Q4_K || Q5) {
        const uint32_t h0 = dword(0), h1 = dword(4), h2 = dword(8), h3 = dword(12);
        const uint32_t j = part >> 1, hi = part & 1u;
        // get_scale_min_k4 (dequant.rs:176-190), by shifts: a byte indexed by
        // the thread's sub-block would live in scratch memory
        const uint32_t sh = 8u * (part & 3u);
        const uint32_t sc6 = part < 4 ? (h1 >> sh) & 63u : ((h3 >> sh) & 15u) | (((h1 >> (sh + 6)) & 3u) << 4);
        scale[(size_t)(8 * sb + part) * np + rr] = f16_bits(h0) * (float)sc6;
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            uint32_t u = (dword((Q5 ? 48u : 16u) + 32u * j + 4 * i) >> (4u * hi)) & 0x0F0F0F0Fu;
            if constexpr (Q5) u |= ((dword(16u + 4 * i) >> part) & 0x01010101u) << 4;
            o[2 * i] = pair_f16(u & 0x00FF00FFu, 0.f);
            o[2 * i + 1] = pair_f16((u >> 8) & 0x00FF00FFu, 0.f);
        }
        // the min term's columns of this super-block: -(dmin * mn) hi, lo, hi
        if (part < 3) {
            const float dmin = f16_bits(h0 >> 16);
            half8 m;
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const uint32_t t = 8u * (s & 3);
                const uint32_t mn = s < 4 ? (h2 >> t) & 63u : ((h3 >> (t + 4)) & 15u) | (((h2 >> (t + 6)) & 3u) << 4);
                const float x = -(dmin * (float)mn);
                const _Float16 xh = (_Float16)x;
                m[s] = part == 1 ? (_Float16)(x - (float)xh) : xh;
            }
            *reinterpret_cast<half8 *>(we + tile_unit(rr, part * bpr + sb, tile_pitch(ext))) = m;
        } else if (part == 3 && sb == 0) {
            for (uint32_t c = 3 * bpr; c < ext / 8; c++) *reinterpret_cast<half8 *>(we + tile_unit(rr, c, tile_pitch(ext))) = half8{};
        }
    } else if constexpr (DT == YULE_DTYPE_Q8_K) {
        scale[(size_t)(8 * sb + part) * np + rr] = __builtin_bit_cast(float, dword(0));
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            const uint32_t u = dword(4 + 32 * part + 4 * i) ^ 0x80808080u;
            o[2 * i] = pair_f16(u & 0x00FF00FFu, 128.f);
            o[2 * i + 1] = pair_f16((u >> 8) & 0x00FF00FFu, 128.f);
        }
    } else if constexpr (DT == YULE_DTYPE_Q6_K) {
        // quarter g of half h: weights 128 h + 32 g + l (dequant.rs:340-372)
        const uint32_t h = part >> 2, g = part & 3u, sc = dword(192u + 8u * h + 2u * g);
        const int s0 = (int8_t)(sc & 0xFFu), s1 = (int8_t)((sc >> 8) & 0xFFu);
        const float d = f16_bits(dword(208));
        const bool dz = d == 0.f;   // (GRAN 256: the unit stays, the operand is zero)
        if constexpr (GRAN == 16) {
            scale[(size_t)(16 * sb + 2 * part) * np + rr] = d * (float)s0;
            scale[(size_t)(16 * sb + 2 * part + 1) * np + rr] = d * (float)s1;
        } else if (part == 0) {
            scale[(size_t)sb * np + rr] = dz ? 1.f : prev / d;
            scale[(size_t)(bpr + sb) * np + rr] = dz ? prev : d;
        }
        const _Float16 f0 = (_Float16)(float)(dz ? 0 : s0), f1 = (_Float16)(float)(dz ? 0 : s1);
        const h2_t S0 = {f0, f0}, S1 = {f1, f1};
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            const uint32_t ql = dword(64u * h + 32u * (g & 1u) + 4 * i), qh = dword(128u + 32u * h + 4 * i);
            const uint32_t u = ((ql >> (4u * (g >> 1))) & 0x0F0F0F0Fu) | (((qh >> (2u * g)) & 0x03030303u) << 4);
            const uint32_t e = pair_f16(u & 0x00FF00FFu, 32.f), f = pair_f16((u >> 8) & 0x00FF00FFu, 32.f);
            o[2 * i] = GRAN == 16 ? e : pk_mul(e, i < 4 ? S0 : S1);
            o[2 * i + 1] = GRAN == 16 ? f : pk_mul(f, i < 4 ? S0 : S1);
        }
    } else {
        const uint32_t b = part * BB;
        scale[(size_t)(8 * sb + part) * np + rr] = f16_bits(dword(b));
        if constexpr (DT == YULE_DTYPE_Q8_0) {
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {
                const uint32_t u = dword(b + 2 + 4 * i) ^ 0x80808080u;
                o[2 * i] = pair_f16(u & 0x00FF00FFu, 128.f);
                o[2 * i + 1] = pair_f16((u >> 8) & 0x00FF00FFu, 128.f);
            }
        } else {
            // weight 2j is the low nibble of quant byte j, 2j + 1 the high one (dequant.rs:77-86)
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t q = dword(b + 2 + 4 * i), lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
                o[4 * i] = pair_f16(__builtin_amdgcn_perm(0u, lo, 0x0C010C00u), 8.f);
                o[4 * i + 1] = pair_f16(__builtin_amdgcn_perm(0u, hi, 0x0C010C00u), 8.f);
                o[4 * i + 2] = pair_f16(__builtin_amdgcn_perm(0u, lo, 0x0C030C02u), 8.f);
                o[4 * i + 3] = pair_f16(__builtin_amdgcn_perm(0u, hi, 0x0C030C02u), 8.f);
            }
        }
    }
#pragma unroll
    for (uint32_t c = 0; c < 4; c++)
        *reinterpret_cast<uint4 *>(wt + tile_unit(rr, 32 * sb + 4 * part + c, tile_pitch(256 * bpr))) =
            make_uint4(o[4 * c], o[4 * c + 1], o[4 * c + 2], o[4 * c + 3]);
}

// ---------------------------------------------------------------- X tiles
// The pre-pass of gemm.hip (power-of-two row scale, f16 hi and lo, sub-block
// sums, RMSNorm or SwiGLU on the way in, a pending split-K reduction first)
// with tiles as output.  A workgroup takes R rows (four, one when that leaves
// the chip idle): the low lane bits the row, the others the 8-element chunk,
// so that a tile's stores are 16 R consecutive bytes; the workgroups of a
// 32-row tile are dealt to one XCD, whose cache then holds whole lines of it.
template <bool F32, uint32_t R>
__global__ __launch_bounds__(256) void x_tiles_kernel(const void *xin, const float *__restrict__ nw, uint32_t K,
                                                      float eps, uint32_t glu, uint32_t rows, uint32_t ext,
                                                      uint8_t *__restrict__ xh, uint8_t *__restrict__ xl,
                                                      uint8_t *__restrict__ xe, float *__restrict__ rowscale,
                                                      const float *__restrict__ part, uint32_t ks, uint32_t ny,
                                                      uint32_t accumulate) {
    constexpr uint32_t PT = 32 / R, CP = 256 / R;   // workgroups per 32-row tile, chunks per pass
    __shared__ float red[4][R], red2[4][R];
    const uint32_t bid = blockIdx.x, g = bid / (8 * PT) * (8 * PT);
    const uint32_t wg = g + 8 * PT <= gridDim.x ? g + PT * (bid % 8) + (bid - g) / 8 : bid;
    const uint32_t tid = threadIdx.x, rl = tid % R, m = R * wg + rl, mc = m < rows ? m : rows - 1u, nch = K / 8;
    auto load4 = [](const float *p, float *v) {
        const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    };
    // the pending reduction of eight columns of this row: partials z
    // ascending, then the row itself (the order of gemm_reduce_kernel); the
    // thread that writes them is the one that reads them again below
    auto reduce8 = [&](uint32_t col) {
        float *y = const_cast<float *>(static_cast<const float *>(xin)) + (size_t)mc * ny + col;
        const float *p = part + (size_t)mc * ny + col;
        const size_t st = (size_t)rows * ny;
        float a[8], b[8];
        load4(p, a);
        if (accumulate) load4(y, b);
        for (uint32_t z = 1; z < ks; z++) {
            float v[8];
            load4(p + z * st, v);
#pragma unroll
            for (int t = 0; t < 8; t++) a[t] += v[t];
        }
        if (accumulate) {
#pragma unroll
            for (int t = 0; t < 8; t++) a[t] = b[t] + a[t];
        }
        if (m < rows) {
            reinterpret_cast<float4 *>(y)[0] = make_float4(a[0], a[1], a[2], a[3]);
            reinterpret_cast<float4 *>(y)[1] = make_float4(a[4], a[5], a[6], a[7]);
        }
    };
    auto load8 = [&](uint32_t c, float *v) {
        if constexpr (F32) {
            const float *x = static_cast<const float *>(xin);
            if (glu) {   // gate * sigmoid(gate) * up of a [gate | up] row (model_runner.rs:967-972)
                float u[8];
                load4(x + (size_t)mc * 2 * K + 8 * c, v);
                load4(x + (size_t)mc * 2 * K + K + 8 * c, u);
#pragma unroll
                for (int t = 0; t < 8; t++) v[t] = v[t] * (1.0f / (1.0f + expf(-v[t]))) * u[t];
            } else {
                load4(x + (size_t)mc * K + 8 * c, v);
            }
        } else {
            const uint4 u = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(xin) + (size_t)mc * K + 8 * c);
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int t = 0; t < 4; t++) {
                v[2 * t] = __builtin_bit_cast(float, w[t] << 16);
                v[2 * t + 1] = __builtin_bit_cast(float, w[t] & 0xFFFF0000u);
            }
        }
    };
    float amax = 0.f, ss = 0.f;
#pragma unroll 4
    for (uint32_t c = tid / R; c < nch; c += CP) {
        if (part) {
            reduce8(8 * c);
            if (glu) reduce8(K + 8 * c);
        }
        float v[8];
        load8(c, v);
        if (nw) {
            float w[8];
            load4(nw + 8 * c, w);
#pragma unroll
            for (int t = 0; t < 8; t++) {
                ss += v[t] * v[t];
                amax = fmaxf(amax, fabsf(v[t] * w[t]));
            }
        } else {
#pragma unroll
            for (int t = 0; t < 8; t++) amax = fmaxf(amax, fabsf(v[t]));   // NaN is dropped here, kept below
        }
    }
#pragma unroll
    for (int off = 32; off >= (int)R; off >>= 1) {
        amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        ss += __shfl_xor(ss, off, 64);
    }
    if ((tid & 63u) < R) {
        red[tid >> 6][rl] = amax;
        red2[tid >> 6][rl] = ss;
    }
    __syncthreads();
    amax = fmaxf(fmaxf(red[0][rl], red[1][rl]), fmaxf(red[2][rl], red[3][rl]));
    const float inv = nw ? 1.0f / sqrtf(((red2[0][rl] + red2[1][rl]) + (red2[2][rl] + red2[3][rl])) / (float)K + eps) : 1.0f;
    amax *= inv;   // the normalised row's largest magnitude, to rounding (the scale only needs its exponent)
    int e = 0;
    (void)frexpf(amax, &e);
    const int es = 10 - e < 126 ? 10 - e : 126;   // rows below 2^-116 keep s = 2^126
    const bool scaled = amax > 0.f && amax <= 3.402823466e38f;
    const float sc = scaled ? ldexpf(1.0f, es) : 1.0f;
    const int perm[8] = {0, 2, 1, 3, 4, 6, 5, 7};
    const uint32_t bpr = K / 256;
    for (uint32_t c0 = 0; c0 < nch; c0 += CP) {   // uniform trip count: the sums below need every lane
        const uint32_t c = c0 + tid / R;
        const bool ok = c < nch && m < rows;
        float v[8];
        load8(c < nch ? c : 0u, v);
        if (nw) {
            float w[8];
            load4(nw + 8 * (c < nch ? c : 0u), w);
#pragma unroll
            for (int t = 0; t < 8; t++) v[t] = v[t] * inv * w[t];
        }
        uint32_t oh[4], ol[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const float a = v[perm[2 * t]] * sc, b = v[perm[2 * t + 1]] * sc;
            const h2_t h = {(_Float16)a, (_Float16)b};
            oh[t] = __builtin_bit_cast(uint32_t, h);
            if constexpr (F32) {
                const h2_t l = {(_Float16)(a - (float)h.x), (_Float16)(b - (float)h.y)};
                ol[t] = __builtin_bit_cast(uint32_t, l);
            }
        }
        float s = 0.f;
#pragma unroll
        for (int t = 0; t < 8; t++) s += v[t] * sc;
        // the four chunks of a 32-element sub-block are R lanes apart
        s += __shfl_xor(s, (int)R, 64);
        s += __shfl_xor(s, 2 * (int)R, 64);
        if (ok) {
            const size_t o = tile_unit(m, c, tile_pitch(K));
            *reinterpret_cast<uint4 *>(xh + o) = make_uint4(oh[0], oh[1], oh[2], oh[3]);
            if constexpr (F32) *reinterpret_cast<uint4 *>(xl + o) = make_uint4(ol[0], ol[1], ol[2], ol[3]);
            if (ext && (c & 3u) == 0) {
                // sub-block c / 4: half c / 4 % 8 of its super-block's unit; sums hi, hi, lo
                const uint32_t sb = c / 32, at = 2 * ((c / 4) & 7u);
                const _Float16 h = (_Float16)s;
                *reinterpret_cast<_Float16 *>(xe + tile_unit(m, sb, tile_pitch(ext)) + at) = h;
                *reinterpret_cast<_Float16 *>(xe + tile_unit(m, bpr + sb, tile_pitch(ext)) + at) = h;
                *reinterpret_cast<_Float16 *>(xe + tile_unit(m, 2 * bpr + sb, tile_pitch(ext)) + at) = (_Float16)(s - (float)h);
            }
        }
    }
    if (m < rows) {
        for (uint32_t c = 3 * bpr + tid / R; c < ext / 8; c += CP)   // the extra range's padding
            *reinterpret_cast<uint4 *>(xe + tile_unit(m, c, tile_pitch(ext))) = make_uint4(0, 0, 0, 0);
        if (tid < R) rowscale[m] = scaled ? ldexpf(1.0f, -es) : 1.0f;
    }
}

// ---------------------------------------------------------------- product
// Four waves, two along m and two along n, each a BM/2 x BN/2 sub-tile of
// 32 x 32 x 16 MFMAs (operand A = X rows, B = weight rows: a result column
// lane % 32 is one weight row, so a scale is one value per lane).  k advances
// in stages of 32: the tiles' blocks (1 KB each, contiguous in memory and in
// LDS, so neither the copy nor the operand reads conflict) of stage s + 1 are
// copied into one LDS buffer while stage s is multiplied out of the other.
template <uint32_t SW, uint32_t GRAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tiled_kernel(
    const uint8_t *__restrict__ xh, const uint8_t *__restrict__ wt, const uint8_t *__restrict__ xl,
    const float *__restrict__ scale, const uint8_t *__restrict__ xe, const uint8_t *__restrict__ we, uint32_t M,
    uint32_t N, uint32_t bpr, uint32_t ext, uint32_t np, uint32_t ks_tail, float *__restrict__ y, uint32_t ldy,
    const float *__restrict__ rowscale, uint32_t accumulate, float *__restrict__ tail_part) {
    constexpr uint32_t BM = kTiledBm, BN = kTiledBn, NBUF = SW == 1 ? 3 : 2;
    constexpr uint32_t MT = BM / 64, NT = BN / 64;                 // MFMA tiles per wave
    constexpr uint32_t AB = BM / 32 * 2, BBK = BN / 32 * 2;        // 1 KB blocks per stage: one X operand, the weights
    constexpr uint32_t SCW = tile_scale_rows(GRAN);               // 1 KB (256 floats) each
    constexpr uint32_t NB = SW * AB + BBK;
    constexpr uint32_t BUF = (NB + SCW) * 1024;
    __shared__ __align__(1024) uint8_t lds[NBUF * BUF];
    static_assert(NB % 4 == 0, "every wave copies the same number of blocks");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 1, wn = wave & 1u;
    const uint32_t nt = (N + BN - 1) / BN, tiles = nt * ((M + BM - 1) / BM);
    // ks_tail: K splits of every tile, or (bit 31) of the last `tail` tiles
    // only, dispatched last; their partials go to tail_part
    const bool has_tail = ks_tail >> 31;
    const uint32_t tail = has_tail ? ks_tail & 0xffffu : 0u, whole = tiles - tail;
    const bool in_tail = has_tail && blockIdx.x >= whole;
    const uint32_t ks = has_tail ? (in_tail ? (ks_tail >> 16) & 0x7fffu : 1u) : ks_tail;
    const uint32_t span = in_tail ? tail : tiles, at = in_tail ? blockIdx.x - whole : blockIdx.x;
    const uint32_t zs = at / span, t = at % span + (in_tail ? whole : 0u), tm = t / nt, tn = t % nt;
    const uint32_t main_s = 8 * bpr, total = main_s + ext / 32;
    // this split's stages: equal shares, cut at super-blocks
    auto cut = [&](uint32_t z) {
        if (z == ks) return total;
        const uint32_t c = (uint32_t)((uint64_t)total * z / ks) & ~7u;
        return c < main_s ? c : main_s;
    };
    const uint32_t s_lo = cut(zs), s_hi = cut(zs + 1);

    typedef __attribute__((address_space(3))) uint8_t *lds_b;
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((lds_b)lds);
    // 64 x W dwords from base + off into LDS; outside the compiler's memory
    // model (its loads and waits know nothing of it): every wait for it is
    // explicit, and so is the wait state that a load into LDS needs after a
    // scalar write of M0 (the compiler does not look for hazards in here)
    auto copy = [&](auto w, const uint8_t *base, uint32_t off, uint32_t dst) {
        if constexpr (decltype(w)::value == 4)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "m0");
        else
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(dst) : "m0");
    };
    // where the next stage's copies come from: this wave's blocks i of the
    // tiles (their offsets fixed but for the step to the extra k range)
    const uint8_t *pa = nullptr, *pl = nullptr, *pb = nullptr, *ps = nullptr;
    uint32_t off[NB / 4], fs = s_lo;
    auto point = [&]() {   // at stage fs
        const bool main = fs < main_s;
        const uint32_t kb = main ? 2 * fs : 2 * (fs - main_s), row_blocks = tile_pitch(main ? 256 * bpr : ext);
        const size_t oa = ((size_t)(tm * (BM / 32)) * row_blocks + kb) * 1024, ob = ((size_t)(tn * (BN / 32)) * row_blocks + kb) * 1024;
        pa = (main ? xh : xe) + oa;
        pl = (main ? xl : xe) + oa;
        pb = (main ? wt : we) + ob;
#pragma unroll
        for (uint32_t i = 0; i < NB / 4; i++) {
            const uint32_t blk = 4 * i + wave, idx = blk < SW * AB ? blk % AB : blk - SW * AB;
            off[i] = ((idx >> 1) * row_blocks + (idx & 1u)) * 1024 + lane * 16;
        }
        ps = reinterpret_cast<const uint8_t *>(scale + (size_t)tile_scale_row(GRAN, fs, main_s) * np + tn * BN + 64 * wave);
    };
    auto fetch = [&](uint32_t b) {   // stage fs into buffer b, then on to the next (the last one again past the end)
        const uint32_t dst = lds0 + b * BUF;
#pragma unroll
        for (uint32_t i = 0; i < NB / 4; i++)
            copy(std::integral_constant<int, 4>{}, 4 * i < AB ? pa : 4 * i < SW * AB ? pl : pb, off[i], dst + (4 * i + wave) * 1024);
        // scales, a quarter of each 1 KB row per wave (with one per
        // super-block: its first stage's copy is the one read)
        if (GRAN != 256 || NBUF > 2 || (fs & 7u) == 0) {
#pragma unroll
            for (uint32_t i = 0; i < SCW; i++)
                copy(std::integral_constant<int, 1>{}, ps + (size_t)i * np * 4, lane * 4, dst + (NB + i) * 1024 + 256 * wave);
        }
        if (fs + 1 < s_hi) {
            fs++;
            pa += 2048;
            pl += 2048;
            pb += 2048;
            ps += (size_t)tile_scale_step(GRAN, fs, main_s) * np * 4;
            if (fs == main_s) point();
        }
    };
    constexpr int LOADS = NB / 4 + SCW;   // copies per wave and stage
    static_assert(AB % 4 == 0, "a copy's four blocks are of one operand");

    f16v acc[MT][NT];
#pragma unroll
    for (uint32_t i = 0; i < MT; i++)
#pragma unroll
        for (uint32_t j = 0; j < NT; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
    const uint32_t col = lane & 31u;
    auto scale_acc = [&](uint32_t j, float f) {
#pragma unroll
        for (uint32_t i = 0; i < MT; i++) acc[i][j] *= f;
    };
    auto units = [&](uint32_t sb) {   // back to absolute units
#pragma unroll
        for (uint32_t j = 0; j < NT; j++)
            scale_acc(j, scale[(size_t)(bpr + sb) * np + tn * BN + wn * (BN / 2) + 32 * j + col]);
    };
    half8 xa[2][MT], xb[2][MT], w[2][NT];
    auto operands = [&](uint32_t b, uint32_t k) {
        const uint8_t *buf = lds + b * BUF;
        const uint8_t *a = buf + wm * (BM / 64) * 2048 + 16 * lane, *q = buf + SW * AB * 1024 + wn * (BN / 64) * 2048 + 16 * lane;
#pragma unroll
        for (uint32_t i = 0; i < MT; i++) {
            xa[k][i] = *reinterpret_cast<const half8 *>(a + (2 * i + k) * 1024);
            if constexpr (SW == 2) xb[k][i] = *reinterpret_cast<const half8 *>(a + AB * 1024 + (2 * i + k) * 1024);
        }
#pragma unroll
        for (uint32_t j = 0; j < NT; j++) w[k][j] = *reinterpret_cast<const half8 *>(q + (2 * j + k) * 1024);
    };
    // the stage in buffer b, of the main range, or of the extra one (absolute
    // units, one X operand)
    auto multiply = [&](uint32_t b, auto main_t) {
        constexpr bool main = decltype(main_t)::value;
        const float *sc = reinterpret_cast<const float *>(lds + b * BUF + NB * 1024) + wn * (BN / 2) + col;
        auto mfma = [](half8 x, half8 z, f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, z, c, 0, 0, 0); };
        const f16v zero = {};
        if constexpr (GRAN == 256 || !main) {
#pragma unroll
            for (uint32_t k = 0; k < 2; k++) {
                if constexpr (GRAN != 256) operands(b, k);
#pragma unroll
                for (uint32_t j = 0; j < NT; j++)
#pragma unroll
                    for (uint32_t i = 0; i < MT; i++) acc[i][j] = mfma(xa[k][i], w[k][j], acc[i][j]);
                if constexpr (SW == 2 && main) {
#pragma unroll
                    for (uint32_t j = 0; j < NT; j++)
#pragma unroll
                        for (uint32_t i = 0; i < MT; i++) acc[i][j] = mfma(xb[k][i], w[k][j], acc[i][j]);
                }
            }
        } else if constexpr (GRAN == 16) {
            // each k-step's products from zero, then added times their scale
#pragma unroll
            for (uint32_t k = 0; k < 2; k++) {
                operands(b, k);
#pragma unroll
                for (uint32_t j = 0; j < NT; j++) {
                    const float f = sc[k * 256 + 32 * j];
#pragma unroll
                    for (uint32_t i = 0; i < MT; i++) {
                        f16v tmp = mfma(xa[k][i], w[k][j], zero);
                        if constexpr (SW == 2) tmp = mfma(xb[k][i], w[k][j], tmp);
                        acc[i][j] += f * tmp;
                    }
                }
            }
        } else {
            operands(b, 0);
            operands(b, 1);
#pragma unroll
            for (uint32_t j = 0; j < NT; j++) {
                const float f = sc[32 * j];
#pragma unroll
                for (uint32_t i = 0; i < MT; i++) {
                    f16v tmp = mfma(xa[0][i], w[0][j], zero);
                    tmp = mfma(xa[1][i], w[1][j], tmp);
                    if constexpr (SW == 2) {
                        tmp = mfma(xb[0][i], w[0][j], tmp);
                        tmp = mfma(xb[1][i], w[1][j], tmp);
                    }
                    acc[i][j] += f * tmp;
                }
            }
        }
    };

    // NBUF - 1 stages in flight (every wave always waits for the same count)
    point();
#pragma unroll
    for (uint32_t i = 0; i < NBUF - 1; i++) fetch(i);
    // stage s has landed (loads complete in issue order: at most the later
    // stages' are outstanding) for every wave, and every wave is done reading
    // the buffer the next copy goes to
    auto arrive = [&]() {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NBUF - 2) * LOADS) : "memory");
    };
    auto stage = [&](uint32_t s, auto bc) {
        constexpr uint32_t b = decltype(bc)::value;
        arrive();
        operands(b, 0);
        operands(b, 1);
        __builtin_amdgcn_sched_barrier(0);   // the operand reads go out before the copies' issue
        fetch((b + NBUF - 1) % NBUF);
        if ((s & 7u) == 0 && s > s_lo) {   // a new super-block
            const float *sc = reinterpret_cast<const float *>(lds + b * BUF + NB * 1024) + wn * (BN / 2) + col;
#pragma unroll
            for (uint32_t j = 0; j < NT; j++) scale_acc(j, sc[32 * j]);
        }
        multiply(b, std::true_type{});   // (the formats of this granularity have no extra range)
    };
    if constexpr (GRAN == 256) {
        for (uint32_t s = s_lo; s < s_hi; s += NBUF) {
            stage(s, std::integral_constant<uint32_t, 0>{});
            if (s + 1 >= s_hi) break;
            stage(s + 1, std::integral_constant<uint32_t, 1>{});
            if constexpr (NBUF > 2) {
                if (s + 2 >= s_hi) break;
                stage(s + 2, std::integral_constant<uint32_t, 2 % NBUF>{});
            }
        }
    } else {
        // (not unrolled over the buffers, operands read where they are used:
        // unrolled, the scheduler spilled the sets' products)
        uint32_t s = s_lo, b = 0;
        auto next = [&]() {
            arrive();
            fetch(b == 0 ? NBUF - 1 : b - 1);
        };
        for (; s < s_hi && s < main_s; s++, b = b + 1 == NBUF ? 0u : b + 1) {
            next();
            multiply(b, std::true_type{});
        }
        for (; s < s_hi; s++, b = b + 1 == NBUF ? 0u : b + 1) {
            next();
            multiply(b, std::false_type{});
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no copy outlives the workgroup
    if constexpr (GRAN == 256)
        if (s_hi > s_lo) units(s_hi / 8 - 1);

    // rows 8 (e / 4) + 4 (lane / 32) + e % 4 of column lane % 32 of each tile
    float *const ys = y + (ks > 1 && !in_tail ? (size_t)zs * M * ldy : 0);
    float *const tp = tail_part + (size_t)at * BM * BN;
#pragma unroll
    for (uint32_t i = 0; i < MT; i++) {
        float rs[16];
#pragma unroll
        for (uint32_t e = 0; e < 16; e++) {
            const uint32_t m = tm * BM + wm * (BM / 2) + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3u);
            rs[e] = rowscale[m < M ? m : M - 1u];
        }
#pragma unroll
        for (uint32_t j = 0; j < NT; j++) {
            const uint32_t r = tn * BN + wn * (BN / 2) + 32 * j + col;
#pragma unroll
            for (uint32_t e = 0; e < 16; e++) {
                const uint32_t ml = wm * (BM / 2) + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3u), m = tm * BM + ml;
                const float v = acc[i][j][e] * rs[e];
                if (in_tail) {
                    tp[ml * BN + wn * (BN / 2) + 32 * j + col] = v;
                } else if (m < M && r < N) {
                    float *p = ys + (size_t)m * ldy + r;
                    *p = accumulate && ks == 1 ? *p + v : v;
                }
            }
        }
    }
}

// y's tail tiles (first..) from their partials part[ks][tail][BM][BN], z ascending
__global__ __launch_bounds__(256) void gemm_tail_kernel(const float *__restrict__ part, float *__restrict__ y, uint32_t M,
                                                        uint32_t N, uint32_t ldy, uint32_t first, uint32_t ks,
                                                        uint32_t accumulate) {
    const uint32_t tail = gridDim.y, nt = (N + kTiledBn - 1) / kTiledBn, t = first + blockIdx.y;
    const uint32_t i = 4 * (blockIdx.x * 256 + threadIdx.x);   // four columns of the tile
    const float4 *p = reinterpret_cast<const float4 *>(part + (size_t)blockIdx.y * kTiledBm * kTiledBn + i);
    float4 s = p[0];
    for (uint32_t z = 1; z < ks; z++) {
        const float4 v = p[(size_t)z * tail * (kTiledBm * kTiledBn / 4)];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    const uint32_t m = t / nt * kTiledBm + i / kTiledBn, r = t % nt * kTiledBn + i % kTiledBn;
    if (m >= M) return;
    const float v[4] = {s.x, s.y, s.z, s.w};
    float *yr = y + (size_t)m * ldy;
#pragma unroll
    for (uint32_t e = 0; e < 4; e++)
        if (r + e < N) yr[r + e] = accumulate ? yr[r + e] + v[e] : v[e];
}

// Without K splits: the tiles past the last whole round of resident
// workgroups (two per CU), when they fill at most half a round, run as K
// splits that fill it (16 of 528 tiles alone took half as long as the 512
// before them).  Returns their number, and their splits.
uint32_t tail_tiles(uint32_t tiles, uint32_t bpr, uint32_t *ks) {
    const uint32_t slots = 2 * (uint32_t)device_cus(), r = tiles % slots;
    *ks = 1;
    if (tiles < slots || r == 0 || r > slots / 2) return 0;
    const uint32_t most = bpr / 2 < 16 ? bpr / 2 : 16;
    *ks = slots / r < most ? slots / r : most;
    return *ks > 1 ? r : 0;
}

template <uint32_t DT, uint32_t GRAN>
int run_pass(hipStream_t s, const TiledPlan &p, const TiledPass &a, uint32_t r_lo, uint32_t n) {
    const uint32_t bpr = a.k / 256, np = (n + kTiledBn - 1) / kTiledBn * kTiledBn;
    const Mats mt{{a.w[0], a.w[1], a.w[2]}, a.s1, a.s2};
    uint8_t *wt = static_cast<uint8_t *>(a.wt), *we = static_cast<uint8_t *>(a.we);
    float *sc = static_cast<float *>(a.ws);
    hipLaunchKernelGGL((tile_weights_kernel<DT, GRAN>), dim3(bpr, (n + 31) / 32), dim3(256), 0, s, mt, r_lo, n, np, bpr,
                       p.ext, wt, we, sc);
    int rc = check_launch("quantized_gemm: weight tiles");
    if (rc) return rc;
    const uint32_t tiles = (n + kTiledBn - 1) / kTiledBn * (p.mp / kTiledBm);
    uint32_t tks = 1;
    const uint32_t tail = p.ks == 1 ? tail_tiles(tiles, bpr, &tks) : 0;
    const uint32_t grid = tail ? tiles - tail + tail * tks : tiles * p.ks;
    const uint32_t ks_tail = tail ? tail | tks << 16 | 1u << 31 : p.ks;
    float *const tp = static_cast<float *>(a.tail);
#define YULE_TILED_ARGS                                                                                              \
    static_cast<const uint8_t *>(a.xh), wt, static_cast<const uint8_t *>(a.xl), sc, static_cast<const uint8_t *>(a.xe), \
        we, a.m, n, bpr, p.ext, np, ks_tail, a.y + r_lo, a.n, a.rowscale, a.accumulate ? 1u : 0u, tp
    hipLaunchKernelGGL((gemm_tiled_kernel<GRAN == 256 ? 1 : 2, GRAN>), dim3(grid), dim3(256), 0, s, YULE_TILED_ARGS);
#undef YULE_TILED_ARGS
    if (tail) {
        if ((rc = check_launch("quantized_gemm: tiled product"))) return rc;
        hipLaunchKernelGGL(gemm_tail_kernel, dim3(kTiledBm * kTiledBn / 1024, tail), dim3(256), 0, s, tp, a.y + r_lo, a.m,
                           n, a.n, tiles - tail, tks, a.accumulate ? 1u : 0u);
    }
    return check_launch("quantized_gemm: tiled product");
}

}  // namespace

// The line between this path and gemm.hip's, in rows and multiply-adds (10^9)
// of the product: below it the expansion of the weights (4.7 TB/s over their
// bytes and 2 per weight when alone) and the extra launches cost more than
// the product saves.  Measured, rows x weight rows x k, gemm.hip -> here, us:
//   f32 X   Q6_K  300 x 2048 x 5632 89 -> 72, 1531 x 2048 x 5632 447 -> 138, 150 x 700 x 14336 69 -> 63,
//                 140 x 4096 x 2048 49 -> 54
//           Q8_0  300 x 4096 x 4096 97 -> 74, 1000 x 512 x 1024 36 -> 41; Q4_0 150 x 4096 x 8192 102 -> 89;
//           Q8_K  256 x 4096 x 4096 90 -> 61, 150 x 1024 x 2048 36 -> 38
//           Q4_K  768 x 11264 x 2048 135 -> 128, 1531 x 11264 x 2048 233 -> 185, 512 x 14336 x 4096 193 -> 196,
//                 1531 x 2560 x 2048 75 -> 76; Q5_K 1000 x 4096 x 4096 145 -> 124
//   bf16 X  Q6_K  1531 x 4096 x 4096 139 -> 110, 800 x 4096 x 4096 88 -> 79, 1024 x 2048 x 2048 43 -> 46
//           the others gain at most 6% at 2048 rows and lose below: gemm.hip
// Q6_K with f32 X of up to 511 rows by whole tiles of 128 rows and from three
// columns of tiles on: 200 x 2048 x 4096 51 -> 56, 256 x 4096 x 2048 52 -> 55, 300 x
// 512 x 14080 72 -> 78, 130 x 3000 x 4096 74 -> 57, 400 x 1200 x 4096 64 -> 57.
// bf16 X (Q6_K): below 1280 rows of X and 84 tiles the product gains nothing,
// but where the columns of tiles are a multiple of four from eight on (an XCD
// then keeps to few of them, and to their weights) and k is long: 776 x 2230 x 8192 97 -> 120, 896 x 1500 x 11520 98 ->
// 102, 1000 x 1024 x 14336 91 -> 96; 776 x 2048 x 11520 121 -> 103, 776 x 3000 x 11520
// 148 -> 131, 1300 x 1500 x 11520 144 -> 126.
// Q4_K of few weight rows gains nothing (2000 x 1024 x 14080 226 -> 243, 1290 x
// 1024 x 14080 168 -> 165), Q5_K does (180 -> 165).
static bool tiled_wins(uint32_t m, uint32_t n, uint32_t k, uint32_t dtype, bool f32x) {
    const bool sums = dtype == YULE_DTYPE_Q4_K || dtype == YULE_DTYPE_Q5_K, q6 = dtype == YULE_DTYPE_Q6_K;
    const double work = 1e-9 * m * n * k;
    if (!f32x) {
        const uint32_t cols = (n + kTiledBn - 1) / kTiledBn, tiles = (m + kTiledBm - 1) / kTiledBm * cols;
        return q6 && m >= 768 && work >= 10 &&
               (tiles >= 84 || (m >= 1280 && tiles >= 44) || (cols >= 8 && cols % 4 == 0 && k >= 8192));
    }
    if (q6 && m < 512) return m > 128 && n > 2 * kTiledBn && 1e-9 * ((m + kTiledBm - 1) / kTiledBm * kTiledBm) * n * k >= 2.25;
    return sums ? m >= 700 && work >= 15 && (n >= 1536 || dtype == YULE_DTYPE_Q5_K) : m > 128 && work >= (q6 ? 1.5 : 3.0);
}

bool gemm_tiled_plan(uint32_t m, uint32_t n, uint32_t k, uint32_t dtype, bool f32x, TiledPlan *p) {
    static const int min_rows = env_int("YULE_GEMM_TILED_MIN", 0);   // (comparison and tests: from this many rows on)
    if (k % 256 || (!f32x && dtype != YULE_DTYPE_Q6_K)) return false;
    if (!(min_rows ? m >= (uint32_t)min_rows : tiled_wins(m, n, k, dtype, f32x))) return false;
    p->gran = dtype == YULE_DTYPE_Q6_K ? (f32x ? 16 : 256) : 32;
    p->mp = (m + kTiledBm - 1) / kTiledBm * kTiledBm;
    p->ext = gemm_ext_cols(dtype, k);
    // passes over at most 256 MB of weight tiles
    const uint32_t most = (uint32_t)(((size_t)256 << 20) / (2 * (size_t)k)) / 256 * 256;
    p->n_chunk = most < 256 ? 256 : n < most ? n : most;
    const uint32_t np = (p->n_chunk + kTiledBn - 1) / kTiledBn * kTiledBn, bpr = k / 256;
    const uint32_t tiles = np / kTiledBn * (p->mp / kTiledBm), slots = 2 * (uint32_t)device_cus();
    p->ks = 1;
    if (p->n_chunk == n && tiles <= slots / 2) {
        p->ks = slots / tiles;
        if (p->ks > bpr / 2) p->ks = bpr / 2 ? bpr / 2 : 1;
    }
    uint32_t tks = 1, last_n = n % p->n_chunk ? n % p->n_chunk : p->n_chunk;
    auto tail_bytes = [&](uint32_t rows) {
        const uint32_t r = p->ks == 1 ? tail_tiles((rows + kTiledBn - 1) / kTiledBn * (p->mp / kTiledBm), bpr, &tks) : 0;
        return (size_t)r * tks * kTiledBm * kTiledBn * sizeof(float);
    };
    p->t_bytes = tail_bytes(p->n_chunk) > tail_bytes(last_n) ? tail_bytes(p->n_chunk) : tail_bytes(last_n);
    p->w_bytes = (size_t)np / 32 * tile_pitch(k) * kTileBytes;
    p->we_bytes = p->ext ? (size_t)np / 32 * tile_pitch(p->ext) * kTileBytes : 0;
    p->s_bytes = ((size_t)(p->gran == 256 ? 2 * bpr : k / p->gran) * np + 256) * sizeof(float);
    p->x_bytes = (size_t)p->mp / 32 * tile_pitch(k) * kTileBytes;
    p->xe_bytes = p->ext ? (size_t)p->mp / 32 * tile_pitch(p->ext) * kTileBytes : 0;
    return true;
}

int launch_x_tiles(hipStream_t s, const void *x, bool f32x, uint32_t m, uint32_t k, uint32_t ext, const float *norm_w,
                   float eps, bool glu, void *xh, void *xl, void *xe, float *rowscale, const GemmRed *pending) {
    const bool red = pending && pending->ks > 1;
#define YULE_X_ARGS                                                                                                  \
    x, norm_w, k, eps, glu ? 1u : 0u, m, ext, static_cast<uint8_t *>(xh), static_cast<uint8_t *>(xl),              \
        static_cast<uint8_t *>(xe), rowscale, red ? pending->part : nullptr, red ? pending->ks : 0u,               \
        red ? pending->ny : 0u, red && pending->accumulate ? 1u : 0u
    if (m >= 4u * (uint32_t)device_cus()) {
        if (f32x) hipLaunchKernelGGL((x_tiles_kernel<true, 4>), dim3((m + 3) / 4), dim3(256), 0, s, YULE_X_ARGS);
        else hipLaunchKernelGGL((x_tiles_kernel<false, 4>), dim3((m + 3) / 4), dim3(256), 0, s, YULE_X_ARGS);
    } else {
        if (f32x) hipLaunchKernelGGL((x_tiles_kernel<true, 1>), dim3(m), dim3(256), 0, s, YULE_X_ARGS);
        else hipLaunchKernelGGL((x_tiles_kernel<false, 1>), dim3(m), dim3(256), 0, s, YULE_X_ARGS);
    }
#undef YULE_X_ARGS
    return check_launch("quantized_gemm: x tiles");
}

int launch_gemm_tiled(hipStream_t s, const TiledPlan &p, const TiledPass &a) {
    for (uint32_t r = 0; r < a.n; r += p.n_chunk) {
        const uint32_t n = a.n - r < p.n_chunk ? a.n - r : p.n_chunk;
        int rc;
        switch (a.dtype) {
        case YULE_DTYPE_Q4_K: rc = run_pass<YULE_DTYPE_Q4_K, 32>(s, p, a, r, n); break;
        case YULE_DTYPE_Q5_K: rc = run_pass<YULE_DTYPE_Q5_K, 32>(s, p, a, r, n); break;
        case YULE_DTYPE_Q8_K: rc = run_pass<YULE_DTYPE_Q8_K, 32>(s, p, a, r, n); break;
        case YULE_DTYPE_Q6_K:
            rc = a.f32x ? run_pass<YULE_DTYPE_Q6_K, 16>(s, p, a, r, n) : run_pass<YULE_DTYPE_Q6_K, 256>(s, p, a, r, n);
            break;
        case YULE_DTYPE_Q8_0: rc = run_pass<YULE_DTYPE_Q8_0, 32>(s, p, a, r, n); break;
        default: rc = run_pass<YULE_DTYPE_Q4_0, 32>(s, p, a, r, n); break;
        }
        if (rc) return rc;
    }
    return YULE_OK;
}

}  // namespace yule
