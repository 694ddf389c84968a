// gemm_tiled.h — prefill GEMM over operands laid out as matrix-core tiles
// (gemm_tiled.hip), used by gemm.hip for products of many rows.
#pragma once

#include "internal.h"

namespace yule {

// Operand tiles: 32 rows x 16 k in f16 as 64 16-byte units, unit 32 h + r =
// the eight k 8 h..8 h + 7 of row r: one 1 KB block is the operand of a 32 x
// 32 x 16 MFMA, read by lane l at byte 16 l.  A matrix is [row / 32][k / 16]
// blocks, each 32 rows' padded by two blocks: workgroups that walk k in step
// over rows a power of two apart would otherwise all be on the same memory
// channels.  k runs in the X pre-pass's order (each four as {0, 2, 1, 3}).
constexpr size_t kTileBytes = 1024;
__host__ __device__ inline uint32_t tile_pitch(uint32_t k) { return k / 16 + 2; }   // blocks from 32 rows to the next
__host__ __device__ inline size_t tile_unit(uint32_t row, uint32_t k8, uint32_t pitch) {   // byte offset of unit (row, k = 8 k8)
    return ((size_t)(row >> 5) * pitch + (k8 >> 1)) * kTileBytes + ((k8 & 1u) << 9) + ((row & 31u) << 4);
}

// The extra k range of the formats with a min term (Q4_K, Q5_K): X's sub-block
// sums (hi, hi, lo) against -(dmin * mn) (hi, lo, hi), K / 32 of each, padded
// with zeros to whole stages of 32; 0 for the others
__host__ __device__ inline uint32_t gemm_ext_cols(uint32_t dtype, uint32_t k) {
    return dtype == YULE_DTYPE_Q4_K || dtype == YULE_DTYPE_Q5_K ? (3 * (k / 32) + 31) / 32 * 32 : 0;
}

// Scales: gemm_tiled_kernel copies a stage's (32 k) rows of the scale array
// [k / gran][np] beside its tiles.  The row a walk over the stages starts
// from at stage `stage`, and by how many rows it moves on when it comes to the
// next one, `stage`: the extra range (from stage main_s on) has no scales of
// its own, and its copies (in the wait counts, never read) stay on the last
// row of the main range.
__host__ __device__ constexpr uint32_t tile_scale_rows(uint32_t gran) { return gran == 16 ? 2u : 1u; }   // per stage
__host__ __device__ inline uint32_t tile_scale_row(uint32_t gran, uint32_t stage, uint32_t main_s) {
    const uint32_t s = stage < main_s ? stage : main_s - 1u;
    return gran == 16 ? 2 * s : gran == 32 ? s : s >> 3;
}
__host__ __device__ inline uint32_t tile_scale_step(uint32_t gran, uint32_t stage, uint32_t main_s) {
    return stage >= main_s || (gran == 256 && (stage & 7u)) ? 0u : tile_scale_rows(gran);
}

struct TiledPlan {
    uint32_t gran;                // k per weight scale (256, 32 or 16)
    uint32_t ks, n_chunk;         // K splits; weight rows per pass (all of them with splits)
    uint32_t mp, ext;             // X rows padded to whole workgroup tiles; extra k
    size_t w_bytes, we_bytes, s_bytes, x_bytes, xe_bytes;   // of one pass's weights, of X (one of hi, lo)
    size_t t_bytes;               // partials of the last tiles
};

// false: gemm.hip's kernels serve this product
bool gemm_tiled_plan(uint32_t m, uint32_t n, uint32_t k, uint32_t dtype, bool f32x, TiledPlan *p);

struct TiledPass {
    const uint8_t *w[3];          // matrices stacked along Y's columns, rows [0, s1), [s1, s2), [s2, n)
    uint32_t s1, s2;
    uint32_t m, n, k, dtype;
    bool f32x, accumulate;
    const void *xh, *xl, *xe;     // X tiles (pre-pass)
    void *wt, *we, *ws, *tail;    // one pass's weight tiles, their extra k, scales; partials of its last tiles
    const float *rowscale;
    float *y;                     // [m][n], or with splits the partials [ks][m][n]
};
// X (bf16, or f32: hi and lo) as tiles, its extra k range and row scales; the
// arguments as gemm_xprep_kernel's (gemm.hip)
int launch_x_tiles(hipStream_t s, const void *x, bool f32x, uint32_t m, uint32_t k, uint32_t ext, const float *norm_w,
                   float eps, bool glu, void *xh, void *xl, void *xe, float *rowscale, const GemmRed *pending);
int launch_gemm_tiled(hipStream_t s, const TiledPlan &p, const TiledPass &a);

}  // namespace yule
