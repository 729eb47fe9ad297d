// qgemm.h -- grouped int8-MFMA GEMM for prefill (many token rows per matrix).
//
// Y[m][n] = s_w[n] * sum_k W[n][k] * x[m][k] for the token rows m of a task,
// with W in the container's q8 (int8) or q4 (nibble) packing, used as exact
// int8 operands of v_mfma_i32_32x32x32_i8.  Activations are quantised per
// token row into three int8 limbs, x ~= s_x * (65536 * hi + 256 * mid + lo)
// with |65536 * hi + 256 * mid + lo| <= 2^22 (23 significant bits against the
// row's max, the precision of an fp32 operand), and every limb is multiplied
// by the same weight fragment; the int32 sums are combined in fp32 in the
// epilogue.  The per-element rounding of x is at most amax / 2^23, so a row
// whose max is 100x its rms still sees ~4e-6 relative error: outputs match the
// fp32 matmul of moonlight_kernels.metal:62-130 to fp32 rounding while every
// product and sum is exact.
//
// A launch covers a table of independent tasks (one per active routed expert
// plus the shared expert, or one dense matrix).  Tiles are 128 token rows x
// 256 weight rows (SwiGLU pairs: 128 gate + 128 matching up rows, 128
// outputs), or 64 or 32 token rows x 256 weight rows where a launch's tasks hold
// few rows each; the tile order groups 4 row tiles of a task so that consecutive
// workgroups on one XCD share weight tiles in that XCD's L2.
#pragma once

#include <algorithm>

#include "gemv_impl.h"

namespace mlh {

constexpr int kQgBM = 128;  // token rows per tile
constexpr int kQgBMMid = 64;
constexpr int kQgBMSmall = 32;  // token rows per tile of few-row launches
constexpr int kQgBW = 256;  // weight rows per tile
constexpr int kQgBK = 64;   // k per pipeline stage
constexpr int kQgGroup = 4; // row tiles per locality group
constexpr int kQgMaxTasks = 272;
// Outputs and residuals of a tile are addressed by 31-bit byte offsets from the
// tile's first row (columns past the last get the largest one, which has to lie
// outside the tile's rows): floats between rows are at most this many.
constexpr long kQgOutside = 0x7FFFFFFFL;
constexpr long kQgMaxStride = kQgOutside / (4 * kQgBM);

// Quantised activations lie in blocks of 8 rows x 128 columns: the three limbs'
// (hi, mid, lo) 8 x 128 bytes one after the other, a row block's column blocks
// one after the other.  A tile's copy of 8 rows of a limb is then 1 KB in one
// piece where its rows follow each other (a probe of the tile's fill alone:
// 1780 clocks a 64-k share from such pieces, 2300 from 128-byte runs of limb
// planes, 2900 from 64-byte runs).
constexpr int kLimbs = 3;
template <int LIMBS = kLimbs>
__host__ __device__ inline long limb_row_block(int width) {  // bytes per 8 rows
    return (long)((width + 127) / 128) * (LIMBS * 1024);
}
template <int LIMBS = kLimbs>
__host__ __device__ inline long limb_bytes(long rows, int width) {
    return (rows + 7) / 8 * limb_row_block<LIMBS>(width);
}
// Byte of limb 0 at (row, col); limb l is 1024 l further.
template <int LIMBS = kLimbs>
__host__ __device__ inline long limb_at(long row, int col, int width) {
    return (row >> 3) * limb_row_block<LIMBS>(width) + (col >> 7) * (LIMBS * 1024) + (row & 7) * 128 +
           (col & 127);
}

// Tasks of gathered rows (a_rows) reach each from row 0 by a 32-bit byte offset;
// offsets from kQgGatherBytes on read zeros.
constexpr long kQgGatherBytes = 0xF0000000L;
// Most token rows of one moe_gemm call, whose expert tasks gather them.
inline long moe_gemm_max_rows(int hidden) { return kQgGatherBytes / limb_row_block(hidden) * 8; }

// One independent product: rows x n_out outputs, reduction length k.
struct GemmTask {
    const uint8_t *w = nullptr, *w2 = nullptr;  // [n_out][k] packed (w2: up rows, SwiGLU)
    const float *s = nullptr, *s2 = nullptr;    // per weight row scales
    int rows = 0, n_out = 0, k = 0;
    int w_ld = 0;  // weight row length in elements (0: k); a k slice of longer rows
    // quantised activations (limb blocks), from their first column on (a
    // multiple of 128); a_width: columns of a whole row
    const int8_t *a = nullptr;
    int a_width = 0;
    const float *a_scale = nullptr;
    // activation row of token row m (of a and a_scale): a_rows[m] if set, else
    // a_row0 + m
    const int *a_rows = nullptr;
    int a_row0 = 0;
    float *y = nullptr;           // output row m at y + m * y_stride
    long y_stride = 0;
    const float *resid = nullptr;  // optional residual (y = resid + product)
    long resid_stride = 0;
};

struct QGemmLaunch {
    const GemmTask *tasks = nullptr;  // device table (MoE); nullptr: `single`
    const int *tile_start = nullptr;  // device [tasks + 1] tile prefix sums
    const int *n_routed = nullptr;    // device: routed task count (shared tasks follow)
    int n_shared = 1;                 // shared-expert tasks after the routed ones
    int range = 0;                    // 0 all tasks, 1 routed only, 2 shared only
    int splits = 1;                   // shares of `single`'s reduction
    GemmTask single;
};

// Per-row activation quantisation (optionally RMSNorm'ed first,
// moonlight_kernels.metal:23-41): rows of `x` (stride x_stride floats) ->
// limb blocks at q (limb_bytes(rows, width)) and scales.
int quantize_activations(const float *x, long x_stride, int rows, int width, const float *norm_w,
                         float eps, int8_t *q, float *scale, hipStream_t stream);

// Tile kinds: the weight-streaming tile with 16 token rows, the LDS tiles
// with 32, 64 or 128.
enum TileKind { kTileStream16 = 0, kTileLds32 = 1, kTileLds64 = 2, kTileLds128 = 3 };

inline int tile_bm(int kind) {
    return kind == kTileStream16 ? 16
           : kind == kTileLds32  ? kQgBMSmall
           : kind == kTileLds64  ? kQgBMMid
                                 : kQgBM;
}

inline int host_tiles(bool dual, int rows, int n_out, int bm) {
    const int outw = dual ? kQgBW / 2 : kQgBW;
    return ((rows + bm - 1) / bm) * ((n_out + outw - 1) / outw);
}

// Dense projections: the smallest tile that covers the matrix in one round of
// the CUs, else 128 rows.  Tiles of 32 / 64 / 128 rows: 2048 x 2048 at 600 rows
// 19.8 / 23.9 / 36.4 us, at 1200 rows 36.8 / 27.5 / 39.1, at 2048 rows 42.4 /
// 31.1 / 45.0; 3648 x 2048 at 600 rows 34.9 / 25.0 / 37.9, at 1200 rows 52.2 /
// 48.0 / 41.0, at 2048 rows 76.4 / 57.8 / 48.6.
inline int dense_tile(int rows, bool k128, int n_out, bool dual) {
    if (k128 && rows <= 16) return kTileStream16;
    if (host_tiles(dual, rows, n_out, kQgBMSmall) <= 256) return kTileLds32;
    return host_tiles(dual, rows, n_out, kQgBMMid) <= 256 ? kTileLds64 : kTileLds128;
}

// One dense task, e.g. a prefill projection.  Epilogue: plain or residual
// (task.resid) or SwiGLU pair (dual, task.w2 = up).
int qgemm_single(int fmt, bool dual, const GemmTask &task, hipStream_t stream);

// gemv() of many token rows on the same tiles with four limbs (30 bits of the
// row's largest value, as the other matrix-core GEMVs): quantises the rows
// into the library's own scratch and multiplies.  False, launching nothing,
// for shapes it does not take; with `name` set it launches nothing and stores
// the kernel's template name.
bool gemv_tiles(const GemvParams &p, hipStream_t stream, std::string *name = nullptr);
// Token rows of one of its launches: what the scratch for their limbs holds.
constexpr long kTilesBytes = 64L << 20;
constexpr int kTilesRows = 8192;
inline long tiles_chunk(long rows, int width) {
    return std::min({rows, (long)kTilesRows, kTilesBytes / limb_row_block<4>(width) * 8});
}

// MoE prefill: builds the per-expert task tables from the device route tables
// and runs both expert stages for all active experts plus the shared expert.
struct MoeGemmParams {
    int rows = 0, experts = 0, top_k = 0, hidden = 0, inter = 0, shared_width = 0;
    // with route_in_prep (rows <= kRouteOneGroupRows, experts <= 64 not
    // required): the routing of the batch from route.logits and its tables
    // run in the first launch (no routing launch before moe_gemm)
    int route_in_prep = 0;
    RouteParams route;
    int expert_fmt = kQ8, shared_fmt = kQ8, has_shared = 1;
    const ExpertWeights *expert_table = nullptr;
    const uint8_t *shared_gate = nullptr, *shared_up = nullptr, *shared_down = nullptr;
    const float *shared_gate_s = nullptr, *shared_up_s = nullptr, *shared_down_s = nullptr;
    const int *n_unique = nullptr, *unique = nullptr, *counts = nullptr, *offsets = nullptr;
    const int *list_rows = nullptr;
    const float *x = nullptr;  // residual stream [rows, hidden]
    const float *norm_w = nullptr;
    float eps = 1e-5f;
    // scratch: limb blocks and scales
    int8_t *xq = nullptr;       // [rows, hidden]
    float *xq_scale = nullptr;  // [rows]
    int8_t *hq = nullptr;       // [rows*top_k, inter]
    float *hq_scale = nullptr;  // [rows*top_k]
    int8_t *sq = nullptr;       // [rows, shared_width]
    float *sq_scale = nullptr;  // [rows]
    GemmTask *tasks = nullptr;                   // [2][kQgMaxTasks]
    int *tile_start = nullptr;                   // [2][kQgMaxTasks + 1]
    // outputs (same layouts as the GEMV expert path)
    float *expert_hidden = nullptr;  // [rows*top_k, inter]
    float *expert_out = nullptr;     // [rows*top_k, hidden]
    float *shared_hidden = nullptr;  // [rows, shared_width]
    float *shared_out = nullptr;     // [rows, hidden]
    // optional [rows, hidden]: the shared down projection runs as two k
    // halves (shared_out + shared_out2) where moe_shared_splits
    float *shared_out2 = nullptr;
};
// Whether the shared down projection can run as two k halves of `inter`
// columns (each a whole number of limb blocks).
__host__ __device__ inline bool moe_shared_splits(int inter, int shared_width) {
    return shared_width == 2 * inter && inter % 128 == 0;
}
int moe_gemm(const MoeGemmParams &p, hipStream_t stream);

// Widest reduction whose int32 sums cannot overflow: a limb and a stored weight
// (q4 on the LDS tiles: 16 times the weight) are at most 128 each.
constexpr int kQgMaxK = 0x7FFFFFFF / (128 * 128) / kQgBK * kQgBK;
// Shapes the MFMA path takes (k a multiple of kQgBK, 16-byte aligned rows).
inline bool qgemm_shape_ok(int fmt, int k) {
    return (fmt == kQ8 || fmt == kQ4) && k > 0 && k <= kQgMaxK && k % kQgBK == 0;
}

}  // namespace mlh
