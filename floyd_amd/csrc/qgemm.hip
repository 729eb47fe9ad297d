// qgemm.hip -- grouped int8-MFMA GEMM for prefill (see qgemm.h for the
// numerics).  gfx950: v_mfma_i32_32x32x32_i8, wave64.
//
// Workgroup: 8 waves in a 4 x 2 arrangement over a 128 (token rows) x 256
// (weight rows) tile; each wave owns 32 x 128 = 1 x 4 MFMA blocks per limb
// (three limbs: 192 int32 accumulators, two waves per SIMD).  Pipeline: k
// slices are 128 wide and copied as stored straight into LDS by buffer loads,
// one in flight while one is multiplied (q4 weights are unpacked as they are
// read); one barrier per slice.
//
// Bound: the copies (the layer without products 457 us, without copies 474, at
// 583 in all for q8 at T = 2048) and the card's power limit (the same launches
// on zero activations: 495 us).  Whole MoE layer on MI355X, T = 2048: q8 655 ->
// 562 us, q4 616 -> 548; T = 600: q8 317 -> 276, q4 275 -> 225; T = 64: q8 161
// -> 159, q4 128 -> 118 (64-wide q8 slices by flat LDS DMA, q4 slices unpacked
// through registers, limb planes and a read-wait-multiply order before).
// MFMA operand layout (measured on gfx950): lane l supplies row (l % 32) and
// the 16-byte k chunk (l / 32) of a 32-wide k step, for A rows and for B
// columns alike; result register r of lane l is
// C[(r / 4) * 8 + (l / 32) * 4 + r % 4][l % 32].
#include "qgemm.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <string>
#include <type_traits>

#include "limb_split.h"

namespace mlh {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr float kQuantMax = 4194304.0f;  // 2^22: |65536 * hi + 256 * mid + lo| bound

// ---------------------------------------------------------------------------
// activation quantisation: one wave per row
// ---------------------------------------------------------------------------

// v * inv rounded to an integer q, |q| <= 2^22, as q = 65536 h + 256 m + l
// with m, l in [-128, 127] and h in [-64, 64]
__device__ __forceinline__ void quant_limbs(float v, float inv, int &h, int &m, int &l) {
    float q = rintf(v * inv);
    q = fminf(fmaxf(q, -kQuantMax), kQuantMax);
    const int qi = (int)q;
    const int t = (qi + 128) >> 8;  // floor: l lands in [-128, 127]
    l = qi - t * 256;
    h = (t + 128) >> 8;
    m = t - h * 256;
}

__device__ __forceinline__ unsigned pack_bytes(int a, int b, int c, int d) {
    return (unsigned)(a & 0xFF) | ((unsigned)(b & 0xFF) << 8) | ((unsigned)(c & 0xFF) << 16) |
           ((unsigned)(d & 0xFF) << 24);
}

// Rows of up to kQuantRegChunks * 256 values stay in registers (one read of
// the row); wider rows (the 11264-wide dense down input) are read per pass.
constexpr int kQuantRegChunks = 16;

// One set of rows to quantise: x (row stride x_stride, optionally
// RMSNorm'ed with norm_w) -> limb blocks at q and scales.
struct QuantSeg {
    const float *x = nullptr;
    long x_stride = 0;
    int rows = 0, width = 0;
    const float *norm_w = nullptr;
    float eps = 0.0f;
    int8_t *q = nullptr;
    float *scale = nullptr;
};

// Row `row` of a segment by one wave.
template <bool REG>
__device__ __forceinline__ void quantize_row(const QuantSeg &s, int row) {
    const float *x = s.x, *norm_w = s.norm_w;
    const int width = s.width;
    const float eps = s.eps;
    float *scale = s.scale;
    const int lane = threadIdx.x & (kWave - 1);
    const float *xr = x + (long)row * s.x_stride;
    const int nchunks = (width / 4 + kWave - 1) / kWave;  // float4 chunks per lane (upper)
    f32x4 v[REG ? kQuantRegChunks : 1];
    if constexpr (REG) {
#pragma unroll
        for (int c = 0; c < kQuantRegChunks; ++c) {
            const int i = (c * kWave + lane) * 4;
            v[c] = (c < nchunks && i < width) ? load_f4(xr + i) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    auto value = [&](int c) -> f32x4 {
        if constexpr (REG) return v[c];
        const int i = (c * kWave + lane) * 4;
        return i < width ? load_f4(xr + i) : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    const int nc = REG ? kQuantRegChunks : nchunks;
    float inv_rms = 1.0f;
    if (norm_w) {
        float ss = 0.0f;
        for (int c = 0; c < nc; ++c) {
            const f32x4 t = value(c);
            ss += t.x * t.x + t.y * t.y + t.z * t.z + t.w * t.w;
        }
        ss = dpp_wave_sum(ss);
        inv_rms = 1.0f / sqrtf(ss / (float)width + eps);
    }
    auto normed = [&](int c) -> f32x4 {
        f32x4 t = value(c);
        const int i = (c * kWave + lane) * 4;
        if (norm_w && i < width) {
            const f32x4 n = load_f4(norm_w + i);
            t.x = t.x * inv_rms * n.x;
            t.y = t.y * inv_rms * n.y;
            t.z = t.z * inv_rms * n.z;
            t.w = t.w * inv_rms * n.w;
        }
        return t;
    };
    float amax = 0.0f;
    for (int c = 0; c < nc; ++c) {
        const f32x4 t = normed(c);
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(t.x), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w))));
    }
    amax = dpp_wave_max(amax);
    const float inv = amax > 0.0f ? kQuantMax / amax : 0.0f;
    if (lane == 0) scale[row] = amax / kQuantMax;
    int8_t *qr = s.q + limb_at(row, 0, width);
    for (int c = 0; c < nc; ++c) {
        const int i = (c * kWave + lane) * 4;
        if (i >= width) continue;
        const f32x4 t = normed(c);
        int h0, h1, h2, h3, m0, m1, m2, m3, l0, l1, l2, l3;
        quant_limbs(t.x, inv, h0, m0, l0);
        quant_limbs(t.y, inv, h1, m1, l1);
        quant_limbs(t.z, inv, h2, m2, l2);
        quant_limbs(t.w, inv, h3, m3, l3);
        int8_t *at = qr + (i >> 7) * (kLimbs * 1024) + (i & 127);
        *reinterpret_cast<unsigned *>(at) = pack_bytes(h0, h1, h2, h3);
        *reinterpret_cast<unsigned *>(at + 1024) = pack_bytes(m0, m1, m2, m3);
        *reinterpret_cast<unsigned *>(at + 2048) = pack_bytes(l0, l1, l2, l3);
    }
}

// Workgroups [0, blocks_a) take 4 rows of segment a each, the rest 4 rows of
// segment b (two segments in one launch).
template <bool REG>
__global__ __launch_bounds__(256) void quantize_act_kernel(QuantSeg a, QuantSeg b, int blocks_a) {
    const bool in_b = (int)blockIdx.x >= blocks_a;
    const QuantSeg s = in_b ? b : a;
    const int row = ((int)blockIdx.x - (in_b ? blocks_a : 0)) * 4 + (int)(threadIdx.x >> 6);
    if (row >= s.rows) return;
    quantize_row<REG>(s, row);
}

static bool quant_seg_ok(const QuantSeg &s) {
    return s.rows == 0 || (s.x && s.q && s.scale && s.rows > 0 && s.width > 0 &&
                           s.width % 4 == 0 && s.x_stride % 4 == 0);
}

static int quantize_segments(const QuantSeg &a, const QuantSeg &b, hipStream_t stream) {
    if (a.rows <= 0 || !quant_seg_ok(a) || !quant_seg_ok(b)) return kErrArgs;
    const int blocks_a = (a.rows + 3) / 4, blocks_b = (b.rows + 3) / 4;
    const bool reg = a.width <= kQuantRegChunks * kWave * 4 &&
                     (b.rows == 0 || b.width <= kQuantRegChunks * kWave * 4);
    if (reg)
        hipLaunchKernelGGL(quantize_act_kernel<true>, dim3(blocks_a + blocks_b), dim3(256), 0,
                           stream, a, b, blocks_a);
    else
        hipLaunchKernelGGL(quantize_act_kernel<false>, dim3(blocks_a + blocks_b), dim3(256), 0,
                           stream, a, b, blocks_a);
    return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int quantize_activations(const float *x, long x_stride, int rows, int width, const float *norm_w,
                         float eps, int8_t *q, float *scale, hipStream_t stream) {
    if (!x || !q || !scale || rows <= 0 || width <= 0) return kErrArgs;
    QuantSeg a;
    a.x = x;
    a.x_stride = x_stride;
    a.rows = rows;
    a.width = width;
    a.norm_w = norm_w;
    a.eps = eps;
    a.q = q;
    a.scale = scale;
    return quantize_segments(a, QuantSeg{}, stream);
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------

// 8 packed nibbles (stored q + 8, column 2j low) -> 8 int8 values in column
// order, q or (TIMES16, two instructions less) 16 q: the nibble in the high
// half of its byte with the offset taken off by an xor.
template <bool TIMES16 = false>
__device__ __forceinline__ void unpack_q4_word(unsigned w, unsigned &out0, unsigned &out1) {
    unsigned lo, hi;  // even and odd columns
    if constexpr (TIMES16) {
        lo = ((w << 4) & 0xF0F0F0F0u) ^ 0x80808080u;
        hi = (w & 0xF0F0F0F0u) ^ 0x80808080u;
    } else {
        lo = w & 0x0F0F0F0Fu;
        hi = (w >> 4) & 0x0F0F0F0Fu;
    }
    // bytes [lo0, hi0, lo1, hi1] and [lo2, hi2, lo3, hi3]
    out0 = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
    out1 = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    if constexpr (!TIMES16) {
        // stored u in [0, 15] -> u - 8 as int8: (u + 0x78) ^ 0x80, no carry between bytes
        out0 = (out0 + 0x78787878u) ^ 0x80808080u;
        out1 = (out1 + 0x78787878u) ^ 0x80808080u;
    }
}

__device__ __forceinline__ int find_task(const int *tile_start, int n, int tile) {
    // last t in [0, n) with tile_start[t] <= tile (tile_start non-decreasing,
    // tile_start[0] = 0): every lane of the wave tests entries lane, lane +
    // 64, ... and the ballots count them -- one round of loads for the first
    // 128 tasks instead of a chain of dependent ones
    const int lane = threadIdx.x & 63;
    const int i0 = lane, i1 = lane + 64;
    const int v0 = tile_start[i0 < n ? i0 : 0];
    const int v1 = tile_start[i1 < n ? i1 : 0];
    int count = __popcll(__ballot(i0 < n && v0 <= tile)) + __popcll(__ballot(i1 < n && v1 <= tile));
    for (int c0 = 128; c0 < n; c0 += 64) {
        const int i = c0 + lane;
        const int v = tile_start[i < n ? i : 0];
        count += __popcll(__ballot(i < n && v <= tile));
    }
    return count - 1;
}

template <bool DUAL, int BM>
__host__ __device__ __forceinline__ int tiles_of(int rows, int n_out) {
    constexpr int outw = DUAL ? kQgBW / 2 : kQgBW;
    return ((rows + BM - 1) / BM) * ((n_out + outw - 1) / outw);
}

// Tile blockIdx.x of a launch -> its task record and the first token row m0
// and output n0 of its BM x 256 tile; false for workgroups past the tiles.
// Tiles run in XCD-contiguous order (workgroup i goes to XCD i % 8): each XCD
// takes a contiguous range of tiles, and within a task groups of kQgGroup row
// tiles share one column tile, so neighbouring workgroups of an XCD reuse
// weight tiles from its L2.  SPLIT: every tile once per share of the reduction,
// all tiles of a share one after the other; tile and share numbers in at.
struct SplitAt {
    int tile = 0, share = 0;
};
template <bool DUAL, int BM, bool SPLIT = false>
__device__ __forceinline__ bool map_tile(const QGemmLaunch &L, GemmTask &tk, int &m0, int &n0,
                                         SplitAt *at = nullptr) {
    int local;
    {
        int begin = 0, end;
        int n_tasks = 1;
        if (L.tasks) {
            const int nr = *L.n_routed;
            n_tasks = nr + L.n_shared;
            end = L.range == 1 ? L.tile_start[nr] : L.tile_start[nr + L.n_shared];
            if (L.range == 2) begin = L.tile_start[nr];
        } else {
            end = tiles_of<DUAL, BM>(L.single.rows, L.single.n_out) * (SPLIT ? L.splits : 1);
        }
        const int total = end - begin;
        const int per = (total + 7) >> 3;
        const int slot = blockIdx.x >> 3;
        if (slot >= per) return false;
        const int tile = begin + (blockIdx.x & 7) * per + slot;
        if (tile >= end) return false;
        if (L.tasks) {
            const int t = find_task(L.tile_start, n_tasks, tile);
            tk = L.tasks[t];
            local = tile - L.tile_start[t];
        } else {
            tk = L.single;
            local = tile;
        }
        if constexpr (SPLIT) {
            const int tiles = end / L.splits;
            at->share = local / tiles;
            at->tile = local -= at->share * tiles;
        }
    }
    constexpr int outw = DUAL ? kQgBW / 2 : kQgBW;
    const int n_tiles = (tk.n_out + outw - 1) / outw;
    const int m_tiles = (tk.rows + BM - 1) / BM;
    const int per_group = kQgGroup * n_tiles;
    const int grp = local / per_group;
    const int gsize = min(kQgGroup, m_tiles - grp * kQgGroup);
    const int rem = local - grp * per_group;
    m0 = (grp * kQgGroup + rem % gsize) * BM;
    n0 = (rem / gsize) * outw;
    return true;
}

// LDS tiles hold one k slice of 128 per stage, as stored: activation rows and
// q8 weight rows of 128 bytes, q4 weight rows of 64 (unpacked as they are
// read), in 16-byte chunks.  Chunk c of row r lives at chunk c ^ g(r):
//   rows of 64 bytes:  g(r) = ((r >> 1) ^ (r >> 3)) & 3
//   rows of 128 bytes: g(r) = (r ^ (r >> 3)) & 7
// so that the MFMA fragment reads (32 consecutive rows, one chunk) and the
// tile writes hit distinct banks whether the LDS serves 8 or 16 lanes of a
// 128-bit access per cycle.
template <int RB>
__device__ __forceinline__ int lds_swizzle(int row) {
    if constexpr (RB == 64) return ((row >> 1) ^ (row >> 3)) & 3;
    else return (row ^ (row >> 3)) & 7;
}

constexpr int kQgSlice = 128;  // k per stage

// Tile shape of a BM-row tile (BM = 128, kQgBMMid = 64 or kQgBMSmall = 32).
// BM = 128: 8 waves (two per SIMD) in a 4 (token rows) x 2 (weight rows) grid,
// each wave 32 x 128 = 4 blocks of 32 x 32 per limb (192 int32 accumulators);
// BM = 64: 8 waves in a 2 x 4 grid, each 32 x 64 = 2 blocks; BM = 32: 4 waves
// side by side, each 32 x 64.  A stage holds
// the three limb tiles of A and the weight tile.  DMA: blocks of 1 KB, wave w
// taking A blocks w, w + kWaves, ... (waves may issue one more than others
// when the count does not divide), B blocks likewise.
template <int FMT, int BM, int LIMBS = kLimbs> struct QgShape {
    static constexpr int kRBB = FMT == kQ8 ? kQgSlice : kQgSlice / 2;  // bytes of a weight row
    static constexpr int kRowsB = 1024 / kRBB;     // weight rows per DMA block
    static constexpr int kRowsA = 8;
    static constexpr int kWaves = BM == 32 ? 4 : 8;
    static constexpr int kThreads = kWaves * kWave;
    static constexpr int kWM = BM / 32;            // waves along the token rows
    static constexpr int kWN = kWaves / kWM;       // waves along the weight rows
    static constexpr int kNF = kQgBW / 32 / kWN;   // 32-row weight blocks per wave
    static constexpr int kStages = FMT == kQ8 && BM == 32 ? 3 : 2;
    static constexpr int kLdsA = LIMBS * BM * kQgSlice;
    static constexpr int kStage = kLdsA + kQgBW * kRBB;
    static constexpr int kLds = kStages * kStage;
    static constexpr int kRowBlocks = BM / kRowsA;
    static constexpr int kAOffs = kRowBlocks > kWaves ? kRowBlocks / kWaves : 1;  // A row blocks per wave
    static constexpr int kABlocks = LIMBS * kRowBlocks;
    static constexpr int kBPer = kQgBW / kRowsB / kWaves;
    static constexpr int kAMax = (kABlocks + kWaves - 1) / kWaves, kAMin = kABlocks / kWaves;
    static constexpr int kDmaMax = kAMax + kBPer, kDmaMin = kAMin + kBPer;
    static_assert(kWaves % kRowBlocks == 0 || kRowBlocks % kWaves == 0, "A row blocks of a wave");
    static_assert(kQgBW / kRowsB % kWaves == 0, "B split");
};
static_assert(QgShape<kQ8, kQgBM>::kLds <= 160 * 1024, "q8 128-row tile exceeds the LDS");
static_assert(QgShape<kQ8, kQgBMMid, 4>::kLds <= 160 * 1024, "q8 four-limb tile exceeds the LDS");
static_assert(QgShape<kQ8, kQgBMSmall>::kLds <= 160 * 1024, "q8 32-row tile exceeds the LDS");
static_assert(2 * QgShape<kQ4, kQgBMSmall>::kLds <= 160 * 1024, "two q4 32-row tiles per CU");

// s_waitcnt on the vector-memory counter only (gfx9 encoding: vmcnt in bits
// 3:0 and 15:14, expcnt 6:4 and lgkmcnt 11:8 left at their no-wait maxima).
template <int N> __device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Buffer of `bytes` from base: loads at offsets of that and more read zero,
// stores there are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *base, long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0,
                                             bytes < 0xFFFFFFFFL ? (unsigned)bytes : 0xFFFFFFFFu, 0x00027000);
}
// 16 bytes per lane from voffset + soffset to consecutive LDS bytes.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t buf, unsigned voffset, int soffset,
                                      __attribute__((address_space(3))) int8_t *dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, dst, 16, voffset, soffset, 0, 0);
}
__device__ __forceinline__ float buffer_load_f32(__amdgpu_buffer_rsrc_t buf, unsigned voffset) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buf, voffset, 0, 0));
}
__device__ __forceinline__ void buffer_store_f32(__amdgpu_buffer_rsrc_t buf, float v, unsigned voffset) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), buf, voffset, 0, 0);
}

// Shares of a split reduction (the library's own memory, static, per GPU:
// launches of one GPU run in order on the library's one stream).  A share is
// the exact integer sum of its tile's limb products, as a double (at most 2^53
// at the four-limb tiles' widths), so the total does not depend on the split.
constexpr int kSplitMaxShares = 256;              // workgroups of a split launch
constexpr int kSplitTile = kQgBMMid * kQgBW;      // outputs of its tiles
constexpr int kSplitCountStride = 32;             // ints between counters (128 bytes)
__device__ double split_part[(long)kSplitMaxShares * kSplitTile];
__device__ int split_count[kSplitMaxShares * kSplitCountStride];  // zero between launches

// Workgroup over a BM x 256 tile (QgShape).  The 32-row tile serves
// batches whose experts hold few rows each: the MFMA work per weight byte is
// a quarter, so the tile is bound by the weight stream instead of by padding.
// SPLIT: over one share of the tile's reduction (whole slices, L.splits shares
// of as equal length as they go); the workgroup that arrives last adds the
// other shares to its own and writes the outputs.
template <int FMT, bool DUAL, int BM, int LIMBS, bool SPLIT>
__global__ __launch_bounds__((QgShape<FMT, BM, LIMBS>::kThreads),
                             (BM != 32 || FMT == kQ8) ? 1 : 2) void qgemm_kernel(QGemmLaunch L) {
    extern __shared__ __attribute__((aligned(16))) int8_t qg_lds[];
    using Sh = QgShape<FMT, BM, LIMBS>;
    constexpr int kRBB = Sh::kRBB;
    constexpr int kStages = Sh::kStages;
    constexpr int kStage = Sh::kStage;
    constexpr int kLdsA = Sh::kLdsA;
    constexpr int kNF = Sh::kNF;
    float *lds_scale = reinterpret_cast<float *>(qg_lds);  // after the products
    GemmTask tk;
    int m0, n0;
    SplitAt at;
    if (!map_tile<DUAL, BM, SPLIT>(L, tk, m0, n0, &at)) return;
    long w_skip = 0;  // bytes of a weight row before the share
    if constexpr (SPLIT) {
        static_assert(!DUAL && BM * kQgBW == kSplitTile, "one sum per output, the shares' layout");
        const int slices = (tk.k + kQgSlice - 1) / kQgSlice;
        const int first = slices * at.share / L.splits, last = slices * (at.share + 1) / L.splits;
        w_skip = (long)first * kRBB;
        tk.w_ld = tk.k;
        tk.w += w_skip;
        tk.a += (long)first * (LIMBS * 1024);
        tk.k = min(tk.k, last * kQgSlice) - first * kQgSlice;
    }

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid >> 6;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    // 8 waves: the two that share a SIMD (waves w and w + 4) take 32-row
    // blocks from different halves of the tile and the same weight rows, so
    // that in a tile whose second half is empty every SIMD still has one wave
    // with products to run.
    constexpr int kHalfM = Sh::kWM == 1 ? 1 : Sh::kWM / 2;  // row blocks of a half
    const int wm = Sh::kWM == 1 ? 0 : wave % kHalfM + (wave >> 2) * kHalfM;
    const int wn = Sh::kWM == 1 ? wave : (wave & 3) / kHalfM;
    static_assert(Sh::kWM == 1 || Sh::kWM * Sh::kWN == 8, "wave grid");
    // a wave whose 32 rows all lie past the task's end skips its products
    // (wave-uniform; it still issues its share of the copies and barriers)
    // (32-row tiles have one wave row: always live, no branch)
    const bool live = Sh::kWM == 1 || __builtin_amdgcn_readfirstlane(m0 + wm * 32) < tk.rows;

    // activation row of tile row r (past the task's end: that of row m0)
    auto arow_of = [&](int r) {
        const int m = m0 + r < tk.rows ? m0 + r : m0;
        return tk.a_rows ? tk.a_rows[m] : tk.a_row0 + m;
    };
    const int w_ld = tk.w_ld ? tk.w_ld : tk.k;
    const long w_row_bytes = FMT == kQ8 ? w_ld : w_ld / 2;
    // the tile's first activation row block and weight row, in 64 bits: the
    // offsets from there fit 32 (gathered rows: moe_gemm_max_rows)
    const int a_first = tk.a_rows ? 0 : (tk.a_row0 + m0) & ~7;
    const int8_t *const a_base = tk.a + limb_at<LIMBS>(a_first, 0, tk.a_width);
    const uint8_t *const w_base = tk.w + n0 * w_row_bytes;
    const uint8_t *const w2_base = DUAL ? tk.w2 + n0 * w_row_bytes : nullptr;
    const long w_bytes = (tk.n_out - n0) * w_row_bytes - w_skip;
    // weight row from n0 held by LDS B row j: SwiGLU tiles give each wave its kNF / 2
    // gate blocks and then the matching up blocks (kNF = 4: blocks f = 0, 1
    // gate, 2, 3 up of a 128-row wave half; kNF = 2: block 0 gate, 1 up of a
    // 64-row wave quarter)
    auto b_out = [&](int j, bool &up) -> int {
        if (!DUAL) {
            up = false;
            return j;
        }
        constexpr int kHalf = kNF / 2;
        const int f = (j >> 5) % kNF;
        up = f >= kHalf;
        return (j / (kNF * 32)) * (kHalf * 32) + (f % kHalf) * 32 + (j & 31);
    };

    // DMA blocks of 1 KB: A block b holds limb b / kRowBlocks of the 8 tile
    // rows 8 (b % kRowBlocks) ..; wave w issues A blocks w, w + kWaves, ...
    // and B blocks likewise (kRowsB weight rows each).  Lane l fills the
    // block's 16 bytes at 16 l: LDS row l / chunks, physical chunk l % chunks,
    // so it loads the logical chunk (l % chunks) ^ g(row).  The limbs share a
    // lane's A rows.  Byte offsets of this lane's A rows; past the task's end
    // outside the buffer (read as zeros):
    constexpr long kABytes = kQgGatherBytes;
    const int alr = lane >> 3, alc = lane & 7;
    unsigned a_off[Sh::kAOffs];
#pragma unroll
    for (int h = 0; h < Sh::kAOffs; ++h) {
        const int r = ((wave + Sh::kWaves * h) % Sh::kRowBlocks) * Sh::kRowsA + alr;
        a_off[h] = m0 + r < tk.rows ? (unsigned)limb_at<LIMBS>(arow_of(r) - a_first, 0, tk.a_width)
                                    : (unsigned)kABytes;
    }
    // one k slice into LDS stage buf (kDmaMin or kDmaMax DMA instructions per
    // wave).  Buffer loads: with a flat LDS DMA in flight the compiler makes
    // every wait for an LDS read a wait for all of them.  Weight rows past
    // the task's last are out of the buffer's range and arrive as zeros.
    auto issue_dma = [&](int ks, int buf) {
        __attribute__((address_space(3))) int8_t *stage =
            (__attribute__((address_space(3))) int8_t *)(qg_lds + buf * kStage);
        const int k0 = ks * kQgSlice;
#pragma unroll
        for (int h = 0; h < Sh::kAMax; ++h) {
            const int b = wave_u + Sh::kWaves * h;  // A block
            if (h >= Sh::kAMin && b >= Sh::kABlocks) break;  // wave-uniform
            const int chunk = alc ^ lds_swizzle<kQgSlice>(b % Sh::kRowBlocks * Sh::kRowsA + alr);
            // a reduction that ends inside the slice: zeros past it (whatever
            // the weights hold there)
            const bool past = k0 + kQgSlice > tk.k && k0 + chunk * 16 >= tk.k;
            dma16(buffer_of(a_base, kABytes),
                  past ? (unsigned)kABytes : a_off[h % Sh::kAOffs] + (unsigned)(chunk * 16),
                  ks * (LIMBS * 1024) + b / Sh::kRowBlocks * 1024, stage + b * 1024);
        }
        constexpr int kCh = kRBB / 16;
#pragma unroll
        for (int q = 0; q < Sh::kBPer; ++q) {
            const int bb = wave_u + Sh::kWaves * q;
            const int j = bb * Sh::kRowsB + lane / kCh;  // B row of this lane
            bool up, u;
            (void)b_out(bb * Sh::kRowsB, up);  // a block's rows are of one matrix
            const int chunk = (lane % kCh) ^ lds_swizzle<kRBB>(j);
            dma16(buffer_of(up ? w2_base : w_base, w_bytes),
                  (unsigned)(b_out(j, u) * w_row_bytes) + (unsigned)(chunk * 16), ks * kRBB,
                  stage + kLdsA + bb * 1024);
        }
    };

    i32x16 acc[LIMBS][kNF];  // [limb][weight-row block]
#pragma unroll
    for (int a = 0; a < LIMBS; ++a)
#pragma unroll
        for (int f = 0; f < kNF; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][f][r] = 0;

    // Fragments of step st (32 columns): lane half h takes 16 of them, q8
    // chunk 2 st + h of both operands; q4 columns 64 (st / 2) + 32 h + 16
    // (st % 2) .., so that a half's packed bytes of two steps are one chunk.
    // LDS byte of this lane's first fragments: steps and blocks differ from
    // it by an xor of the chunk bits (lds_swizzle; 32 rows on flip the top
    // bit of a 128-byte row's swizzle) and by constants, computed where used:
    // kept over the loop they would spill
    const int frow = lane & 31;
    const int half = lane >> 5;
    const int arow_lds = wm * 32 + frow, brow_lds = wn * (kNF * 32) + frow;
    const int a_frag =
        arow_lds * kQgSlice + (((FMT == kQ8 ? half : 2 * half) ^ lds_swizzle<kQgSlice>(arow_lds)) << 4);
    const int b_frag = kLdsA + brow_lds * kRBB + ((half ^ lds_swizzle<kRBB>(brow_lds)) << 4);
    using BRaw = typename std::conditional<FMT == kQ8, i32x4, u32x2>::type;
    // Slices ks + 1 .. ks + kStages - 1 stream into LDS while slice ks is
    // multiplied.  A wave's DMA completes in order, its kDmaMax or kDmaMin
    // instructions per slice, so a slice has landed when at most that many for
    // each later slice in flight remain; the barrier after the wait makes
    // every wave's part visible and frees the stage of the slice before it.
    // (A bare barrier: __syncthreads() would also wait for the loads of the
    // fence it implies.)
    static_assert(kStages == 2 || kStages == 3, "waits below");
    const bool more = Sh::kDmaMax == Sh::kDmaMin || wave_u + Sh::kWaves * Sh::kAMin < Sh::kABlocks;
    const int nk = (tk.k + kQgSlice - 1) / kQgSlice;
    // slice ks has landed for every wave, and the stage of slice ks - 1 is
    // free: it takes slice ks + kStages - 1
    auto next_slice = [&](int ks) {
        if (kStages == 3 && ks + 1 < nk) {
            if (more) wait_vmcnt<Sh::kDmaMax>();
            else wait_vmcnt<Sh::kDmaMin>();
        } else {
            wait_vmcnt<0>();
        }
        __builtin_amdgcn_s_barrier();
        if (ks + kStages - 1 < nk) issue_dma(ks + kStages - 1, (ks + kStages - 1) % kStages);
    };
    // Fragments are read ahead of their products, the weights by two blocks
    // and the activations by a step.  The sched_barriers keep the order: left
    // to itself the compiler reads a block, waits for it and multiplies it,
    // because the accumulators leave it few registers.  (Reading ahead across
    // slices too, the barrier two blocks before a slice's end: the T = 2048 q8
    // MoE layer 568 against 557 us.)
    constexpr int kSteps = kQgSlice / 32, kBlocks = kSteps * kNF;
    static_assert(kBlocks % 4 == 0 && kSteps == 4, "register rings, chunk bits");
    i32x4 fa[2][LIMBS];
    BRaw fb[4];
    auto read_a = [&](int base, int st, int a) {
        const int bits = FMT == kQ8 ? st << 5 : ((st & 1) << 4) | ((st >> 1) << 6);
        fa[st & 1][a] = *reinterpret_cast<const i32x4 *>(qg_lds + ((base + a_frag) ^ bits) +
                                                         a * (BM * kQgSlice));
    };
    auto read_b = [&](int base, int i) {
        const int st = i / kNF, f = i % kNF;
        const int bits = FMT == kQ8 ? (st << 5) ^ ((f & 1) << 6) : ((st >> 1) << 5) | ((st & 1) << 3);
        fb[i % 4] = *reinterpret_cast<const BRaw *>(qg_lds + ((base + b_frag) ^ bits) + f * 32 * kRBB);
    };
    auto weights = [&](const BRaw &d) -> i32x4 {
        if constexpr (FMT == kQ8) {
            return d;
        } else {
            unsigned o0, o1, o2, o3;
            unpack_q4_word<true>(d.x, o0, o1);
            unpack_q4_word<true>(d.y, o2, o3);
            return i32x4{(int)o0, (int)o1, (int)o2, (int)o3};
        }
    };
    for (int st = 0; st < kStages - 1 && st < nk; ++st) issue_dma(st, st);
    next_slice(0);
    if (live) {
        int base = 0;
        for (int ks = 0; ks < nk; ++ks) {
            if (ks) next_slice(ks);
            asm("" : "+s"(base));  // (see a_frag)
#pragma unroll
            for (int a = 0; a < LIMBS; ++a) read_a(base, 0, a);
            read_b(base, 0);
            read_b(base, 1);
#pragma unroll
            for (int i = 0; i < kBlocks; ++i) {
                const int st = i / kNF, f = i % kNF;
                if (i + 2 < kBlocks) read_b(base, i + 2);
                if (st + 1 < kSteps) {
                    constexpr int per = (LIMBS + kNF - 1) / kNF;
#pragma unroll
                    for (int a = f * per; a < (f + 1) * per && a < LIMBS; ++a) read_a(base, st + 1, a);
                }
                __builtin_amdgcn_sched_barrier(0);
                const i32x4 w = weights(fb[i % 4]);
#pragma unroll
                for (int a = 0; a < LIMBS; ++a)
                    acc[a][f] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[st & 1][a], w, acc[a][f], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            base = (ks + 1) % kStages * kStage;
        }
    } else {
        for (int ks = 1; ks < nk; ++ks) next_slice(ks);
    }

    // ---- shares: stored, and added by the tile's last workgroup
    double total[SPLIT ? kNF : 1][16];
    if constexpr (SPLIT) {
        constexpr int kShift = FMT == kQ4 ? 4 : 0;
#pragma unroll
        for (int f = 0; f < kNF; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                double v = acc[0][f][r] >> kShift;
#pragma unroll
                for (int a = 1; a < LIMBS; ++a) v = fma(v, 256.0, (double)(acc[a][f][r] >> kShift));
                total[f][r] = v;
            }
        auto part_of = [&](int share) {
            return split_part + (long)(at.tile * L.splits + share) * kSplitTile + tid;
        };
        if (live) {
            double *part = part_of(at.share);
#pragma unroll
            for (int f = 0; f < kNF; ++f)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    __hip_atomic_store(part + (f * 16 + r) * Sh::kThreads, total[f][r], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        }
        int *count = split_count + at.tile * kSplitCountStride;
        if (!agent_handoff_arrive(count, L.splits)) return;
        if (tid == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (live) {
            for (int share = 0; share < L.splits; ++share) {
                if (share == at.share) continue;
                const double *part = part_of(share);
                double v[kNF * 16];
#pragma unroll
                for (int i = 0; i < kNF * 16; ++i)
                    v[i] = __hip_atomic_load(part + i * Sh::kThreads, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int i = 0; i < kNF * 16; ++i) total[i / 16][i % 16] += v[i];
            }
        }
    }

    // ---- epilogue, without a branch: stores and residual loads go through
    // buffers of the tile's own rows, so rows past the task's end are out of
    // range (dropped, read as zero), as are the columns past n_out, whose
    // offset is set there.  Weight scales and residual rows are loaded before
    // the stores they precede: a wait for a load after a store waits for both.
    constexpr int kF = DUAL ? kNF / 2 : kNF;
    constexpr unsigned kOutside = (unsigned)kQgOutside;
    const int rows_here = min(tk.rows - m0, BM);
    float sw[kF], su[kF];
    unsigned ycol[kF], rcol[kF];
    const auto s_buf = buffer_of(tk.s, (long)tk.n_out * 4);
    const auto s2_buf = buffer_of(DUAL ? tk.s2 : tk.s, (long)tk.n_out * 4);
    const auto y_buf = buffer_of(tk.y + (long)m0 * tk.y_stride, (long)rows_here * tk.y_stride * 4);
    const int lane_row = wm * 32 + half * 4;  // + 8 (r / 4) + r % 4: row of result register r
#pragma unroll
    for (int f = 0; f < kF; ++f) {
        const int n = n0 + wn * kF * 32 + f * 32 + frow;
        sw[f] = buffer_load_f32(s_buf, n * 4);
        su[f] = DUAL ? buffer_load_f32(s2_buf, n * 4) : 0.0f;
        ycol[f] = n < tk.n_out ? (unsigned)(lane_row * tk.y_stride + n) * 4 : kOutside;
        rcol[f] = n < tk.n_out ? (unsigned)(lane_row * tk.resid_stride + n) * 4 : kOutside;
    }
    // every wave has read its last fragments: the LDS takes the row scales
    __syncthreads();
    if (tid < BM) lds_scale[tid] = tid < rows_here ? tk.a_scale[arow_of(tid)] : 0.0f;
    __syncthreads();
    // the limbs' sum of one result register, 256 apart (the int32 sums are
    // exact; q4 ones are 16 times the products')
    auto limb_sum = [&](int f, int r) -> float {
        if constexpr (SPLIT) return (float)total[f][r];
        constexpr int kShift = FMT == kQ4 ? 4 : 0;
        float v = (float)(acc[LIMBS - 1][f][r] >> kShift), unit = 1.0f;
#pragma unroll
        for (int a = LIMBS - 2; a >= 0; --a) {
            unit *= 256.0f;
            v = fmaf((float)(acc[a][f][r] >> kShift), unit, v);
        }
        return v;
    };
    auto epilogue = [&](auto with_resid) {
        constexpr bool kResid = decltype(with_resid)::value;
        const auto r_buf = buffer_of(kResid ? tk.resid + (long)m0 * tk.resid_stride : tk.y,
                                     (long)rows_here * tk.resid_stride * 4);
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            const f32x4 sx = *reinterpret_cast<const f32x4 *>(lds_scale + lane_row + 8 * rg);
            float res[4][kF];
            if (kResid) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int f = 0; f < kF; ++f)
                        res[q][f] = buffer_load_f32(
                            r_buf, rcol[f] + (unsigned)((8 * rg + q) * tk.resid_stride * 4));
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = 4 * rg + q;
                const float s = q == 0 ? sx.x : q == 1 ? sx.y : q == 2 ? sx.z : sx.w;
                const unsigned row = (unsigned)((8 * rg + q) * tk.y_stride * 4);
#pragma unroll
                for (int f = 0; f < kF; ++f) {
                    float v = limb_sum(f, r) * s * sw[f];
                    // in this order: g u may leave fp32's range where silu(g) u does not
                    if (DUAL) v = silu(v) * (limb_sum(f + kF, r) * s * su[f]);
                    if (kResid) v = res[q][f] + v;
                    buffer_store_f32(y_buf, v, ycol[f] + row);
                }
            }
        }
    };
    if (!DUAL && tk.resid) epilogue(std::true_type{});
    else epilogue(std::false_type{});
}

// ---------------------------------------------------------------------------
// Weight-streaming tile (launches whose tasks hold few token rows, e.g. the
// MoE layer of a decode batch): BM = 16 * MB token rows x 256 weight rows per
// workgroup, each of its 4 waves owning 64 weight rows (4 blocks of 16) for
// all BM rows, with no barrier.  Weights, read once, are the stream: a wave
// copies its rows into a private LDS ring by DMA, 128 contiguous bytes of a
// row per lane group (a DMA instruction covers 8 rows x 128 bytes: on MI355X
// a plain read of such runs moves ~6 TB/s, of the 64-byte pieces an MFMA
// fragment holds ~4.2 TB/s), kStages steps of 128 k ahead; the activation
// limbs of the BM rows (L2-resident, shared by every tile of the task) load
// straight into registers.  Products on v_mfma_i32_16x16x64_i8: lane l
// supplies row / column l % 16 and the 16 k values 16 (l / 16) .. + 15 of a
// 64-wide step, for activations (A) and weights (B) alike; result register r
// of lane l is C[4 (l / 16) + r][l % 16].
// ---------------------------------------------------------------------------

template <int FMT, int MB> struct QsShape {
    static constexpr int kBM = 16 * MB;
    static constexpr int kStages = 2;                  // 128-k steps in flight
    static constexpr int kRowBytes = FMT == kQ8 ? 128 : 64;  // weight bytes per row and step
    static constexpr int kWaveStage = 64 * kRowBytes;        // one wave's rows per step
    static constexpr int kLds = 4 * kStages * kWaveStage;
    // per lane and step: weight DMA (64 rows of kRowBytes, 1 KB per
    // instruction) + activation loads (2 slices x 3 limbs x MB row blocks)
    static constexpr int kDma = kWaveStage / 1024;
    static constexpr int kLoads = kDma + 2 * kLimbs * MB;
    static_assert((kStages - 1) * kLoads <= 63, "vmcnt range");
};

template <int FMT, bool DUAL, int MB>
__global__ __launch_bounds__(256, 2) void qgemm_stream_kernel(QGemmLaunch L) {
    using Sh = QsShape<FMT, MB>;
    constexpr int BM = Sh::kBM;
    constexpr int S = Sh::kStages;
    constexpr int NL = Sh::kLoads;
    constexpr int RB = Sh::kRowBytes;
    extern __shared__ __attribute__((aligned(16))) unsigned char qs_lds[];
    GemmTask tk;
    int m0, n0;
    if (!map_tile<DUAL, BM>(L, tk, m0, n0)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int l16 = lane & 15, kq = lane >> 4;
    unsigned char *my_lds = qs_lds + wave * S * Sh::kWaveStage;

    // activation rows of this lane (A row l16 of each row block); rows past
    // the task's end read its first row (their results are never stored)
    const int8_t *a_src[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = m0 + 16 * i + l16;
        const int mm = m < tk.rows ? m : m0;
        const int arow = tk.a_rows ? tk.a_rows[mm] : tk.a_row0 + mm;
        a_src[i] = tk.a + limb_at(arow, 0, tk.a_width) + 16 * kq;
    }
    // weight row of LDS row j (0..63) of this wave: SwiGLU tiles give a wave
    // 32 gate rows (LDS rows 0..31) and the matching 32 up rows (32..63)
    const int w_ld = tk.w_ld ? tk.w_ld : tk.k;
    const long w_row_bytes = FMT == kQ8 ? w_ld : w_ld / 2;
    auto w_row = [&](int j, int &n) -> const uint8_t * {
        const uint8_t *base = tk.w;
        if (DUAL) {
            n = n0 + wave * 32 + (j & 31);
            if (j >= 32) base = tk.w2;
        } else {
            n = n0 + wave * 64 + j;
        }
        const int nn = n < tk.n_out ? n : 0;
        return base + (long)nn * w_row_bytes;
    };
    // DMA lane roles: instruction d covers LDS rows 8 d .. 8 d + 7 (q8) or
    // 16 d .. 16 d + 15 (q4), lane l row (l / (RB / 16)), physical 16-byte
    // chunk l % (RB / 16), which holds the row's logical chunk
    // (l % (RB / 16)) ^ (row & 7) (q8; q4 rows of 4 chunks XOR row & 3)
    constexpr int kChunks = RB / 16;
    constexpr int kRowsPerDma = 64 / kChunks;
    const uint8_t *dma_src[Sh::kDma];
#pragma unroll
    for (int d = 0; d < Sh::kDma; ++d) {
        const int j = d * kRowsPerDma + lane / kChunks;
        int n;
        const uint8_t *row = w_row(j, n);
        const int logical = (lane % kChunks) ^ (j & (kChunks - 1));
        dma_src[d] = row + logical * 16;
    }
    const int nk = tk.k / 64;
    i32x4 ra[S][2][kLimbs][MB];
    auto issue = [&](int step, int st) {
        __attribute__((address_space(3))) unsigned char *dst =
            (__attribute__((address_space(3))) unsigned char *)(my_lds + st * Sh::kWaveStage);
        const long koff = (long)step * RB;
#pragma unroll
        for (int d = 0; d < Sh::kDma; ++d)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void *)(dma_src[d] + koff),
                dst + d * 1024, 16, 0, 0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int slice = min(2 * step + h, nk - 1);
#pragma unroll
            for (int a = 0; a < kLimbs; ++a)
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    const u32x4 v =
                        load_global16(a_src[i] + (slice >> 1) * (kLimbs * 1024) + a * 1024 + (slice & 1) * 64);
                    ra[st][h][a][i] = i32x4{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
                }
        }
    };
    i32x4 acc[kLimbs][MB][4];
#pragma unroll
    for (int a = 0; a < kLimbs; ++a)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int f = 0; f < 4; ++f) acc[a][i][f] = i32x4{0, 0, 0, 0};
    // the two 64-wide slices of a step (nh = 1: only the first exists)
    auto compute = [&](int st, int nh) {
        const unsigned char *stage = my_lds + st * Sh::kWaveStage;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h >= nh) break;  // uniform
            i32x4 bw[4];
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const int j = f * 16 + l16;
                if constexpr (FMT == kQ8) {
                    const int phys = (h * 4 + kq) ^ (j & 7);
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + j * RB + phys * 16);
                    bw[f] = i32x4{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
                } else {
                    // 8 packed bytes = the 16 k values of this lane
                    const int phys = (h * 2 + (kq >> 1)) ^ (j & 3);
                    const u32x2 v = *reinterpret_cast<const u32x2 *>(stage + j * RB + phys * 16 +
                                                                    (kq & 1) * 8);
                    unsigned o0, o1, o2, o3;
                    unpack_q4_word(v.x, o0, o1);
                    unpack_q4_word(v.y, o2, o3);
                    bw[f] = i32x4{(int)o0, (int)o1, (int)o2, (int)o3};
                }
            }
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int a = 0; a < kLimbs; ++a)
                        acc[a][i][f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            ra[st][h][a][i], bw[f], acc[a][i][f], 0, 0, 0);
        }
    };
    const int steps = (nk + 1) / 2;  // the last step may hold one slice
#pragma unroll
    for (int j = 0; j < S; ++j)
        if (j < steps) issue(j, j);
    for (int t0 = 0; t0 < steps; t0 += S) {
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const int t = t0 + j;
            if (t < steps) {  // uniform
                if (t + S - 1 < steps) wait_vmcnt<(S - 1) * NL>();
                else wait_vmcnt<0>();
                compute(j, min(2, nk - 2 * t));
                if (t + S < steps) issue(t + S, j);
            }
        }
    }

    // ---- epilogue: lane l holds C[4 (l / 16) + r][l % 16] of each block
    constexpr int kF = DUAL ? 2 : 4;
    int ncol[kF];
    float sw[kF], su[kF];
#pragma unroll
    for (int f = 0; f < kF; ++f) {
        w_row(f * 16 + l16, ncol[f]);
        const bool ok = ncol[f] < tk.n_out;
        sw[f] = ok ? load_global_f32(tk.s + ncol[f]) : 0.0f;
        su[f] = (DUAL && ok) ? load_global_f32(tk.s2 + ncol[f]) : 0.0f;
    }
    float sx[MB][4];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * kq + r;
            const int mm = m < tk.rows ? m : m0;
            sx[i][r] = load_global_f32(tk.a_scale + (tk.a_rows ? tk.a_rows[mm] : tk.a_row0 + mm));
        }
    __builtin_amdgcn_s_waitcnt(0);
    auto limb_sum = [&](int i, int f, int r) -> float {
        return (float)acc[0][i][f][r] * 65536.0f +
               ((float)acc[1][i][f][r] * 256.0f + (float)acc[2][i][f][r]);
    };
    const bool resid = !DUAL && tk.resid;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * kq + r;
            if (m >= tk.rows) continue;
            float *yrow = tk.y + (long)m * tk.y_stride;
#pragma unroll
            for (int f = 0; f < kF; ++f) {
                if (ncol[f] >= tk.n_out) continue;
                if (DUAL) {
                    const float g = limb_sum(i, f, r) * sx[i][r] * sw[f];
                    const float u = limb_sum(i, f + 2, r) * sx[i][r] * su[f];
                    store_global(yrow + ncol[f], silu(g) * u);
                } else {
                    float v = limb_sum(i, f, r) * sx[i][r] * sw[f];
                    if (resid)
                        v = load_global_f32(tk.resid + (long)m * tk.resid_stride + ncol[f]) + v;
                    store_global(yrow + ncol[f], v);
                }
            }
        }
}

template <int FMT, bool DUAL, int BM, int LIMBS = kLimbs, bool SPLIT = false>
static void launch_qgemm(const QGemmLaunch &L, int grid, hipStream_t stream) {
    using Sh = QgShape<FMT, BM, LIMBS>;
    static const bool attr = [] {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(&qgemm_kernel<FMT, DUAL, BM, LIMBS, SPLIT>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                   Sh::kLds) == hipSuccess;
    }();
    (void)attr;
    hipLaunchKernelGGL((qgemm_kernel<FMT, DUAL, BM, LIMBS, SPLIT>), dim3((unsigned)grid), dim3(Sh::kThreads),
                       Sh::kLds, stream, L);
}

template <int BM, int LIMBS = kLimbs>
static void launch_qgemm_bm(int fmt, bool dual, const QGemmLaunch &L, int grid,
                            hipStream_t stream) {
    if (fmt == kQ8) {
        if (dual) launch_qgemm<kQ8, true, BM, LIMBS>(L, grid, stream);
        else launch_qgemm<kQ8, false, BM, LIMBS>(L, grid, stream);
    } else {
        if (dual) launch_qgemm<kQ4, true, BM, LIMBS>(L, grid, stream);
        else launch_qgemm<kQ4, false, BM, LIMBS>(L, grid, stream);
    }
}

template <int FMT, bool DUAL, int MB>
static void launch_stream(const QGemmLaunch &L, int grid, hipStream_t stream) {
    constexpr int kLds = QsShape<FMT, MB>::kLds;
    static const bool attr = [] {
        return hipFuncSetAttribute(
                   reinterpret_cast<const void *>(&qgemm_stream_kernel<FMT, DUAL, MB>),
                   hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess;
    }();
    (void)attr;
    hipLaunchKernelGGL((qgemm_stream_kernel<FMT, DUAL, MB>), dim3((unsigned)grid), dim3(256),
                       kLds, stream, L);
}

template <int MB>
static void launch_stream_mb(int fmt, bool dual, const QGemmLaunch &L, int grid,
                             hipStream_t stream) {
    if (fmt == kQ8) {
        if (dual) launch_stream<kQ8, true, MB>(L, grid, stream);
        else launch_stream<kQ8, false, MB>(L, grid, stream);
    } else {
        if (dual) launch_stream<kQ4, true, MB>(L, grid, stream);
        else launch_stream<kQ4, false, MB>(L, grid, stream);
    }
}

// Tile choices, measured on MI355X.  A batch of at most 16 token rows streams
// the weights (every task fits one row tile); the streaming tile needs
// reductions that are whole multiples of 128 (`k128`).
// MoE layer: 16-row streaming tile up to 16 rows (T = 8: 99 against 108 us
// on the 32-row LDS tile), then by the average rows per expert.  q8: the
// 32-row tile up to 32 (T = 256: 212 us, 64-row 221, 128-row 229), the 64-row
// tile, which copies the weights once where that takes two, up to 64 (T = 600:
// 304, 278, 297), 128 rows above (T = 1400: 570, 471, 446).  q4: two 32-row
// workgroups share a CU and win up to 140 (T = 600: 228, 250, 294; T = 1400:
// 419, 430, 435; T = 2048: 572, 586, 557).
static int moe_tile(int fmt, int rows, double rows_per_expert, bool k128) {
    if (k128 && rows <= 16) return kTileStream16;
    if (fmt == kQ4) return rows_per_expert <= 140.0 ? kTileLds32 : kTileLds128;
    return rows_per_expert <= 32.0 ? kTileLds32 : rows_per_expert <= 64.0 ? kTileLds64 : kTileLds128;
}

static int launch_qgemm_fmt(int fmt, bool dual, int kind, const QGemmLaunch &L, int tiles_bound,
                            hipStream_t stream) {
    if (tiles_bound <= 0) return kOk;
    if (fmt != kQ8 && fmt != kQ4) return kErrArgs;
    const int grid = ((tiles_bound + 7) / 8) * 8;
    switch (kind) {
    case kTileStream16: launch_stream_mb<1>(fmt, dual, L, grid, stream); break;
    case kTileLds32: launch_qgemm_bm<kQgBMSmall>(fmt, dual, L, grid, stream); break;
    case kTileLds64: launch_qgemm_bm<kQgBMMid>(fmt, dual, L, grid, stream); break;
    case kTileLds128: launch_qgemm_bm<kQgBM>(fmt, dual, L, grid, stream); break;
    default: return kErrArgs;
    }
    return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int qgemm_single(int fmt, bool dual, const GemmTask &task, hipStream_t stream) {
    if (!qgemm_shape_ok(fmt, task.k) || task.rows <= 0 || task.n_out <= 0 || !task.w ||
        !task.s || !task.a || task.a_width < task.k || !task.a_scale || !task.y ||
        task.y_stride > kQgMaxStride || (task.resid && task.resid_stride > kQgMaxStride) ||
        (dual && (!task.w2 || !task.s2)))
        return kErrArgs;
    QGemmLaunch L;
    L.single = task;
    const int kind = dense_tile(task.rows, task.k % 128 == 0, task.n_out, dual);
    return launch_qgemm_fmt(fmt, dual, kind, L,
                            host_tiles(dual, task.rows, task.n_out, tile_bm(kind)), stream);
}

// ---------------------------------------------------------------------------
// gemv() of many token rows
// ---------------------------------------------------------------------------

// Limb blocks and scales of one call's token rows: the library's own memory,
// static, per GPU.  Launches of one GPU run in order on the library's one
// stream, and a call's launches are queued under a lock, so no other call's
// come between them; wider batches run in row chunks.  (No allocation: a call
// may be captured.)
constexpr int kTilesMaxWidth = 65536;  // the shares' doubles are exact to here
static_assert(kTilesMaxWidth <= kQgMaxK, "int32 sums");
__device__ int8_t tiles_limbs[kTilesBytes];
__device__ float tiles_scale[kTilesRows];
static std::mutex tiles_mutex;

// Four limbs of one row (x, or x * norm_w), a workgroup per row: step and split
// as in gemv_batch.hip, over the whole row; the row's scale is the step times
// 1 / rms, NaN where the row holds a NaN or an infinity.
__global__ __launch_bounds__(256) void quantize4_kernel(const float *x, long x_stride, int width,
                                                        const float *norm_w, float eps) {
    __shared__ float red[2][4];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *xr = x + (long)row * x_stride;
    float amax = 0.0f, ss = 0.0f;
    auto load = [&](int i, float (&v)[4]) {
        const f32x4 a = load_f4(xr + i);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    };
    auto weigh = [&](int i, float (&v)[4]) {
        if (!norm_w) return;
        const f32x4 n = load_f4(norm_w + i);
        v[0] *= n.x, v[1] *= n.y, v[2] *= n.z, v[3] *= n.w;
    };
    for (int i = tid * 4; i < width; i += 1024) {
        float v[4];
        load(i, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(v[e], v[e], ss);
        weigh(i, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) amax = __builtin_elementwise_maximum(amax, __builtin_fabsf(v[e]));
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        amax = __builtin_elementwise_maximum(amax, __shfl_xor(amax, o));
        ss += __shfl_xor(ss, o);
    }
    if (lane == 0) red[0][wave] = amax, red[1][wave] = ss;
    __syncthreads();
    amax = __builtin_elementwise_maximum(__builtin_elementwise_maximum(red[0][0], red[0][1]),
                                         __builtin_elementwise_maximum(red[0][2], red[0][3]));
    const unsigned bits = __float_as_uint(amax) & 0x7FFFFFFFu;
    const int ex = min(156 - (int)(bits >> 23), 126);  // amax 2^ex < 2^30
    const float step_inv = __uint_as_float((unsigned)(127 + ex) << 23);
    if (tid == 0) {
        const float step = bits >= 0x7F800000u ? __builtin_nanf("")
                                               : __uint_as_float((unsigned)(127 - ex) << 23);
        const float tot = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
        tiles_scale[row] = norm_w ? step * (1.0f / sqrtf(tot / (float)width + eps)) : step;
    }
    int8_t *q = tiles_limbs + limb_at<4>(row, 0, width);
    for (int i = tid * 4; i < width; i += 1024) {
        float v[4];
        load(i, v);
        weigh(i, v);
        unsigned l[4];
        split_limbs4(v, step_inv, l[0], l[1], l[2], l[3]);
#pragma unroll
        for (int L = 0; L < 4; ++L)
            *reinterpret_cast<unsigned *>(q + (i >> 7) * 4096 + L * 1024 + (i & 127)) = l[L];
    }
}

// Shares of the reduction: as many as keep the launch in one round of the CUs
// (a 2048-row matrix has 8 tiles per 64 token rows), none shorter than
// kSplitMinSlices slices (2048 columns), where storing and adding the shares (128
// KB each) costs as much as it saves.  2048 x 11264 at 777 rows (104 tiles,
// 2 shares) 139 -> 96 us, at 330 rows (48 tiles, 5 shares) 120 -> 60.
constexpr int kSplitMinSlices = 16;
static int tile_splits(const GemvParams &p, long rows) {
    if (p.epilogue == kEpiSiluDual) return 1;
    const long tiles = host_tiles(false, (int)rows, p.O, kQgBMMid);
    const long fit = kSplitMaxShares / tiles, slices = (p.I + kQgSlice - 1) / kQgSlice;
    return (int)std::max<long>(1, std::min<long>(fit, slices / kSplitMinSlices));
}

bool gemv_tiles(const GemvParams &p, hipStream_t stream, std::string *name) {
    const bool dual = p.epilogue == kEpiSiluDual;
    auto al = [](const void *v) { return ((uintptr_t)v & 15u) == 0; };
    if (!qgemm_shape_ok(p.fmt, p.I) || p.I > kTilesMaxWidth || p.router_parts || !al(p.w) ||
        (dual && !al(p.w2)) || !al(p.x) || p.x_stride % 4 || (p.norm_w && !al(p.norm_w)) ||
        p.y_stride > kQgMaxStride || (p.resid && p.resid_stride > kQgMaxStride))
        return false;
    if (name) {
        char buf[64];
        snprintf(buf, sizeof(buf), "mlh::qgemm_kernel<%d, %s, %d, 4, %s>", p.fmt,
                 dual ? "true" : "false", kQgBMMid, tile_splits(p, tiles_chunk(p.rows, p.I)) > 1 ? "true" : "false");
        *name = buf;
        return true;
    }
    static int8_t *limbs[64] = {};  // device addresses, looked up once per GPU
    static float *scale[64] = {};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return false;
    const std::lock_guard<std::mutex> lock(tiles_mutex);
    if (!limbs[device] &&
        (hipGetSymbolAddress((void **)&scale[device], HIP_SYMBOL(tiles_scale)) != hipSuccess ||
         hipGetSymbolAddress((void **)&limbs[device], HIP_SYMBOL(tiles_limbs)) != hipSuccess)) {
        (void)hipGetLastError();  // not sticky: the caller falls back
        return false;
    }
    const long chunk = tiles_chunk(p.rows, p.I);
    for (long r0 = 0; r0 < p.rows; r0 += chunk) {
        const int n = (int)std::min<long>(chunk, p.rows - r0);
        hipLaunchKernelGGL(quantize4_kernel, dim3(n), dim3(256), 0, stream, p.x + r0 * p.x_stride,
                           p.x_stride, p.I, p.norm_w, p.eps);
        QGemmLaunch L;
        GemmTask &t = L.single;
        t.w = p.w;
        t.s = p.s;
        t.w2 = p.w2;
        t.s2 = p.s2;
        t.rows = n;
        t.n_out = p.O;
        t.k = p.I;
        t.a = limbs[device];
        t.a_width = p.I;
        t.a_scale = scale[device];
        t.y = p.y + r0 * p.y_stride;
        t.y_stride = p.y_stride;
        if (p.epilogue == kEpiResidual) {
            t.resid = p.resid + r0 * p.resid_stride;
            t.resid_stride = p.resid_stride;
        }
        L.splits = tile_splits(p, n);
        const int grid = (host_tiles(dual, n, p.O, kQgBMMid) * L.splits + 7) / 8 * 8;
        if (L.splits == 1) launch_qgemm_bm<kQgBMMid, 4>(p.fmt, dual, L, grid, stream);
        else if (p.fmt == kQ8) launch_qgemm<kQ8, false, kQgBMMid, 4, true>(L, grid, stream);
        else launch_qgemm<kQ4, false, kQgBMMid, 4, true>(L, grid, stream);
    }
    return true;
}

// ---------------------------------------------------------------------------
// MoE prefill: device-built task tables
// ---------------------------------------------------------------------------

struct MoeScheduleParams {
    MoeGemmParams p;
    int bm;  // token rows per tile of the launches that read the tables
};

// Tasks of the shared down projection: 2 k halves where they can be and a
// second output exists, else 1.
__host__ __device__ inline int moe_shared_down_parts(const MoeGemmParams &p) {
    return p.has_shared && p.shared_out2 && moe_shared_splits(p.inter, p.shared_width) ? 2 : 1;
}

// With L (routing in the same workgroup) the route tables and the expert
// table (ew_lds, [experts]) come from LDS instead of global memory.  Called
// by whole workgroups of at least two waves.
__device__ __forceinline__ void moe_schedule_body(const MoeScheduleParams &sp,
                                                  const RouteLds *L = nullptr,
                                                  const ExpertWeights *ew_lds = nullptr) {
    const MoeGemmParams &p = sp.p;
    const int bm = sp.bm;
    auto tiles_rt = [bm](bool dual, int rows, int n_out) {
        const int outw = dual ? kQgBW / 2 : kQgBW;
        return ((rows + bm - 1) / bm) * ((n_out + outw - 1) / outw);
    };
    __shared__ int tiles[2][kQgMaxTasks];
    const int nr = L ? L->unique_total : *p.n_unique;
    GemmTask *t0 = p.tasks;
    GemmTask *t1 = p.tasks + kQgMaxTasks;
    for (int u = threadIdx.x; u < nr; u += blockDim.x) {
        const int e = L ? L->unique[u] : p.unique[u];
        const int cnt = L ? L->counts[e] : p.counts[e], off = L ? L->offsets[e] : p.offsets[e];
        const ExpertWeights ew = ew_lds ? ew_lds[e] : p.expert_table[e];
        GemmTask a;
        a.w = ew.gate;
        a.w2 = ew.up;
        a.s = ew.gate_s;
        a.s2 = ew.up_s;
        a.rows = cnt;
        a.n_out = p.inter;
        a.k = p.hidden;
        a.a = p.xq;
        a.a_scale = p.xq_scale;
        a.a_width = p.hidden;
        a.a_rows = p.list_rows + off;
        a.y = p.expert_hidden + (long)off * p.inter;
        a.y_stride = p.inter;
        t0[u] = a;
        tiles[0][u] = tiles_rt(true, cnt, p.inter);
        GemmTask b;
        b.w = ew.down;
        b.s = ew.down_s;
        b.rows = cnt;
        b.n_out = p.hidden;
        b.k = p.inter;
        b.a = p.hq;
        b.a_scale = p.hq_scale;
        b.a_width = p.inter;
        b.a_row0 = off;
        b.y = p.expert_out + (long)off * p.hidden;
        b.y_stride = p.hidden;
        t1[u] = b;
        tiles[1][u] = tiles_rt(false, cnt, p.hidden);
    }
    const int nsd = moe_shared_down_parts(p);  // shared down tasks (k parts)
    if (threadIdx.x == 0) {
        tiles[0][nr] = 0;
        for (int i = 0; i < nsd; ++i) tiles[1][nr + i] = 0;
        if (p.has_shared) {
            GemmTask a;
            a.w = p.shared_gate;
            a.w2 = p.shared_up;
            a.s = p.shared_gate_s;
            a.s2 = p.shared_up_s;
            a.rows = p.rows;
            a.n_out = p.shared_width;
            a.k = p.hidden;
            a.a = p.xq;
            a.a_scale = p.xq_scale;
            a.a_width = p.hidden;
            a.y = p.shared_hidden;
            a.y_stride = p.shared_width;
            t0[nr] = a;
            tiles[0][nr] = tiles_rt(true, p.rows, p.shared_width);
            // the shared down projection as nsd k parts of `inter` columns
            // (its tiles then last as long as the routed ones'), part i into
            // shared_out (i = 0) or shared_out2 (i = 1)
            const int kpart = p.shared_width / nsd;
            for (int i = 0; i < nsd; ++i) {
                GemmTask b;
                const long col = (long)i * kpart;
                b.w = p.shared_down + (p.shared_fmt == kQ8 ? col : col / 2);
                b.s = p.shared_down_s;
                b.rows = p.rows;
                b.n_out = p.hidden;
                b.k = kpart;
                b.w_ld = p.shared_width;
                b.a = p.sq + limb_at(0, (int)col, p.shared_width);
                b.a_scale = p.sq_scale;
                b.a_width = p.shared_width;
                b.y = i == 0 ? p.shared_out : p.shared_out2;
                b.y_stride = p.hidden;
                t1[nr + i] = b;
                tiles[1][nr + i] = tiles_rt(false, p.rows, p.hidden);
            }
        }
    }
    lds_barrier();  // the tables are read by the next launch
    // tile prefix sums tile_start[u] = sum of tiles[s][v < u], u = 0..n: wave
    // s scans stage s, kPer consecutive entries per lane (one round of
    // independent LDS reads) and a wave scan over the lanes' sums (a loop of
    // dependent LDS reads per entry waited for each read in turn)
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (wave < 2) {
        const int s = wave;
        const int n = nr + (s == 0 ? 1 : nsd);  // tiles[s][0 .. n - 1] are set
        constexpr int kPer = (kQgMaxTasks + 1 + 63) / 64;
        int v[kPer], local = 0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int u = lane * kPer + i;
            v[i] = tiles[s][u < n ? u : 0];
            v[i] = u < n ? v[i] : 0;
            local += v[i];
        }
        int incl = local;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(incl, o, 64);
            if (lane >= o) incl += up;
        }
        int run = incl - local;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int u = lane * kPer + i;
            if (u <= n) p.tile_start[s * (kQgMaxTasks + 1) + u] = run;
            run += v[i];
        }
    }
}

// The token-row quantisation of the MoE input (RMSNorm'ed) and, in the last
// workgroup, the GEMM task and tile tables: one launch before stage 0.  Eight
// waves: a row each to quantise, or to route (the routing workgroup).
constexpr int kPrepWaves = 8;
static_assert(kPrepWaves >= 2, "moe_schedule_body scans with two waves");
template <bool REG>
__global__ __launch_bounds__(64 * kPrepWaves) void moe_prep_kernel(QuantSeg a, MoeScheduleParams sp,
                                                                   int blocks_a) {
    if ((int)blockIdx.x == blocks_a) {
        if (sp.p.route_in_prep) {
            // route_kernel's work: selection (wave w: row w), the route tables
            // kept in LDS for the schedule, the expert table staged in LDS
            // meanwhile
            __shared__ RouteLds L;
            __shared__ ExpertWeights ew[64];
            __shared__ __align__(16) unsigned long long keys[kPrepWaves][64];
            const RouteParams &rp = sp.p.route;  // rows <= kPrepWaves, experts <= 64
            const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
            if (wave == 0 && lane < rp.experts) ew[lane] = sp.p.expert_table[lane];
            if (wave < rp.rows) (void)select_row_64(rp, wave, lane, L.ids, keys[wave]);
            lds_barrier();
            small_tables(rp, L);
            lds_barrier();
            moe_schedule_body(sp, &L, ew);
            return;
        }
        moe_schedule_body(sp);
        return;
    }
    const int row = (int)blockIdx.x * kPrepWaves + (int)(threadIdx.x >> 6);
    if (row >= a.rows) return;
    quantize_row<REG>(a, row);
}


int moe_gemm(const MoeGemmParams &p, hipStream_t stream) {
    if (p.rows <= 0 || p.experts <= 0 || p.experts + 2 > kQgMaxTasks || p.top_k <= 0 ||
        p.rows > moe_gemm_max_rows(p.hidden) ||
        !qgemm_shape_ok(p.expert_fmt, p.hidden) || !qgemm_shape_ok(p.expert_fmt, p.inter) ||
        (p.has_shared && (!qgemm_shape_ok(p.shared_fmt, p.hidden) ||
                          !qgemm_shape_ok(p.shared_fmt, p.shared_width))))
        return kErrArgs;
    const int entries = p.rows * p.top_k;
    const int max_tasks = entries < p.experts ? entries : p.experts;
    // one tile kind for the whole layer, from the average rows per expert
    const bool k128 = p.hidden % 128 == 0 && p.inter % 128 == 0 &&
                      (!p.has_shared || p.shared_width % 128 == 0);
    const int fmt = p.expert_fmt == kQ8 || (p.has_shared && p.shared_fmt == kQ8) ? kQ8 : kQ4;
    const int kind = moe_tile(fmt, p.rows, (double)entries / p.experts, k128);
    const int bm = tile_bm(kind);
    MoeScheduleParams sp;
    sp.p = p;
    sp.bm = bm;
    // token rows (RMSNorm'ed) into limbs, and the task / tile tables in the
    // launch's last workgroup
    QuantSeg xs;
    xs.x = p.x;
    xs.x_stride = p.hidden;
    xs.rows = p.rows;
    xs.width = p.hidden;
    xs.norm_w = p.norm_w;
    xs.eps = p.eps;
    xs.q = p.xq;
    xs.scale = p.xq_scale;
    if (!p.x || !p.xq || !p.xq_scale || !quant_seg_ok(xs))
        return kErrArgs;
    if (p.route_in_prep &&
        (p.route.rows != p.rows || p.rows > kRouteOneGroupRows || !p.route.logits ||
         p.route.experts != p.experts || p.route.top_k != p.top_k || p.top_k > kMaxTopK ||
         p.experts > 64 || p.rows * p.top_k > kRouteFusedMaxPositions ||
         !p.route.ids || !p.route.weights || !p.route.n_unique || !p.route.unique ||
         !p.route.counts || !p.route.offsets || !p.route.list_rows || !p.route.list_slots ||
         !p.route.list_pos || !p.route.error))
        return kErrArgs;
    static_assert(kRouteOneGroupRows <= kPrepWaves, "a wave per routed row");
    const int blocks_x = (p.rows + kPrepWaves - 1) / kPrepWaves;
    if (p.hidden <= kQuantRegChunks * kWave * 4)
        hipLaunchKernelGGL(moe_prep_kernel<true>, dim3(blocks_x + 1), dim3(64 * kPrepWaves), 0,
                           stream, xs, sp, blocks_x);
    else
        hipLaunchKernelGGL(moe_prep_kernel<false>, dim3(blocks_x + 1), dim3(64 * kPrepWaves), 0,
                           stream, xs, sp, blocks_x);
    if (hipGetLastError() != hipSuccess) return kErrLaunch;
    int st = kOk;

    const bool same = !p.has_shared || p.shared_fmt == p.expert_fmt;
    for (int stage = 0; stage < 2; ++stage) {
        const bool dual = stage == 0;
        QGemmLaunch L;
        L.tasks = p.tasks + stage * kQgMaxTasks;
        L.tile_start = p.tile_start + stage * (kQgMaxTasks + 1);
        L.n_routed = p.n_unique;
        L.n_shared = dual ? 1 : moe_shared_down_parts(p);
        // upper bounds of the tile counts: sum_e ceil(n_e / BM) <= entries / BM + tasks
        const int routed_mt = entries / bm + max_tasks;
        const int routed_nt = host_tiles(dual, 1, dual ? p.inter : p.hidden, bm);
        const int shared_t =
            p.has_shared ? L.n_shared * host_tiles(dual, p.rows, dual ? p.shared_width : p.hidden, bm)
                         : 0;
        if (same) {
            L.range = 0;
            st = launch_qgemm_fmt(p.expert_fmt, dual, kind, L, routed_mt * routed_nt + shared_t,
                                  stream);
        } else {
            L.range = 1;
            st = launch_qgemm_fmt(p.expert_fmt, dual, kind, L, routed_mt * routed_nt, stream);
            if (!st) {
                L.range = 2;
                st = launch_qgemm_fmt(p.shared_fmt, dual, kind, L, shared_t, stream);
            }
        }
        if (st) return st;
        if (stage == 0) {
            // the expert hidden rows and the shared hidden rows in one launch
            QuantSeg hs, ss;
            hs.x = p.expert_hidden;
            hs.x_stride = p.inter;
            hs.rows = entries;
            hs.width = p.inter;
            hs.q = p.hq;
            hs.scale = p.hq_scale;
            if (p.has_shared) {
                ss.x = p.shared_hidden;
                ss.x_stride = p.shared_width;
                ss.rows = p.rows;
                ss.width = p.shared_width;
                ss.q = p.sq;
                ss.scale = p.sq_scale;
            }
            st = quantize_segments(hs, ss, stream);
            if (st) return st;
        }
    }
    return kOk;
}

}  // namespace mlh
