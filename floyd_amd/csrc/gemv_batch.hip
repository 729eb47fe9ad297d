// gemv_batch.hip -- q8 / q4 dequant matmul for a batch of token rows on int8
// matrix cores (gfx950: v_mfma_i32_16x16x64_i8), any width.
//
// Semantics are those of gemv() (moonlight_kernels.metal:43-130 and the
// RMSNorm / residual / SwiGLU variants, :23-41, :533-541).
//
// Numerics: those of gemv_mfma.hip.  A wave splits its 256-column range of a
// token row (a part of it, below) into four int8 limbs against a power-of-two
// step that maps the range's largest |x| below 2^30 (what lies below the step is
// cut: columns 2^6 and more below the largest keep fewer than 24 bits), the products
// with the stored weights are exact int32 sums, and the ranges' sums are added
// in fp32.  A NaN or infinity in the range makes the token row's outputs NaN.
//
// Work decomposition.  A workgroup (8 waves) owns 16 NB weight rows (SwiGLU:
// half gate, half up) and TOK = 4, 8 or 16 token rows; wave w takes 256
// columns of each 2048-column chunk.  No operand goes through LDS: lane (g, n)
// holds 16 columns of weight row n, the matrix core's B layout, and of token
// row n % TOK, loaded 64 contiguous bytes per token row, split into limbs and
// exchanged between the wave's four lane rows in registers.  With TOK < 16 the
// 16 / TOK lanes of a token row split different 64-column steps of the range
// (their products with the other parts' weights are dropped), so a wave's
// vector work falls with TOK.  The waves' sums meet in LDS.  With few row
// blocks and several chunks the chunks are split over workgroups (grid.y);
// each stores its sums and the last to arrive adds them in split order, as in
// gemv_mfma_splitk_kernel.
//
// Bound: the vector kernel (gemv_impl.h) reads the weights once per 4 token
// rows and multiplies on the vector units; here they are read once per TOK,
// and what is left is the split of x, which every workgroup repeats (about 8
// vector instructions per element and lane).  Measured on MI355X, graph
// replays over rotating weights, before and after: q8 3072 x 2048 at 6 rows
// 10.5 -> 5.0 us, at 64 rows 61.7 -> 10.4; q4 11264 x 2048 at 6 rows 15.8 ->
// 7.4, at 16 rows 30.1 -> 10.1; q8 2048 x 11264 at 3 rows 60.8 -> 9.5, at 16
// rows 278 -> 15.9.
//
// FP32X: the calls that the vector kernel does not take (ragged widths,
// unaligned operands, rows past its LDS) keep x in fp32, as the kernel that
// takes them otherwise (gemv.hip, gemv_generic_kernel) does: a range's step
// would hold the columns far below its largest in few bits, which shows in the
// outputs whose weight at the largest is small (999 columns, one of them 1e5
// times the rest, weight 0: 3.5e-5 against 1e-7).  The products then run on
// v_mfma_f32_16x16x4_f32, each started from zero and added pairwise, so a sum's
// chain is no longer than the other kernel's (error against 64 bits, 11999 x
// 11999 2.5e-7 there, 1.3e-7 here).  Widths that are no multiple of 16 columns
// (q8) or 32 (q4) are cut there: the rest of a row, under 32 products, is added
// in the epilogue.  Bound: the fp32 matrix units and the loads' latency; generic
// kernel against this one, q8: 1001 x 999 at 6 rows 9.8 / 6.0 us, at 200 rows
// 120 / 18; 11999 x 11999 at 1 row 189 / 126, at 16 rows 1769 / 143.
#include "limb_split.h"

#include <algorithm>
#include <cstdio>
#include <string>

namespace mlh {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kBtWaves = 8;
constexpr int kBtThreads = 64 * kBtWaves;
constexpr int kBtSteps = 4;                       // 64-column steps per wave and chunk
constexpr int kBtRange = 64 * kBtSteps;           // columns per wave and chunk
constexpr int kBtChunk = kBtWaves * kBtRange;     // 2048
constexpr int kBtMaxSplits = 16;
constexpr int kBtMaxParts = 256;                  // workgroups of a split launch (kBtTarget)
constexpr int kBtPartFloats = 64 * 16;            // their largest tile
constexpr int kBtCountStride = 32;                // ints between counters (128 bytes)

// Shares of a split launch (the library's own memory, static, per GPU:
// launches of one GPU run in order on the library's one stream).
__device__ float bt_part[kBtMaxParts * kBtPartFloats];
__device__ float bt_part_ss[kBtMaxParts * 16];
__device__ int bt_count[kBtMaxParts * kBtCountStride];  // zero between launches

struct BatchGeom {
    int chunks = 0, splits = 1;
    int k_main = 0;  // columns that the matrix cores take
};

// 16 bytes at any address.
__device__ __forceinline__ u32x4 load16_any(const void *p) {
    typedef unsigned u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
    return *(const __attribute__((address_space(1))) u32x4_any *)p;
}

// 16 packed nibbles (two words) as signed int8 in column order.
__device__ __forceinline__ i32x4 unpack_nibbles(unsigned a, unsigned b) {
    // u in [0, 15] -> u - 8: (u + 0x78) ^ 0x80, no carry between bytes
    auto word = [](unsigned lo, unsigned hi, unsigned sel) {
        return (int)((__builtin_amdgcn_perm(hi, lo, sel) + 0x78787878u) ^ 0x80808080u);
    };
    const unsigned la = a & 0x0F0F0F0Fu, ha = (a >> 4) & 0x0F0F0F0Fu;
    const unsigned lb = b & 0x0F0F0F0Fu, hb = (b >> 4) & 0x0F0F0F0Fu;
    return i32x4{word(la, ha, 0x05010400u), word(la, ha, 0x07030602u),
                 word(lb, hb, 0x05010400u), word(lb, hb, 0x07030602u)};
}

// Transposes a 4 x 4 block of words over the four 16-lane rows of a wave:
// afterwards r[j] of row g holds what r[g] of row j held.
__device__ __forceinline__ void transpose_rows(unsigned &r0, unsigned &r1, unsigned &r2,
                                               unsigned &r3) {
    const auto a = __builtin_amdgcn_permlane32_swap(r0, r2, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(r1, r3, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    r0 = c[0];
    r1 = c[1];
    r2 = d[0];
    r3 = d[1];
}

// Largest magnitude of four values and m; NaN if one of them is.
__device__ __forceinline__ float max_mag4(float m, const float (&v)[4]) {
    m = __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(m, __builtin_fabsf(v[0])), __builtin_fabsf(v[1]));
    return __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(m, __builtin_fabsf(v[2])), __builtin_fabsf(v[3]));
}

template <int FMT>
__device__ __forceinline__ float weight_at(const uint8_t *row, int k) {
    if constexpr (FMT == kQ8) return (float)reinterpret_cast<const int8_t *>(row)[k];
    const uint8_t b = row[k >> 1];
    return (float)((k & 1) ? (b >> 4) - 8 : (b & 15) - 8);
}

// A wave's sums over a chunk in fp32: sum[b][r] += token row 4 g + r times weight
// block b, and with a norm ss += x^2 of this lane's columns.  The wave takes
// every kBtWaves-th piece of 64 columns (q8) or 128 (q4), so that a short row is
// spread over the waves; lane (g, n) supplies the same 16 or 32 consecutive
// columns of a piece for token row n and for weight row n.
template <int FMT, int NB>
__device__ __forceinline__ void chunk_f32(const float *xrow, const float *norm_w,
                                          const uint8_t *const (&wrow)[NB], int chunk, int wave,
                                          int k_main, int g, float (&sum)[NB][4], float &ss) {
    typedef float f32x4v __attribute__((ext_vector_type(4)));
    constexpr int kPieces = FMT == kQ8 ? 4 : 2, kCols = 64 / kPieces, kQuads = kCols / 4;
    u32x4 x[kPieces][kQuads], nw[kPieces][kQuads] = {}, w[kPieces][NB];
    int first[kPieces];  // column of the piece
    bool in[kPieces];    // this lane's columns lie inside the row
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        first[i] = ((chunk * kPieces + i) * kBtWaves + wave) * (4 * kCols);
        if (first[i] >= k_main) break;  // uniform; the later pieces lie further on
        int at = first[i] + kCols * g;
        in[i] = at < k_main;
        if (!in[i]) at = 0;  // x is taken as zero there
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            x[i][j] = load16_any(xrow + at + 4 * j);
            if (norm_w) nw[i][j] = load16_any(norm_w + at + 4 * j);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) w[i][b] = load16_any(wrow[b] + (FMT == kQ8 ? at : at / 2));
    }
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        if (first[i] >= k_main) break;
        f32x4v part[kQuads / 4][NB];
#pragma unroll
        for (int h = 0; h < kQuads / 4; ++h) {
            f32x4v quad[4][NB];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int q = 4 * h + j;
                const u32x4 xq = x[i][q], nq = nw[i][q];
                float v[4] = {__uint_as_float(xq.x), __uint_as_float(xq.y), __uint_as_float(xq.z),
                              __uint_as_float(xq.w)};
                const float n4[4] = {__uint_as_float(nq.x), __uint_as_float(nq.y),
                                     __uint_as_float(nq.z), __uint_as_float(nq.w)};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = in[i] ? v[e] : 0.0f;
                    if (norm_w) {
                        ss = fmaf(v[e], v[e], ss);
                        v[e] = in[i] ? v[e] * n4[e] : 0.0f;
                    }
                }
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const u32x4 d = w[i][b];
                    const int word = FMT == kQ8 ? q : q / 2;  // of the four columns' weights
                    const unsigned bits = word == 0 ? d.x : word == 1 ? d.y : word == 2 ? d.z : d.w;
                    f32x4v m[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float wv = FMT == kQ8
                                             ? (float)(int8_t)(bits >> (8 * e))
                                             : (float)((int)((bits >> (16 * (q & 1) + 4 * e)) & 15) - 8);
                        m[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], wv, f32x4v{0.f, 0.f, 0.f, 0.f},
                                                                    0, 0, 0);
                    }
                    quad[j][b] = (m[0] + m[1]) + (m[2] + m[3]);
                }
                // the next products after these sums: 4 NB results in
                // registers, not all of the piece's
                if (q + 1 < kQuads) {
#pragma unroll
                    for (int b = 0; b < NB; ++b) asm("" : "+v"(quad[j][b]), "+v"(x[i][q + 1]));
                }
            }
#pragma unroll
            for (int b = 0; b < NB; ++b)
                part[h][b] = (quad[0][b] + quad[1][b]) + (quad[2][b] + quad[3][b]);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                sum[b][r] += kQuads == 8 ? part[0][b][r] + part[kQuads / 4 - 1][b][r] : part[0][b][r];
    }
}

template <int FMT, bool DUAL, int NB, int TOK, bool FP32X>
__global__ __launch_bounds__(kBtThreads) void gemv_batch_kernel(GemvParams p, BatchGeom q) {
    constexpr int NR = 16 * NB;              // weight rows
    constexpr int NO = DUAL ? NR / 2 : NR;   // output columns
    constexpr int S = kBtSteps;
    constexpr int NW = FMT == kQ8 ? S : S / 2;  // 16-byte pieces per weight row and lane
    constexpr int kSubs = 16 / TOK;          // parts of a range over the lanes of a token row
    constexpr int SS = S / kSubs;            // steps per part
    static_assert(!DUAL || NB % 2 == 0, "gate and up blocks");
    static_assert(!FP32X || TOK == 16, "a token row per lane of a lane row");
    static_assert(TOK * NR <= kBtPartFloats && TOK % 4 == 0, "share size; a C row group in one part");
    __shared__ __attribute__((aligned(16))) float red[kBtWaves][16][NR];
    __shared__ float red_ss[kBtWaves][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    const int rb = blockIdx.x, split = blockIdx.y, t0 = blockIdx.z * TOK;
    const long row_bytes = FMT == kQ8 ? p.I : (p.I + 1) / 2;
    const bool has_norm = p.norm_w != nullptr;

    const uint8_t *wrow[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int o = rb * NO + (DUAL ? b % (NB / 2) : b) * 16 + n;
        wrow[b] = (DUAL && b >= NB / 2 ? p.w2 : p.w) + (long)(o < p.O ? o : p.O - 1) * row_bytes;
    }
    const int sub = n / TOK, xr = min(t0 + n % TOK, p.rows - 1);
    const float *xrow = p.x + (long)xr * p.x_stride;
    float sum[NB][4], ss = 0.0f;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[b][r] = 0.0f;

    for (int c = split; c < q.chunks; c += q.splits) {
        if constexpr (FP32X) {
            chunk_f32<FMT, NB>(xrow, p.norm_w, wrow, c, wave, q.k_main, g, sum, ss);
            continue;
        }
        const int base = (c * kBtWaves + wave) * kBtRange;
        if (base >= q.k_main) break;  // this wave's later chunks lie past the end too
        const bool whole = base + kBtRange <= q.k_main;
        // four consecutive columns per lane and load, 64 contiguous bytes
        // per token row and part: v[4 i + j] holds those that become word
        // j of the part's step i (q4: a lane's 16 columns of two steps
        // lie together, so the steps' loads alternate)
        float v[4 * SS][4];
        int col[4 * SS];
#pragma unroll
        for (int i = 0; i < 4 * SS; ++i) {
            const int s = sub * SS + i / 4;
            col[i] = base + 16 * (FMT == kQ8 ? 4 * s + i % 4
                                             : 8 * (s >> 1) + 2 * (i % 4) + (s & 1));
            const u32x4 d = load_global16(xrow + (col[i] < q.k_main ? col[i] : 0) + 4 * g);
            v[i][0] = __uint_as_float(d.x);
            v[i][1] = __uint_as_float(d.y);
            v[i][2] = __uint_as_float(d.z);
            v[i][3] = __uint_as_float(d.w);
        }
        u32x4 nw[4 * SS] = {};
        if (has_norm) {
#pragma unroll
            for (int i = 0; i < 4 * SS; ++i)
                nw[i] = load_global16(p.norm_w + (col[i] < q.k_main ? col[i] : 0) + 4 * g);
        }
        // weights: first column of this lane's 16 at step s (q4: a 16-byte
        // piece holds the lane's columns of two steps); column 0 past the end,
        // where x is zero
        int at[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            at[i] = base + (FMT == kQ8 ? 64 * i + 16 * g : 128 * i + 32 * g);
            if (at[i] >= q.k_main) at[i] = 0;
        }
        u32x4 w[NB][NW];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < NW; ++i)
                w[b][i] = load_global16(wrow[b] + (FMT == kQ8 ? at[i] : at[i] / 2));
        if (!whole) {
#pragma unroll
            for (int i = 0; i < 4 * SS; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][e] = col[i] < q.k_main ? v[i][e] : 0.0f;
        }
        if (has_norm) {
#pragma unroll
            for (int i = 0; i < 4 * SS; ++i) {
                const float n4[4] = {__uint_as_float(nw[i].x), __uint_as_float(nw[i].y),
                                     __uint_as_float(nw[i].z), __uint_as_float(nw[i].w)};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ss = fmaf(v[i][e], v[i][e], ss);
                    v[i][e] *= n4[e];
                }
            }
        }
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 4 * SS; ++i) amax = max_mag4(amax, v[i]);
        amax = __builtin_elementwise_maximum(amax, __shfl_xor(amax, 16));
        amax = __builtin_elementwise_maximum(amax, __shfl_xor(amax, 32));
        // 2^ex with amax 2^ex < 2^30
        const unsigned bits = __float_as_uint(amax) & 0x7FFFFFFFu;
        const int ex = min(156 - (int)(bits >> 23), 126);
        const float step_inv = __uint_as_float((unsigned)(127 + ex) << 23);
        // a value that the limbs cannot carry makes the token row NaN
        const float step = bits >= 0x7F800000u ? __builtin_nanf("")
                                               : __uint_as_float((unsigned)(127 - ex) << 23);
        i32x4 acc[kSubs][4][NB];
#pragma unroll
        for (int u = 0; u < kSubs; ++u)
#pragma unroll
            for (int L = 0; L < 4; ++L)
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[u][L][b] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < SS; ++i) {
            // the limbs of step i's four loads, then each lane row takes
            // its own 16 columns
            unsigned l[4][4];  // [limb][word]
#pragma unroll
            for (int j = 0; j < 4; ++j)
                split_limbs4(v[4 * i + j], step_inv, l[0][j], l[1][j], l[2][j], l[3][j]);
#pragma unroll
            for (int L = 0; L < 4; ++L) transpose_rows(l[L][0], l[L][1], l[L][2], l[L][3]);
            // every part's weights meet all 16 operand rows; a part's own
            // rows are picked below
#pragma unroll
            for (int u = 0; u < kSubs; ++u) {
                const int s = u * SS + i;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    i32x4 B;
                    if constexpr (FMT == kQ8) {
                        const u32x4 d = w[b][s];
                        B = i32x4{(int)d.x, (int)d.y, (int)d.z, (int)d.w};
                    } else {
                        const u32x4 d = w[b][s >> 1];
                        B = (s & 1) ? unpack_nibbles(d.z, d.w) : unpack_nibbles(d.x, d.y);
                    }
#pragma unroll
                    for (int L = 0; L < 4; ++L)
                        acc[u][L][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            i32x4{(int)l[L][0], (int)l[L][1], (int)l[L][2], (int)l[L][3]}, B,
                            acc[u][L][b], 0, 0, 0);
                }
            }
        }
        // register r holds operand row 4 g + r, part 4 g / TOK: its step
        // from that row's lane.  |limb sums| <= 2^22 (limb 0: 2^21), so
        // pairs combine exactly
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float sc = __shfl(step, 4 * g + r);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                int c4[4];
#pragma unroll
                for (int L = 0; L < 4; ++L) {
                    c4[L] = acc[0][L][b][r];
#pragma unroll
                    for (int u = 1; u < kSubs; ++u)
                        c4[L] = 4 * g / TOK == u ? acc[u][L][b][r] : c4[L];
                }
                const int hi = c4[0] * 256 + c4[1], lo = c4[2] * 256 + c4[3];
                sum[b][r] = fmaf(fmaf((float)hi, 65536.0f, (float)lo), sc, sum[b][r]);
            }
        }
    }
    if (has_norm) {
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (lane < 16) red_ss[wave][lane] = ss;
    }

    // ---- the waves' sums in wave order, and the epilogue
    const int part = (blockIdx.z * gridDim.x + rb) * q.splits + split;
    auto finish = [&](int t, int j, float v, float u, float tss) {
        const int row = t0 + t, o = rb * NO + j;
        if (row >= p.rows || o >= p.O) return;
        if (FP32X && q.k_main < p.I) {
            // eight columns' loads at a time
            float vt = 0.0f, ut = 0.0f;
            const float *x = p.x + (long)row * p.x_stride;
            const uint8_t *wr = p.w + (long)o * row_bytes;
            const uint8_t *ur = DUAL ? p.w2 + (long)o * row_bytes : wr;
            for (int k0 = q.k_main; k0 < p.I; k0 += 8) {
                float xv[8], nv[8], wv[8], uv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int k = min(k0 + e, p.I - 1);
                    xv[e] = x[k];
                    nv[e] = has_norm ? p.norm_w[k] : 1.0f;
                    wv[e] = weight_at<FMT>(wr, k);
                    uv[e] = DUAL ? weight_at<FMT>(ur, k) : 0.0f;
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (k0 + e >= p.I) break;
                    tss = fmaf(xv[e], xv[e], tss);
                    const float xn = xv[e] * nv[e];
                    vt = fmaf(xn, wv[e], vt);
                    if (DUAL) ut = fmaf(xn, uv[e], ut);
                }
            }
            v += vt;
            u += ut;
        }
        const float inv = has_norm ? 1.0f / sqrtf(tss / (float)p.I + p.eps) : 1.0f;
        float out = v * inv * p.s[o];
        if (DUAL) out = silu(out) * (u * inv * p.s2[o]);
        else if (p.epilogue == kEpiResidual) out = p.resid[(long)row * p.resid_stride + o] + out;
        p.y[(long)row * p.y_stride + o] = out;
    };
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][4 * g + r][16 * b + n] = sum[b][r];
    __syncthreads();
    for (int i = tid; i < TOK * NO; i += kBtThreads) {
        const int m = i / NO, j = i % NO;
        auto total = [&](int col) {
            float v = 0.0f;
#pragma unroll
            for (int w8 = 0; w8 < kBtWaves; ++w8)
#pragma unroll
                for (int u = 0; u < kSubs; ++u) v += red[w8][u * TOK + m][col];
            return v;
        };
        const float v = total(j), u = DUAL ? total(NO + j) : 0.0f;
        float tss = 0.0f;
        if (has_norm) {
#pragma unroll
            for (int w8 = 0; w8 < kBtWaves; ++w8)
#pragma unroll
                for (int u8 = 0; u8 < kSubs; ++u8) tss += red_ss[w8][u8 * TOK + m];
        }
        if (q.splits == 1) {
            finish(m, j, v, u, tss);
        } else {
            float *dst = bt_part + (long)part * kBtPartFloats + m * NR + j;
            __hip_atomic_store(dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (DUAL)
                __hip_atomic_store(dst + NO, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (j == 0)
                __hip_atomic_store(bt_part_ss + part * 16 + m, tss, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (q.splits == 1) return;
    int *count = bt_count + (blockIdx.z * gridDim.x + rb) * kBtCountStride;
    if (!agent_handoff_arrive(count, q.splits)) return;
    const int part0 = part - split;
    for (int i = tid; i < TOK * NO; i += kBtThreads) {
        const int m = i / NO, j = i % NO;
        float v = 0.0f, u = 0.0f, tss = 0.0f;
        for (int k = 0; k < q.splits; ++k) {
            const float *src = bt_part + (long)(part0 + k) * kBtPartFloats + m * NR + j;
            v += __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (DUAL)
                u += __hip_atomic_load(src + NO, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (has_norm)
                tss += __hip_atomic_load(bt_part_ss + (part0 + k) * 16 + m, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
        }
        finish(m, j, v, u, tss);
    }
    if (tid == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct BatchPlan {
    int nb = 2, tok = 16;
    bool fp32x = false;
    BatchGeom geom;
    dim3 grid;
};

// Weight rows per workgroup: the fewest that leave at most one workgroup per
// CU over row blocks, token groups and chunks (each workgroup splits all of
// its token rows, so more row blocks than CUs only repeat that: q8 3072 x 2048
// at 64 rows 19.5 us with 16 rows, 14.9 with 32, 10.4 with 64; at 16 rows 7.3,
// 8.1 and 10.3).  Up to 4 token rows the split is a quarter and 16 rows are
// best throughout (2048 x 11264 at 3 rows 9.8 against 12.9 us).  Chunks are
// split over workgroups up to the same count (2048 x 11264 at 128 rows 43.1
// us; 52.9 when split up to 512).
constexpr int kBtTarget = kBtMaxParts;

BatchPlan plan_batch(const GemvParams &p, bool fp32x) {
    BatchPlan pl;
    const bool dual = p.epilogue == kEpiSiluDual;
    const int cut = p.fmt == kQ8 ? 16 : 32;
    pl.fp32x = fp32x;
    pl.geom.k_main = p.I / cut * cut;
    pl.geom.chunks = (pl.geom.k_main + kBtChunk - 1) / kBtChunk;
    pl.tok = fp32x || p.rows > 8 ? 16 : p.rows > 4 ? 8 : 4;
    const int groups = (p.rows + pl.tok - 1) / pl.tok;
    const long weight_rows = (long)p.O * (dual ? 2 : 1);
    auto blocks = [&](int nb) { return (int)((weight_rows + 16 * nb - 1) / (16 * nb)); };
    auto units = [&](int nb) { return (long)blocks(nb) * groups * pl.geom.chunks; };
    pl.nb = 2;
    if (!dual && (pl.tok == 4 || units(1) <= kBtTarget)) pl.nb = 1;
    else if (!fp32x && pl.tok >= 8 && units(2) > kBtTarget) pl.nb = 4;
    const int n = blocks(pl.nb);
    int splits = 1;
    while (splits < pl.geom.chunks && splits < kBtMaxSplits &&
           (long)n * groups * (splits + 1) <= kBtTarget)
        ++splits;
    pl.geom.splits = splits;
    pl.grid = dim3(n, splits, groups);
    return pl;
}

template <int FMT, bool DUAL, int NB, int TOK, bool FP32X = false>
void launch(const GemvParams &p, const BatchPlan &pl, hipStream_t stream) {
    hipLaunchKernelGGL((gemv_batch_kernel<FMT, DUAL, NB, TOK, FP32X>), pl.grid, dim3(kBtThreads), 0,
                       stream, p, pl.geom);
}
template <int FMT, bool DUAL, int TOK>
void launch_nb(const GemvParams &p, const BatchPlan &pl, hipStream_t stream) {
    if constexpr (!DUAL) {
        if (pl.nb == 1) return launch<FMT, DUAL, 1, TOK>(p, pl, stream);
    }
    if constexpr (TOK >= 8) {
        if (pl.nb == 4) return launch<FMT, DUAL, 4, TOK>(p, pl, stream);
    }
    launch<FMT, DUAL, 2, TOK>(p, pl, stream);
}
template <int FMT, bool DUAL>
void launch_tok(const GemvParams &p, const BatchPlan &pl, hipStream_t stream) {
    if (pl.fp32x) {
        if constexpr (!DUAL) {
            if (pl.nb == 1) return launch<FMT, DUAL, 1, 16, true>(p, pl, stream);
        }
        launch<FMT, DUAL, 2, 16, true>(p, pl, stream);
    } else if (pl.tok == 4) launch_nb<FMT, DUAL, 4>(p, pl, stream);
    else if (pl.tok == 8) launch_nb<FMT, DUAL, 8>(p, pl, stream);
    else launch_nb<FMT, DUAL, 16>(p, pl, stream);
}

}  // namespace

// Launches the kernel for p (q8 / q4, no router partials), with
// x in fp32 (FP32X) or, where the vector kernel takes p, in limbs; false,
// launching nothing, when it does not take it.  With `name` set it
// launches nothing and stores the kernel's template name.
bool gemv_batch(const GemvParams &p, bool fp32x, hipStream_t stream, std::string *name) {
    if ((p.fmt != kQ8 && p.fmt != kQ4) || p.router_parts) return false;
    const bool dual = p.epilogue == kEpiSiluDual;
    const BatchPlan pl = plan_batch(p, fp32x);
    if (name) {
        char buf[96];
        snprintf(buf, sizeof(buf),
                 "mlh::(anonymous namespace)::gemv_batch_kernel<%d, %s, %d, %d, %s>", p.fmt,
                 dual ? "true" : "false", pl.nb, pl.tok, pl.fp32x ? "true" : "false");
        *name = buf;
        return true;
    }
    const int slice = 65535 * pl.tok;  // token rows of a launch's grid
    for (long r0 = 0; r0 < p.rows; r0 += slice) {
        GemvParams q = p;
        q.rows = (int)std::min<long>(slice, p.rows - r0);
        q.x += r0 * p.x_stride;
        q.y += r0 * p.y_stride;
        if (p.resid) q.resid += r0 * p.resid_stride;
        const BatchPlan ql = plan_batch(q, fp32x);
        if (p.fmt == kQ8) {
            if (dual) launch_tok<kQ8, true>(q, ql, stream);
            else launch_tok<kQ8, false>(q, ql, stream);
        } else {
            if (dual) launch_tok<kQ4, true>(q, ql, stream);
            else launch_tok<kQ4, false>(q, ql, stream);
        }
    }
    return true;
}

}  // namespace mlh
