// mlh_host.h -- host-side interface of the Moonlight HIP kernels (internal).
// The public C ABI (include/*.h) is implemented on top of these launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

namespace mlh {

enum Fmt { kF32 = 0, kQ8 = 1, kQ4 = 2 };
enum Epilogue { kEpiPlain = 0, kEpiResidual = 1, kEpiSiluDual = 2 };
enum Status { kOk = 0, kErrArgs = -1, kErrLaunch = -2, kErrDevice = -3, kErrSize = -4 };

constexpr int kMaxGemvRows = 4;

// y[b, o] = epilogue((sum_i xn[b, i] * W[o, i]) * s[o]) for b < rows, where
// xn = RMSNorm(x) * norm_w when norm_w is set, else x.
struct GemvParams {
    int fmt = kQ8;
    const uint8_t *w = nullptr;   // [O, row_bytes]
    const float *s = nullptr;     // [O] (unused for f32)
    const uint8_t *w2 = nullptr;  // up projection for kEpiSiluDual
    const float *s2 = nullptr;
    int O = 0;                    // output width (rows of W)
    int I = 0;                    // input width
    int rows = 0;                 // token rows
    const float *x = nullptr;
    long x_stride = 0;            // floats between token rows of x
    const float *norm_w = nullptr;
    float eps = 1e-5f;
    float *y = nullptr;
    long y_stride = 0;
    const float *resid = nullptr;  // kEpiResidual: y = resid + result
    long resid_stride = 0;
    int epilogue = kEpiPlain;
    // optional, one token row of a plain or residual epilogue on the int8
    // matrix-core kernels (gemv_router_ok): router logit partials of the
    // output row y for the next MoE layer's router.  Workgroup j of the
    // launch writes router_parts[e * n + j] = sum over its output rows o of
    // router_w[e, o] * (y[o] * router_nw[o]) for e < router_experts and
    // router_parts[router_experts * n + j] = sum of y[o]^2 (n = the launch's
    // workgroups, gemv_router_parts)
    const float *router_w = nullptr;   // [router_experts, O] f32
    const float *router_nw = nullptr;  // [O] the router input's RMSNorm weight
    float *router_parts = nullptr;
    int router_experts = 0;
};

int gemv(const GemvParams &p, hipStream_t stream);

// Whether a q8 / q4 projection of several token rows stays on the batch kernel
// (gemv_batch.hip, one launch, x split in every workgroup) rather than
// quantising its rows once for the GEMM tiles (qgemm.hip).  The batch kernel
// takes 30 us per 1000 workgroups of 64 weight rows, 16 token rows and 2048
// columns; the tiles take 28 us for 2048 columns, 50 for 4096 and 120 for 11264
// until their tiles fill the CUs.  Measured on MI355X, batch against tiles: 3072
// x 2048 at 256 rows 28.9 / 29.9 us, at 512 56.7 / 32.6; 11264 x 2048 at 64 rows
// 29.3 / 31.6, at 128 56.7 / 32.1; 8000 x 4096 at 64 rows 36.7 / 56.0, at 300
// 173 / 58; 2048 x 11264 at 256 rows 87 / 123, at 777 282 / 139.
inline bool gemv_batch_fits(long weight_rows, int rows, int in_width) {
    const long chunks = (in_width + 2047) / 2048;
    return (weight_rows + 63) / 64 * ((rows + 15) / 16) * chunks <= 300 + 600 * chunks;
}
// The same for a gemv() call: its tiles split a long reduction over the CUs
// (SwiGLU pairs don't) and then take 37 us for 4096 columns, 41 for 6144, 44 for
// 8192 and 48 for 11264.  Batch against tiles: 2048 x 4096 at 200 rows 37.1 / 36.5
// us, at 350 54.9 / 38.4; 2048 x 6144 at 150 49.6 / 40.1; 2048 x 8192 at 100 32.9 /
// 42.1, at 200 63.8 / 44.1; 2048 x 11264 at 96 43.4 / 47.8, at 192 84.5 / 49.1;
// 576 x 11264 at 200 28.6 / 50.8, at 700 86.5 / 59.0.
inline bool gemv_batch_fits(const GemvParams &p) {
    const long chunks = (p.I + 2047) / 2048;
    if (p.epilogue == kEpiSiluDual || chunks == 1)
        return gemv_batch_fits((long)p.O * (p.epilogue == kEpiSiluDual ? 2 : 1), p.rows, p.I);
    return ((long)p.O + 63) / 64 * ((p.rows + 15) / 16) * chunks <= 600 + 110 * chunks;
}
// Token rows of a workgroup of the f32 batch kernel (gemv_f32_batch.hip: a
// workgroup holds them in LDS) for a matrix of `weight_rows` rows: 4, 8 or 16,
// halved until they fit; 0 where the vector kernel, which takes 4 token rows a
// pass, is as fast.  A wave's pass over its few weight rows costs some 4 us of
// reductions and latency whatever their length, so narrow matrices stay off it.
// With a norm, which the vector kernel applies again for each of its weight
// rows, the line is 352 columns, and 8192 over the token rows of a 16-row
// workgroup (their padding is multiplied too); without one 1024 columns and at
// least 5 token rows, and with 16-row workgroups either all of their passes of 4
// or two full rounds of workgroups over the CUs.  Measured on MI355X, this kernel
// against the vector kernel, with norm: 163840 x 2048 at 2 rows 211 / 231 us, 3
// rows 212 / 384, 8 rows 214 / 838, 16 rows 327 / 1673; 9000 x 352 at 4 rows 8 / 9,
// at 9 rows 24 / 17; 9000 x 1024 at 9 rows 32 / 33; 20000 x 256 at 3 rows 13 / 9;
// 70000 x 64 at 16 rows 49 / 27; 4100 x 2048 at 3 rows 15.8 / 16.1.  Without:
// 163840 x 2048 at 4 rows 212 / 224, at 6 rows 212 / 423; 20000 x 704 at 8 rows 25 /
// 21, 20000 x 1024 29 / 33; 9000 x 2048 at 9 rows 45 / 36, at 16 rows 45 / 49; 20000 x
// 1024 at 9 rows 45 / 46; 20000 x 5120 at 6 rows (two workgroups of 4) 139 / 125;
// 4100 x 2048 at 6 rows 18.7 / 13.9.
constexpr long kF32BatchLds = 144 * 1024;
inline int f32_batch_rows(long weight_rows, int in_width, int rows, bool norm) {
    if (rows < (norm ? 3 : 5) || weight_rows < (norm ? 4096 : 8192) || in_width < (norm ? 352 : 1024))
        return 0;
    int b = rows <= 4 ? 4 : rows <= 8 ? 8 : 16;
    while (b > 4 && 4L * b * in_width > kF32BatchLds) b /= 2;
    if (4L * b * in_width > kF32BatchLds || (!norm && b < 8)) return 0;
    if (b < 16) return b;
    const int groups = (rows + 15) / 16;
    const bool pays = norm ? (long)in_width * rows >= 8192L * groups
                           : weight_rows >= 16384 || (rows + 3) / 4 == 4 * groups;
    return pays ? b : 0;
}

// Whether gemv() can write router logit partials for p (router fields
// aside), and how many partials per expert it then writes.
bool gemv_router_ok(const GemvParams &p);
int gemv_router_parts(const GemvParams &p);

struct GemvPlan;
// Launch geometry the planner picks for a GEMV shape (exposed for the grouped
// expert launches, which share the GEMV core).
GemvPlan plan_gemv(int fmt, int O, int I, int rows, bool dual);
std::string gemv_kernel_name(int fmt, int O, int I, int rows, bool dual);

// Packs f32 rows like tools/convert_moonlight.py:46-66 (bits 8 or 4).
int quantize_rows(int bits, const float *w, int rows, int cols, uint8_t *q, float *s,
                  hipStream_t stream);
// out[i] = bf16_round(mean + std * N(0,1)) from a counter-based generator
// (synthetic weights; the distribution, not the stream, is the contract).
int fill_normal(float *out, int64_t n, uint64_t seed, float mean, float std, int bf16,
                hipStream_t stream);

// dst = src with 16-byte non-temporal loads/stores (bandwidth yardstick).
int copy16(const void *src, void *dst, size_t bytes, hipStream_t stream);
// Reads `bytes` of src with `blocks` workgroups (out: blocks*4 words).
int read16(const void *src, size_t bytes, int blocks, unsigned *out, hipStream_t stream);

}  // namespace mlh
