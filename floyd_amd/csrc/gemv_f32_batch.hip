// gemv_f32_batch.hip -- f32 matrices of many rows (the output head) against 2
// or more token rows: y = W x (moonlight_kernels.metal:43-61, with the RMSNorm
// prologue and the residual of gemv()).
//
// The vector kernel (gemv_impl.h) reads every token row and the norm weight
// again from the caches for each of its few weight rows: 4 to 9 bytes of them
// per weight byte, and 4 token rows a pass.  Here a workgroup holds its token
// rows (x * norm_w) in LDS and streams weight rows past them: a wave takes R
// rows, 1 KB of each per load, the next loads in flight while these are
// multiplied, and reads the LDS once per R of them, so it moves B / R bytes of
// LDS per weight byte.  fp32 FMAs; a lane's sums meet in a butterfly; the
// norm's 1 / rms is applied to the sums.
//
// Bound: HBM up to 8 token rows (163840 x 2048 at 8 rows with norm on MI355X: 838
// -> 214 us, 6.3 TB/s), the vector units at 16.
#include "gemv_impl.h"

#include <cstdio>
#include <string>

namespace mlh {

namespace {

constexpr int kFbWaves = 8;
constexpr int kFbThreads = 64 * kFbWaves;

template <int B> struct FbShape {
    static constexpr int kR = B <= 8 ? 8 : 4;          // weight rows per wave and pass
    static constexpr int kRows = kFbWaves * kR;        // per workgroup and pass
    static_assert(kR * B <= 64, "the butterfly's values");
};

template <int B>
__global__ __launch_bounds__(kFbThreads) void gemv_f32_batch_kernel(GemvParams p, int passes) {
    constexpr int R = FbShape<B>::kR, NV = R * B;
    extern __shared__ __attribute__((aligned(16))) float fb_x[];  // [B][I]
    __shared__ float ss_part[kFbWaves][B];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = blockIdx.y * B;
    const bool has_norm = p.norm_w != nullptr;

    // ---- token rows into LDS (rows past the last repeat it)
    float ss[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const float *x = p.x + (long)min(t0 + b, p.rows - 1) * p.x_stride;
        ss[b] = 0.0f;
        for (int i = tid * 4; i < p.I; i += kFbThreads * 4) {
            f32x4 v = load_f4(x + i);
            if (has_norm) {
                const f32x4 n = load_f4(p.norm_w + i);
                ss[b] += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                v = f32x4{v.x * n.x, v.y * n.y, v.z * n.z, v.w * n.w};
            }
            *reinterpret_cast<f32x4 *>(fb_x + (long)b * p.I + i) = v;
        }
        ss[b] = wave_sum(ss[b]);
        if (lane == 0) ss_part[wave][b] = ss[b];
    }
    __syncthreads();
    const int vi = butterfly_index<NV, 64>(lane), vr = vi / B, vb = vi % B;
    float inv = 1.0f;  // of this lane's token row
    if (has_norm) {
        float tot = 0.0f;
#pragma unroll
        for (int w = 0; w < kFbWaves; ++w) tot += ss_part[w][vb];
        inv = 1.0f / sqrtf(tot / (float)p.I + p.eps);
    }

    const int nc = p.I / 4;  // 16-byte chunks of a row
    for (int pass = 0; pass < passes; ++pass) {
        const int row0 = ((blockIdx.x * passes + pass) * kFbWaves + wave) * R;
        if (row0 >= p.O) break;
        const uint8_t *wr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) wr[r] = p.w + (long)min(row0 + r, p.O - 1) * p.I * 4;
        float acc[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = 0.0f;
        auto fetch = [&](u32x4 (&w)[R], int c) {
#pragma unroll
            for (int r = 0; r < R; ++r) w[r] = load_stream16(wr[r] + (long)min(c, nc - 1) * 16);
        };
        auto multiply = [&](const u32x4 (&w)[R], int c) {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const f32x4 x = *reinterpret_cast<const f32x4 *>(fb_x + (long)b * p.I + 4 * c);
                const float xv[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    // a chunk's four products first: a lane's running sum then
                    // takes a quarter of the roundings
                    const float d = __uint_as_float(w[r].x) * xv[0];
                    acc[r * B + b] += fmaf(__uint_as_float(w[r].w), xv[3],
                                           fmaf(__uint_as_float(w[r].z), xv[2],
                                                fmaf(__uint_as_float(w[r].y), xv[1], d)));
                }
            }
        };
        u32x4 w0[R], w1[R];
        fetch(w0, lane);
        for (int c0 = 0; c0 < nc; c0 += 128) {
            const int c = c0 + lane;
            fetch(w1, c + 64);
            if (c < nc) multiply(w0, c);
            if (c0 + 128 < nc) fetch(w0, c + 128);
            if (c + 64 < nc) multiply(w1, c + 64);
        }
        butterfly_reduce<NV, 64>(acc, lane);
        const int row = row0 + vr, t = t0 + vb;
        if (butterfly_writer<NV, 64>(lane) && row < p.O && t < p.rows) {
            float out = acc[0] * inv;
            if (p.epilogue == kEpiResidual) out = p.resid[(long)t * p.resid_stride + row] + out;
            p.y[(long)t * p.y_stride + row] = out;
        }
    }
}

template <int B>
void launch(const GemvParams &p, hipStream_t stream) {
    const int lds = B * p.I * 4;
    static const bool attr = [] {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_f32_batch_kernel<B>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)kF32BatchLds) == hipSuccess;
    }();
    (void)attr;
    // as many workgroups as fit the CUs at once, twice over, so that the token
    // rows are staged for at least a few passes of weight rows
    const int blocks = (p.O + FbShape<B>::kRows - 1) / FbShape<B>::kRows;
    const int resident = 256 * (lds <= 36 * 1024 ? 2 : 1);
    const int passes = (blocks + 2 * resident - 1) / (2 * resident);
    hipLaunchKernelGGL((gemv_f32_batch_kernel<B>),
                       dim3((blocks + passes - 1) / passes, (p.rows + B - 1) / B), dim3(kFbThreads), lds,
                       stream, p, passes);
}

}  // namespace

// Launches the kernel for p; false, launching nothing, where it does not take p
// or the vector kernel is as fast (f32_batch_rows).  With `name` set it launches
// nothing and stores the kernel's template name.
bool gemv_f32_batch(const GemvParams &p, hipStream_t stream, std::string *name) {
    auto al = [](const void *q) { return ((uintptr_t)q & 15u) == 0; };
    if (p.fmt != kF32 || p.epilogue == kEpiSiluDual || p.router_parts || p.I % 4 ||
        !al(p.w) || !al(p.x) || p.x_stride % 4 || (p.norm_w && !al(p.norm_w)))
        return false;
    const int b = f32_batch_rows(p.O, p.I, p.rows, p.norm_w != nullptr);
    if (!b || (p.rows + b - 1) / b > 65535) return false;
    if (name) {
        char buf[80];
        snprintf(buf, sizeof(buf), "mlh::(anonymous namespace)::gemv_f32_batch_kernel<%d>", b);
        *name = buf;
        return true;
    }
    if (b == 4) launch<4>(p, stream);
    else if (b == 8) launch<8>(p, stream);
    else launch<16>(p, stream);
    return true;
}

}  // namespace mlh
