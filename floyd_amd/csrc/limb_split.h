// limb_split.h -- the four-limb int8 split of fp32 values (30 bits of the largest
// of a range) that the matrix-core GEMV kernels share (gemv_mfma.hip,
// gemv_batch.hip, the four-limb tiles of qgemm.hip).
#pragma once

#include "mlh_device.h"
#include "mlh_host.h"

namespace mlh {

// The four limbs of 8 elements of x (already scaled by the step's inverse),
// packed as the limb rows store them: lw[L][w] holds limb L of the elements
// at byte positions 4 w .. 4 w + 3 (q8: element order; q4: elements 0,2,4,6 |
// 1,3,5,7, the order in which the nibbles of packed bytes unpack).  The
// balanced base-256 digits of q are the bytes of (q + 0x808080) ^ 0x808080:
// adding 128 to each of the three low digits makes them the plain bytes of
// the sum (each in 0..255), the xor takes the 128 off again in int8, and the
// top byte is L0.  So an element costs a rounding, a conversion, an add and
// an xor, and a 4 x 4 byte transpose by v_perm_b32 gathers the limbs of 4
// elements.
__device__ __forceinline__ void limb_transpose(unsigned e0, unsigned e1, unsigned e2, unsigned e3,
                                               unsigned &l0, unsigned &l1, unsigned &l2,
                                               unsigned &l3) {
    const unsigned a01 = __builtin_amdgcn_perm(e1, e0, 0x06020400u);  // e0.b0 e1.b0 e0.b2 e1.b2
    const unsigned b01 = __builtin_amdgcn_perm(e1, e0, 0x07030501u);  // e0.b1 e1.b1 e0.b3 e1.b3
    const unsigned a23 = __builtin_amdgcn_perm(e3, e2, 0x06020400u);
    const unsigned b23 = __builtin_amdgcn_perm(e3, e2, 0x07030501u);
    l3 = __builtin_amdgcn_perm(a23, a01, 0x05040100u);  // byte 0 of e0..e3
    l2 = __builtin_amdgcn_perm(b23, b01, 0x05040100u);  // byte 1
    l1 = __builtin_amdgcn_perm(a23, a01, 0x07060302u);  // byte 2
    l0 = __builtin_amdgcn_perm(b23, b01, 0x07060302u);  // byte 3
}
// The limbs of 4 elements, one word per limb, in element order.  The integer is
// truncated, not rounded (at 30 bits it is exact for every element within 2^-6
// of the largest), and the xor is done on the transposed words.
__device__ __forceinline__ void split_limbs4(const float (&v4)[4], float step_inv, unsigned &l0,
                                             unsigned &l1, unsigned &l2, unsigned &l3) {
    unsigned e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = (unsigned)((int)(v4[i] * step_inv) + 0x808080);
    limb_transpose(e[0], e[1], e[2], e[3], l0, l1, l2, l3);
    l1 ^= 0x80808080u;
    l2 ^= 0x80808080u;
    l3 ^= 0x80808080u;
}
template <int FMT>
__device__ __forceinline__ void split_limbs8(const float (&v8)[8], float step_inv,
                                             unsigned (&lw)[4][2]) {
    unsigned e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        e[i] = (unsigned)((int)rintf(v8[i] * step_inv) + 0x808080) ^ 0x808080u;
    // q8: bytes in element order; q4: elements 0,2,4,6 | 1,3,5,7
    constexpr int i1 = FMT == kQ4 ? 2 : 1, i2 = FMT == kQ4 ? 4 : 2, i3 = FMT == kQ4 ? 6 : 3;
    constexpr int j0 = FMT == kQ4 ? 1 : 4, j1 = FMT == kQ4 ? 3 : 5, j2 = FMT == kQ4 ? 5 : 6, j3 = 7;
    limb_transpose(e[0], e[i1], e[i2], e[i3], lw[0][0], lw[1][0], lw[2][0], lw[3][0]);
    limb_transpose(e[j0], e[j1], e[j2], e[j3], lw[0][1], lw[1][1], lw[2][1], lw[3][1]);
}

}  // namespace mlh
