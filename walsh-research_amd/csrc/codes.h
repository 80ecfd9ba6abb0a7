// Ternary weight codes as the kernels hold them, and their expansion.
#pragma once

#include "common.h"

namespace walsh {

// A ternary weight is stored as the top two bits (sign, exponent's high bit)
// of the float it stands for: 00 = 0, 01 = +2.0 (0x4000 in bf16, 0x40000000
// in float32), 11 = -2.0.  A 32-bit word holds 16 codes as 8 pairs, pair p at
// bits (15 - 2p, 14 - 2p) of both halves, so a shift by 2p and one mask give
// a register with two bf16 weights: two VALU operations per pair, no table.
// The factor 2 is a power of two and is taken back with the transforms'
// 1/32 (kCodeScale), exactly, but float32 sums reach infinity one power of two
// earlier than with +-1 weights (six in hadamard_wide3_kernel, whose table held
// +-1/32).  A byte -> 4 x bf16 table in LDS costs a conflicting 8-byte read per
// lane and 4 weights, a build loop per launch and 2 to 10 KB of LDS that the
// wavefront pairs need for themselves.  By itself the change is small: general
// bf16 kernel, 64 -> 64 columns per group at 8,192 rows 292 -> 286 us.
constexpr uint32_t kCodeMask = 0xC000C000u;
constexpr float kCodeScale = 0.015625f;      // 1/32 of the two transforms, 1/2 of the +-2.0 weights
constexpr float kTransformScale = 0.03125f;  // the two transforms alone (dense weights)

// Code bits of packed code v (0, 1, 2 for -1, 0, +1; 3 is never written by
// the packer and counts as +1).
__host__ __device__ __forceinline__ uint32_t code_bits(uint32_t v) { return v == 0 ? 3u : (v == 1 ? 0u : 1u); }

// 4 weights (pairs 2k, 2k + 1) of a word: one group of a 16-column chunk.
__device__ __forceinline__ uint2 codes_bf16x4(uint32_t w, int k) {
    return uint2{(w << (4 * k)) & kCodeMask, (w << (4 * k + 2)) & kCodeMask};
}
__device__ __forceinline__ f32x4 codes_f32x4(uint32_t w, int k) {
    f32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        r[j] = __uint_as_float((w << (4 * k + 2 * (j >> 1) + ((j & 1) ? 0 : 16))) & 0xC0000000u);
    return r;
}
// float32 kernels of the Hadamard layers: a table of the four weights in a byte
// of a word (entry b, element i: the code at bits 7 - 2i, 6 - 2i).  The float32
// products share the VALU's issue, so two operations for each weight's register
// lengthened the launches by 2 to 18% (512 -> 512 features, 16 rows 10.7 ->
// 11.2 us; 2,048 -> 2,048, 16,384 rows 162 -> 184; backward of 4,096 -> 4,096 at
// 1,024 rows 166 -> 190); one 16-byte LDS read gives four.
constexpr int kCodeLut = 256;
__device__ __forceinline__ f32x4 code_lut_entry(uint32_t byte) {
    return f32x4{__uint_as_float((byte << 24) & 0xC0000000u), __uint_as_float((byte << 26) & 0xC0000000u),
                 __uint_as_float((byte << 28) & 0xC0000000u), __uint_as_float((byte << 30) & 0xC0000000u)};
}
// The weights of groups 2m and 2m + 1 of a 16-column chunk's word: its bytes
// hold the first and third (lower half) and the second and fourth (upper half)
// of both.
__device__ __forceinline__ void codes_f32x8(const f32x4 *__restrict__ lut, uint32_t w, int m, f32x4 &w0, f32x4 &w1) {
    const f32x4 lo = lut[(w >> (8 - 8 * m)) & 0xffu], hi = lut[(w >> (24 - 8 * m)) & 0xffu];
    w0 = f32x4{lo[0], hi[0], lo[1], hi[1]};
    w1 = f32x4{lo[2], hi[2], lo[3], hi[3]};
}
// 8 weights (pairs 4k .. 4k + 3): one group of a 32-column chunk.
__device__ __forceinline__ uint4 codes_bf16x8(uint32_t w, int k) {
    return uint4{(w << (8 * k)) & kCodeMask, (w << (8 * k + 2)) & kCodeMask, (w << (8 * k + 4)) & kCodeMask,
                 (w << (8 * k + 6)) & kCodeMask};
}

}  // namespace walsh
