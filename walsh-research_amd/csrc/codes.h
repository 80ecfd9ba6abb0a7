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
// 1/32 (kCodeScale), exactly.  The former byte -> 4 x bf16 table in LDS cost
// a conflicting 8-byte read per lane and 4 weights, a build loop per launch
// and 2 to 10 KB of LDS.  Measured, outputs bitwise equal: the chunk-loop
// SwiGLU and down projection at n_embd 768, 6,007 rows 108.3 -> 103.3 us;
// the launches bound elsewhere (n_embd 4096 linear, 16,384 rows 104.8 ->
// 104.6 us) keep their time.
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
// 8 weights (pairs 4k .. 4k + 3): one group of a 32-column chunk.
__device__ __forceinline__ uint4 codes_bf16x8(uint32_t w, int k) {
    return uint4{(w << (8 * k)) & kCodeMask, (w << (8 * k + 2)) & kCodeMask, (w << (8 * k + 4)) & kCodeMask,
                 (w << (8 * k + 6)) & kCodeMask};
}

}  // namespace walsh
