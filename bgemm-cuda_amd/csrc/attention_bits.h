// What the attention kernels share: fp4 operands from words of sign bits.
#pragma once
#include "mfma_engines.h"
#include "pack_bits.h"

namespace bgemm {

constexpr int ATTN_STAGE = 144;       // bytes of a staged row of 64 scores (padded)

// fp4 operands of one word at step s.  A bit that counts stays where it is (0.5, 1, 2; at step 3 it moves to 1.0), five instructions a
// word; the other side has the reciprocals of those values: of a sign x = +-1 (given inverted) as -2 x, so that a sum that starts from
// the sum of x is that of x (1 - 2 b), or of a bit as 1.
__device__ __forceinline__ unsigned attn_bit(const unsigned w, const int s) { return s == 3 ? (w >> 2) & 0x22222222u : w & (0x11111111u << s); }
__device__ __forceinline__ unsigned attn_sign(const unsigned inverted, const int s)
{
    return ((inverted << (3 - s)) & 0x88888888u) | (s == 0 ? 0x66666666u : s == 2 ? 0x22222222u : 0x44444444u);
}
__device__ __forceinline__ unsigned attn_one(const unsigned w, const int s)
{
    return s == 0 ? (w << 2) & 0x44444444u : s == 1 ? w & 0x22222222u : (w >> 2) & (s == 2 ? 0x11111111u : 0x22222222u);
}

// Orders a wave's own LDS accesses for the compiler (LDS executes them in order).
__device__ __forceinline__ void attn_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace bgemm
