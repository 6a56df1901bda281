// Element-to-bit helpers shared by the pack kernels and by the GEMM kernels that read
// unpacked activations themselves.
#pragma once
#include "common.h"
#include <type_traits>

namespace bgemm {

__device__ __forceinline__ uint16_t half_bits(const float f)
{
    return __half_as_ushort(__float2half_rn(f));
}

// Sign (and nonzero) bits of eight fp16 bit patterns, element e at bit 7 - e.
__device__ __forceinline__ void bits8(const uint16_t (&h)[8], uint32_t& sg, uint32_t& nz)
{
    sg = 0; nz = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        sg |= (uint32_t)(h[e] >> 15) << (7 - e);
        nz |= (uint32_t)((h[e] & 0x7fff) != 0) << (7 - e);
    }
}

// The same for eight fp16 as they come out of one 16-byte load (element 2i in the low half of word i),
// two halves at a time: a half is nonzero iff adding 0x7fff to its low 15 bits reaches bit 15.
__device__ __forceinline__ void bits8(const uint4 v, uint32_t& sg, uint32_t& nz)
{
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    sg = 0; nz = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t s = d[i] & 0x80008000u;
        const uint32_t u = d[i] & 0x7fff7fffu;
        const uint32_t z = ((u + 0x7fff7fffu) | u) & 0x80008000u;
        sg |= (s >> (8 + 2 * i)) | (s >> (25 + 2 * i));          // low half -> bit 7 - 2i, high half -> bit 6 - 2i
        nz |= (z >> (8 + 2 * i)) | (z >> (25 + 2 * i));
    }
    sg &= 0xffu; nz &= 0xffu;
}

// Which magnitudes (fp32 bit patterns without the sign) count as nonzero: lo .. lo + span.
struct NonzeroRule { uint32_t lo, span; };
// of a value's fp16 rounding (`.to(torch.half)`): zero up to and including 2^-25, half the smallest fp16 number, a tie that goes to even
constexpr uint32_t HALF_NONZERO = 0x33000001u, INF_BITS = 0x7f800000u;
__host__ __device__ static inline NonzeroRule nonzero_half() { return {HALF_NONZERO, 0x7fffffffu - HALF_NONZERO}; }
// the same as torch.sign has it, for which NaN is zero, and that of the fp32 value itself
__host__ __device__ static inline NonzeroRule nonzero_sign_half() { return {HALF_NONZERO, INF_BITS - HALF_NONZERO}; }
__host__ __device__ static inline NonzeroRule nonzero_sign_float() { return {1u, INF_BITS - 1u}; }

// Sign (and nonzero) bits of eight fp32 values, element e at bit 7 - e (rounding to fp16 keeps the sign).
__device__ __forceinline__ void bits8(const float (&f)[8], const NonzeroRule rule, uint32_t& sg, uint32_t& nz)
{
    sg = 0; nz = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const uint32_t u = __float_as_uint(f[e]);
        sg = (sg << 1) | (u >> 31);
        nz = (nz << 1) | (uint32_t)((u & 0x7fffffffu) - rule.lo <= rule.span);
    }
}

// Eight consecutive elements of a source row as loaded: one 16-byte load (fp16) or two (fp32), at element alignment
// (the hardware takes vector loads at any address).
template <bool F32> struct Raw8 { uint4 v[F32 ? 2 : 1]; };

template <bool F32>
__device__ __forceinline__ Raw8<F32> load_raw8(const void* row, const int64_t k)
{
    typedef typename std::conditional<F32, uint32_t, uint16_t>::type E;
    Raw8<F32> r;
    __builtin_memcpy(&r, reinterpret_cast<const E*>(row) + k, sizeof r);
    return r;
}

// Their sign and nonzero bits, element e at bit 7 - e, after subtracting the zero point if there is one.
template <bool F32>
__device__ __forceinline__ void bits8(const Raw8<F32>& r, const bool centred, const float zf, const NonzeroRule rule, uint32_t& sg, uint32_t& nz)
{
    if constexpr (F32) {
        const uint32_t d[8] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w, r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w};
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = centred ? __fsub_rn(__uint_as_float(d[e]), zf) : __uint_as_float(d[e]);
        bits8(f, rule, sg, nz);
    } else if (centred) {
        const uint32_t d[4] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w};
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; e++)
            f[e] = __fsub_rn(__half2float(__ushort_as_half((uint16_t)(d[e >> 1] >> (16 * (e & 1))))), zf);
        bits8(f, rule, sg, nz);
    } else
        bits8(r.v[0], sg, nz);
}

// fp16 bit patterns of elements k0 .. k0 + 7 of one source row (fp16, or fp32 rounded to fp16 as
// `.to(torch.half)` rounds), after subtracting the zero point if there is one; elements from K on
// read as +0.0.  `row` points at the row's first element.
__device__ __forceinline__ void load8_as_half(const void* row, const bool f32, const int64_t k0, const int64_t K,
                                              const bool centred, const float zf, uint16_t (&h)[8])
{
#pragma unroll
    for (int e = 0; e < 8; e++) h[e] = 0;
    if (k0 >= K) return;
    if (f32) {
        const float* p = reinterpret_cast<const float*>(row) + k0;
        if (k0 + 8 <= K && (((uintptr_t)p) & 15) == 0) {
            const float4 u = *reinterpret_cast<const float4*>(p), v = *reinterpret_cast<const float4*>(p + 4);
            const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; e++) h[e] = half_bits(centred ? __fsub_rn(f[e], zf) : f[e]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) if (k0 + e < K) h[e] = half_bits(centred ? __fsub_rn(p[e], zf) : p[e]);
        }
    } else {
        const uint16_t* p = reinterpret_cast<const uint16_t*>(row) + k0;
        if (k0 + 8 <= K && (((uintptr_t)p) & 15) == 0) {
            const uint4 v = *reinterpret_cast<const uint4*>(p);
            h[0] = v.x & 0xffff; h[1] = v.x >> 16; h[2] = v.y & 0xffff; h[3] = v.y >> 16;
            h[4] = v.z & 0xffff; h[5] = v.z >> 16; h[6] = v.w & 0xffff; h[7] = v.w >> 16;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) if (k0 + e < K) h[e] = p[e];
        }
        if (centred) {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (k0 + e < K) h[e] = half_bits(__fsub_rn(__half2float(__ushort_as_half(h[e])), zf));
        }
    }
}

// The 32 x 32 bit matrix held by the 32 lanes of a wave half, transposed in registers with five masked exchanges: lane i's
// bit j becomes lane j's bit i.
__device__ __forceinline__ unsigned transpose32(unsigned w, const int lane)
{
#pragma unroll
    for (int j = 16; j >= 1; j >>= 1) {
        const unsigned m = j == 16 ? 0x0000ffffu : j == 8 ? 0x00ff00ffu : j == 4 ? 0x0f0f0f0fu : j == 2 ? 0x33333333u : 0x55555555u;
        const unsigned other = __shfl_xor(w, j);
        w = (lane & j) ? (w & (m << j)) | ((other >> j) & m) : (w & m) | ((other & m) << j);
    }
    return w;
}

// Byte of the tile that holds elements 8c .. 8c + 7 of tile row 0 (add 16 per row): word c >> 2 of the
// row goes to slot h * 32 + r, position q; the row's first element is the word's most significant bit,
// i.e. byte 3 of the little-endian word.
__device__ __forceinline__ int tile_byte_of_chunk(const int c)
{
    return (((c >> 4) * 32) * 4 + ((c >> 2) & 3)) * 4 + (3 - (c & 3));
}

}  // namespace bgemm
