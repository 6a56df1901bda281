// Training the binary Linear layer: what its backward pass needs besides the two dense products.
//
//   forward   y[n,m] = half(acc[n,m]) * sw[m] * sa (+ bias[m]),  acc = sum_k sign(x - zpa)[n,k] sign(w - zpw)[m,k]
//   backward  g16 = half((G * sa) * sw[m])                     -> the upstream operand of both dense products
//             grad_sw[m] = sum_n (G * sa) * half(acc)           grad_sa = sum_n,m G * (half(acc) * sw[m])
//             grad_bias[m] = sum_n G
// (tests/python/bgemm_linear.py:479-484 as autograd differentiates it, :149-165).  As separate elementwise and reduction
// kernels this is a dozen passes over [N][M] fp32 matrices.  Here it is one: acc is not kept from the forward pass but
// multiplied again from the two operands' sign bits (a hundredth of the bytes), in the shadow of the read of G.
#include "common.h"
#include "mfma_engines.h"
#include "pack_bits.h"
#include <type_traits>

namespace bgemm {

struct LinearGradArgs {
    const uint4* W; const uint4* X;      // sign bits, tiled
    const void* g;                        // upstream gradient [N][M], fp32 or fp16
    const void* sw; const void* sa;       // parameters, same type
    __half* g16;                          // [N][M]
    float* part;                          // [chunks][3][Mpad]: per row chunk sums of G, (G sa) acc, G (acc sw)
    uint32_t* ticket;
    int64_t N, M, K;
    int NT, KT, MT, rt_per_chunk;
    int64_t mpad;
};

// One 32-bit word of signed fp4 operands at step s: +1.0, or -1.0 where the bit is set, in a nibble each.
__device__ __forceinline__ unsigned pm1_nibbles(const unsigned w, const int s)
{
    return (s == 3 ? w & 0x88888888u : (w << (3 - s)) & 0x88888888u) | 0x22222222u;
}

template <bool F32>
__device__ __forceinline__ float param(const void* p, const int64_t i)
{
    if constexpr (F32) return reinterpret_cast<const float*>(p)[i];
    else return __half2float(reinterpret_cast<const __half*>(p)[i]);
}

// A wave owns 64 columns (weight rows) and walks rt_per_chunk row tiles of 32: a lane holds the two neighbouring columns 2c
// and 2c + 1 of sixteen rows, so G arrives as 8 (fp16: 4) bytes a lane and g16 leaves as 4, a half-wave a whole line; the
// column sums stay in registers to the end.  A row tile's G is requested before its bits are multiplied.
// The operands are signed fp4 (+1 / -1), so the accumulator is the layer's output up to the padding bits of K, which are
// +1 * +1 each: no popcounts, no row terms.  Bound by reading G and writing g16: [8192][3072] fp32
// (150 MB), K = 768, 40.7 us = 3.7 TB/s on three waves a SIMD; with the next tile's G held in registers as well, on two, 54.2.
template <bool F32>
__global__ __launch_bounds__(256, 3) void linear_grad_kernel(const LinearGradArgs a)
{
    typedef typename std::conditional<F32, float, __half>::type E;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, c = lane & 31;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *a.ticket = 0;      // for the kernel that adds the chunks up
    const int mg = blockIdx.x * 4 + wave, chunk = blockIdx.y;
    if ((int64_t)mg * 64 >= a.M) return;
    const int64_t m = (int64_t)mg * 64 + 2 * c, mc = m < a.M - 2 ? m : a.M - 2;      // (M >= 2)
    const bool ok0 = m < a.M, ok1 = m + 1 < a.M, moved = m != mc;                    // the last column of an odd M: loaded as a pair's second
    const float sa = param<F32>(a.sa, 0);
    const float sw0 = ok0 ? param<F32>(a.sw, m) : 0.f, sw1 = ok1 ? param<F32>(a.sw, m + 1) : 0.f;
    const uint4* wp[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int r = 2 * c + j;
        const int64_t rt = mg * 2 + (r >> 5) < a.MT ? mg * 2 + (r >> 5) : a.MT - 1;
        wp[j] = a.W + rt * a.KT * TILE_U4 + (lane & 32) + (r & 31);
    }
    const float pad = (float)((int64_t)a.KT * TILE_KBITS - a.K);
    const bool even = (a.M & 1) == 0;

    typedef typename std::conditional<F32, uint2, uint32_t>::type Pair;
    const int t0 = chunk * a.rt_per_chunk, t1 = min(a.NT, t0 + a.rt_per_chunk);
    float s_b[2] = {0.f, 0.f}, s_w[2] = {0.f, 0.f}, s_a[2] = {0.f, 0.f};
    const bool cols_in = ((int64_t)mg + 1) * 64 <= a.M;
    for (int t = t0; t < t1; t++) {
        Pair g[16];
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int64_t n = (int64_t)t * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
            __builtin_memcpy(&g[v], reinterpret_cast<const E*>(a.g) + (n < a.N ? n : a.N - 1) * a.M + mc, sizeof(Pair));
        }
        const uint4* xp = a.X + (int64_t)t * a.KT * TILE_U4 + lane;
        EngF4::Acc acc[2];
#pragma unroll
        for (int v = 0; v < 16; v++) acc[0][v] = acc[1][v] = -pad;
        for (int kt = 0; kt < a.KT; kt++) {
            const uint4 x = xp[kt * TILE_U4], w0 = wp[0][kt * TILE_U4], w1 = wp[1][kt * TILE_U4];
            const unsigned xd[4] = {x.x, x.y, x.z, x.w}, wd0[4] = {w0.x, w0.y, w0.z, w0.w}, wd1[4] = {w1.x, w1.y, w1.z, w1.w};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                unsigned fx[4], f0[4], f1[4];
#pragma unroll
                for (int q = 0; q < 4; q++) { fx[q] = pm1_nibbles(xd[q], s); f0[q] = pm1_nibbles(wd0[q], s); f1[q] = pm1_nibbles(wd1[q], s); }
                acc[0] = EngF4::mma(EngF4::make(fx), EngF4::make(f0), acc[0]);
                acc[1] = EngF4::mma(EngF4::make(fx), EngF4::make(f1), acc[1]);
            }
        }
        auto finish = [&](auto whole_c) {
            constexpr bool WHOLE = decltype(whole_c)::value;      // every row and column of the wave's piece exists
            __half* const to0 = a.g16 + ((int64_t)t * 32 + 4 * h) * a.M + m;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int r = 8 * (v >> 2) + (v & 3);
                float G0, G1;
                if constexpr (F32) { G0 = __uint_as_float(g[v].x); G1 = __uint_as_float(g[v].y); }
                else { G0 = __half2float(__ushort_as_half((uint16_t)(g[v] & 0xffff))); G1 = __half2float(__ushort_as_half((uint16_t)(g[v] >> 16))); }
                const bool row = WHOLE || (int64_t)t * 32 + r + 4 * h < a.N;
                if (!WHOLE) {
                    G0 = row && ok0 ? (moved ? G1 : G0) : 0.f;
                    G1 = row && ok1 ? G1 : 0.f;
                }
                const float a0 = __half2float(__float2half_rn(acc[0][v])), a1 = __half2float(__float2half_rn(acc[1][v]));
                float p0, p1;                         // (G * sa), then times sw, every step rounded to the parameters' type
                __half h0, h1;
                {
#pragma clang fp contract(off)
                    if constexpr (F32) {
                        p0 = G0 * sa; p1 = G1 * sa;
                        h0 = __float2half_rn(p0 * sw0); h1 = __float2half_rn(p1 * sw1);
                    } else {
                        const _Float16 q0 = (_Float16)G0 * (_Float16)sa, q1 = (_Float16)G1 * (_Float16)sa;
                        const _Float16 r0 = q0 * (_Float16)sw0, r1 = q1 * (_Float16)sw1;
                        p0 = (float)q0; p1 = (float)q1;
                        __half_raw hr; hr.data = r0; h0 = __half(hr); hr.data = r1; h1 = __half(hr);
                    }
                    s_b[0] += G0; s_b[1] += G1;
                }
                s_w[0] += p0 * a0; s_w[1] += p1 * a1;
                s_a[0] += G0 * (a0 * sw0); s_a[1] += G1 * (a1 * sw1);
                __half* const to = to0 + r * a.M;
                if (WHOLE) {
                    *reinterpret_cast<uint32_t*>(to) = (uint32_t)__half_as_ushort(h0) | (uint32_t)__half_as_ushort(h1) << 16;
                } else if (row) {
                    if (ok0) to[0] = h0;
                    if (ok1) to[1] = h1;
                }
            }
        };
        if (even && cols_in && (t + 1) * 32 <= a.N) finish(std::true_type{});
        else finish(std::false_type{});
    }
    float* const part = a.part + (int64_t)chunk * 3 * a.mpad + m;
#pragma unroll
    for (int e = 0; e < 2; e++) {
        s_b[e] += __shfl_xor(s_b[e], 32);
        s_w[e] += __shfl_xor(s_w[e], 32);
        s_a[e] += __shfl_xor(s_a[e], 32);
    }
    if (h == 0) {                                 // (mpad is a multiple of 64: columns past M hold zeros)
        *reinterpret_cast<float2*>(part) = make_float2(s_b[0], s_b[1]);
        *reinterpret_cast<float2*>(part + a.mpad) = make_float2(s_w[0], s_w[1]);
        *reinterpret_cast<float2*>(part + 2 * a.mpad) = make_float2(s_a[0], s_a[1]);
    }
}

// Adds the chunks up: a block of 1024 threads takes 64 columns, sixteen threads a column; the last block to finish adds the
// blocks' shares of the scalar.
template <bool F32>
__global__ __launch_bounds__(1024) void linear_grad_sum_kernel(const float* __restrict__ part, float* __restrict__ block_sa,
                                                              uint32_t* ticket, const int chunks, const int64_t mpad, const int64_t M,
                                                              void* grad_bias, void* grad_sw, void* grad_sa)
{
    __shared__ float sum[3][16][64];
    __shared__ bool last;
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int64_t m = (int64_t)blockIdx.x * 64 + c;
    float s[3] = {0.f, 0.f, 0.f};
    for (int k = q; k < chunks; k += 16)
#pragma unroll
        for (int i = 0; i < 3; i++) s[i] += part[((int64_t)k * 3 + i) * mpad + m];
#pragma unroll
    for (int i = 0; i < 3; i++) sum[i][q][c] = s[i];
    __syncthreads();
    auto put = [](void* to, const int64_t i, const float v) {
        if constexpr (F32) reinterpret_cast<float*>(to)[i] = v;
        else reinterpret_cast<__half*>(to)[i] = __float2half_rn(v);
    };
    if (q < 3) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) t += sum[q][i][c];
        if (q < 2) {
            void* const to = q == 0 ? grad_bias : grad_sw;
            if (to && m < M) put(to, m, t);
        } else {
#pragma unroll
            for (int d = 32; d; d >>= 1) t += __shfl_xor(t, d);
            if (c == 0) {
                __hip_atomic_store(&block_sa[blockIdx.x], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
            }
        }
    }
    __syncthreads();
    if (last && threadIdx.x < 64) {
        float t = 0.f;
        for (unsigned i = threadIdx.x; i < gridDim.x; i += 64) t += __hip_atomic_load(&block_sa[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int d = 32; d; d >>= 1) t += __shfl_xor(t, d);
        if (threadIdx.x == 0 && grad_sa) put(grad_sa, 0, t);
    }
}

// Row tiles a wave walks: enough waves for about three on every SIMD, at most 16 row tiles (the fewer chunks, the less there is to add up).
static int grad_rows_per_chunk(int64_t N, int64_t M)
{
    const int64_t want = row_tiles(N) * cdiv(M, 64) / 3072;
    return (int)(want < 1 ? 1 : want > 16 ? 16 : want);
}

// Sign and nonzero planes of up to two operands -> fp16 matrices of -1, 0, +1.  A wave takes a tile: eight elements (a byte
// of each plane) and one 16-byte store a lane.
struct UnpackJob { const unsigned char* sg; const unsigned char* nz; __half* dst; int64_t rows, K, KT, waves; };

__global__ __launch_bounds__(256) void unpack_signs_kernel(const UnpackJob j0, const UnpackJob j1)
{
    const int lane = threadIdx.x & 63;
    int64_t gw = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const bool first = gw < j0.waves;
    const UnpackJob& j = first ? j0 : j1;
    if (!first) gw -= j0.waves;
    if (gw >= j.waves) return;
    const int64_t rt = gw / j.KT, kt = gw - rt * j.KT;
    const int c = lane & 31;
    const int64_t k = kt * TILE_KBITS + 8 * c;
    if (k >= j.K) return;
    const bool whole = k + 8 <= j.K && (j.K & 7) == 0;
    const unsigned char* const s = j.sg + gw * 1024 + tile_byte_of_chunk(c);
    const unsigned char* const z = j.nz + gw * 1024 + tile_byte_of_chunk(c);
    unsigned sb[16], zb[16];
#pragma unroll
    for (int i = 0; i < 16; i++) { sb[i] = s[(2 * i + (lane >> 5)) * 16]; zb[i] = z[(2 * i + (lane >> 5)) * 16]; }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int64_t row = rt * TILE_ROWS + 2 * i + (lane >> 5);
        if (row >= j.rows) break;
        union { uint32_t w[4]; uint16_t e[8]; uint4 u; } o;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const uint32_t lo = (zb[i] >> (7 - 2 * p) & 1u) * (0x3c00u | (sb[i] >> (7 - 2 * p) & 1u) << 15);
            const uint32_t hi = (zb[i] >> (6 - 2 * p) & 1u) * (0x3c00u | (sb[i] >> (6 - 2 * p) & 1u) << 15);
            o.w[p] = lo | hi << 16;
        }
        uint16_t* const to = reinterpret_cast<uint16_t*>(j.dst) + row * j.K + k;
        if (whole) *reinterpret_cast<uint4*>(to) = o.u;
        else
            for (int e = 0; e < 8 && k + e < j.K; e++) to[e] = o.e[e];
    }
}

// Bi-Real's surrogate on the input gradient: gx * (2 - 2 min(|x - zp|, 1)), every step rounded to fp16 as the separate
// torch kernels round it (tests/python/bgemm_linear.py:186-219).
template <bool F32>
__global__ __launch_bounds__(256) void bireal_grad_kernel(const __half* __restrict__ gx, const void* __restrict__ x, const int64_t ld,
                                                          const void* __restrict__ zp, void* __restrict__ out, const int64_t rows, const int64_t K)
{
    const float z = param<F32>(zp, 0);
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x)
    for (int64_t k = threadIdx.x; k < K; k += 256) {
        const int64_t i = r * K + k;
        const _Float16 xh = (_Float16)__fsub_rn(param<F32>(x, r * ld + k), z);
        const _Float16 ax = (_Float16)fabsf((float)xh);
        const _Float16 cl = ax > (_Float16)1.0f ? (_Float16)1.0f : ax;
        const _Float16 d = (_Float16)2.0f - (_Float16)2.0f * cl;        // both steps exact or one fp16 rounding
        __half_raw hr = __half_raw(gx[i]);
        const _Float16 o = hr.data * d;
        if constexpr (F32) reinterpret_cast<float*>(out)[i] = (float)o;
        else reinterpret_cast<_Float16*>(out)[i] = o;
    }
}

}  // namespace bgemm

using namespace bgemm;

static size_t grad_round(size_t b) { return (b + 255) / 256 * 256; }

extern "C" size_t bgemm_linear_grad_workspace_bytes(int64_t N, int64_t M)
{
    if (N <= 0 || M <= 0) return 0;
    const int64_t chunks = cdiv(row_tiles(N), grad_rows_per_chunk(N, M)), cols = cdiv(M, 64);
    return 256 + grad_round((size_t)cols * 4) + grad_round((size_t)chunks * 3 * cols * 64 * 4);
}

extern "C" int bgemm_linear_grad(const void* W_sign, const void* X_sign, const void* grad_out, int param_dtype, int64_t N, int64_t M,
                                 int64_t K, const void* sw, const void* sa, void* g16, void* grad_bias, void* grad_sw, void* grad_sa,
                                 void* ws, size_t ws_bytes, void* stream)
{
    const char* who = "bgemm_linear_grad";
    if (param_dtype != BGEMM_SRC_F16 && param_dtype != BGEMM_SRC_F32) return fail(BGEMM_EINVAL, "%s: unknown parameter type %d", who, param_dtype);
    if (N < 1 || M < 2 || K < 1 || K >= (1LL << 24) || N > 0x7fffffff || M > 0x7fffffff)
        return fail(BGEMM_EINVAL, "%s: bad shape N=%lld M=%lld K=%lld", who, (long long)N, (long long)M, (long long)K);
    if (!W_sign || !X_sign || !grad_out || !sw || !sa || !g16 || !ws) return fail(BGEMM_ENULL, "%s: null pointer", who);
    const unsigned esz = param_dtype == BGEMM_SRC_F32 ? 4 : 2;
    if (((uintptr_t)W_sign & 15) || ((uintptr_t)X_sign & 15) || ((uintptr_t)g16 & 3) || ((uintptr_t)ws & 255) || ((uintptr_t)grad_out & (esz - 1)))
        return fail(BGEMM_EALIGN, "%s: an operand is not aligned", who);
    if (ws_bytes < bgemm_linear_grad_workspace_bytes(N, M)) return fail(BGEMM_EWORKSPACE, "%s: workspace of %zu bytes is too small", who, ws_bytes);
    LinearGradArgs a;
    a.W = (const uint4*)W_sign; a.X = (const uint4*)X_sign; a.g = grad_out; a.sw = sw; a.sa = sa; a.g16 = (__half*)g16;
    a.N = N; a.M = M; a.K = K; a.NT = (int)row_tiles(N); a.KT = (int)k_tiles(K); a.MT = (int)row_tiles(M);
    a.rt_per_chunk = grad_rows_per_chunk(N, M);
    const int64_t chunks = cdiv(a.NT, a.rt_per_chunk), cols = cdiv(M, 64);
    if (chunks > 65535) return fail(BGEMM_EINVAL, "%s: too many rows", who);
    a.mpad = cols * 64;
    a.ticket = (uint32_t*)ws;
    float* const block_sa = (float*)((char*)ws + 256);
    a.part = (float*)((char*)ws + 256 + grad_round((size_t)cols * 4));
    const hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)cdiv(cols, 4), (unsigned)chunks);
    if (param_dtype == BGEMM_SRC_F32) {
        hipLaunchKernelGGL(linear_grad_kernel<true>, grid, dim3(256), 0, st, a);
        hipLaunchKernelGGL(linear_grad_sum_kernel<true>, dim3((unsigned)cols), dim3(1024), 0, st, a.part, block_sa, a.ticket, (int)chunks, a.mpad, M,
                           grad_bias, grad_sw, grad_sa);
    } else {
        hipLaunchKernelGGL(linear_grad_kernel<false>, grid, dim3(256), 0, st, a);
        hipLaunchKernelGGL(linear_grad_sum_kernel<false>, dim3((unsigned)cols), dim3(1024), 0, st, a.part, block_sa, a.ticket, (int)chunks, a.mpad, M,
                           grad_bias, grad_sw, grad_sa);
    }
    return check_launch(who);
}

static int unpack_job(UnpackJob* j, const void* sg, const void* nz, void* dst, int64_t rows, int64_t K, const char* who)
{
    j->sg = (const unsigned char*)sg; j->nz = (const unsigned char*)nz; j->dst = (__half*)dst;
    j->rows = rows; j->K = K; j->KT = k_tiles(K); j->waves = dst ? row_tiles(rows) * j->KT : 0;
    if (!dst) return BGEMM_OK;
    if (rows < 1 || K < 1) return fail(BGEMM_EINVAL, "%s: bad shape rows=%lld K=%lld", who, (long long)rows, (long long)K);
    if (!sg || !nz) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (((uintptr_t)dst & 15)) return fail(BGEMM_EALIGN, "%s: destination not 16-byte aligned", who);
    return BGEMM_OK;
}

extern "C" int bgemm_unpack_signs_pair(const void* sign_a, const void* nonzero_a, void* dst_a, int64_t rows_a, const void* sign_b,
                                       const void* nonzero_b, void* dst_b, int64_t rows_b, int64_t K, void* stream)
{
    const char* who = "bgemm_unpack_signs_pair";
    UnpackJob j0, j1;
    int rc = unpack_job(&j0, sign_a, nonzero_a, dst_a, rows_a, K, who);
    if (!rc) rc = unpack_job(&j1, sign_b, nonzero_b, dst_b, rows_b, K, who);
    if (rc) return rc;
    const int64_t blocks = cdiv(j0.waves + j1.waves, 4);
    if (blocks == 0) return BGEMM_OK;
    if (blocks > 0x7fffffffLL) return fail(BGEMM_EINVAL, "%s: operand too large", who);
    hipLaunchKernelGGL(unpack_signs_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, j0, j1);
    return check_launch(who);
}

extern "C" int bgemm_bireal_grad(const void* grad_x16, const void* x, int x_dtype, int64_t ld, const void* zero_point, void* out,
                                 int64_t rows, int64_t K, void* stream)
{
    const char* who = "bgemm_bireal_grad";
    if (x_dtype != BGEMM_SRC_F16 && x_dtype != BGEMM_SRC_F32) return fail(BGEMM_EINVAL, "%s: unknown type %d", who, x_dtype);
    if (rows < 0 || K < 0 || ld < K) return fail(BGEMM_EINVAL, "%s: bad shape rows=%lld K=%lld ld=%lld", who, (long long)rows, (long long)K, (long long)ld);
    if (rows == 0 || K == 0) return BGEMM_OK;
    if (!grad_x16 || !x || !zero_point || !out) return fail(BGEMM_ENULL, "%s: null pointer", who);
    const dim3 grid((unsigned)(rows < 16384 ? rows : 16384));
    if (x_dtype == BGEMM_SRC_F32)
        hipLaunchKernelGGL(bireal_grad_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, (const __half*)grad_x16, x, ld, zero_point, out, rows, K);
    else
        hipLaunchKernelGGL(bireal_grad_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, (const __half*)grad_x16, x, ld, zero_point, out, rows, K);
    return check_launch(who);
}
