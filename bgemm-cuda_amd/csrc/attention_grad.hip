// Training both attention products on batches of [N][M] matrices, fp16 in and out, fp32 sums (tests/python/bert/bert.py:245-259 as
// autograd differentiates it, tests/python/bgemm_linear.py:28-42, 64-86):
//
//   scores = sign(A) sign(B)^T     grad_A[n,:] = sum_m G[n,m] sign(B)[m,:]          grad_B[m,:] = sum_n G[n,m] sign(A)[n,:]
//   context = P01 sign(V)          grad_P[n,m] = half(sum_c G[n,c] sign(V)[m,c]) / 2   grad_V[m,:] = sum_n w(P)[n,m] G[n,:]
//                                  w = 1, and 0.5 where P is 0
//
// with A, B, V of D columns.  As separate kernels (sign, the weights w in six elementwise passes over [N][M], four library products,
// the halving, copies of the head-split gradients) 12 heads of 64, 4 x 512 tokens, took 20 launches and a dozen passes over 25 MB;
// here each product pair is one launch that reads or writes an [N][M] matrix once a product, in its own order, and the gradients
// leave in the operands' strides.  What is left is that traffic: the contraction is D = 32 .. 128 long on one side, far below what
// the matrix cores could do in the time.  A training step of both products is that of the host, 160 us in all; of its 68 us of kernels
// those here take 31 (context) and 19 us (scores), neither bandwidth's (3.1 and 5.3
// TB/s counted) nor the matrix cores' (5 % busy): waves wait for 47 and 44 % of their cycles, and LDS, where fragments that lie across
// the rows are read two bytes a lane, is active for 18 and 33 % of the compute units' time.
#include "common.h"

namespace bgemm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

// [outer][inner][rows][D], D dense.
struct HeadView { const __half* p; int64_t so, si, row; };

struct AttnGradArgs {
    const __half* m;                  // [batch][N][M], dense: G of the scores, or P
    HeadView a, b, ga, gb;            // scores: A, B and their gradients.  context: a = G, b = V, gb = grad_V
    __half* gp;                       // context: grad_P, dense
    int N, M, inner, first;           // first: blocks a matrix of the first kind
    int per_batch;                    // blocks a matrix
};

constexpr int AG_ROW = 72;            // staged row of 64 halves, padded by a 16-byte unit

__device__ __forceinline__ __half* head_at(const HeadView& v, const int z, const int inner)
{
    return const_cast<__half*>(v.p) + (z / inner) * v.so + (z % inner) * v.si;
}

// Two fp16 numbers -> their signs; zeros and NaN give 0.
__device__ __forceinline__ unsigned sign_pair(const unsigned x)
{
    auto one = [](const unsigned b) { return ((b & 0x7fffu) - 1u < 0x7c00u ? 0x3c00u : 0u) | (b & 0x8000u); };
    return one(x & 0xffffu) | one(x >> 16) << 16;
}
// Two entries of P -> their weights.
__device__ __forceinline__ unsigned weight_pair(const unsigned x)
{
    auto one = [](const unsigned b) { return (b & 0x7fffu) - 1u < 0x7c00u ? 0x3c00u : 0x3800u; };
    return one(x & 0xffffu) | one(x >> 16) << 16;
}
__device__ __forceinline__ uint4 sign8(const uint4 x) { return make_uint4(sign_pair(x.x), sign_pair(x.y), sign_pair(x.z), sign_pair(x.w)); }
__device__ __forceinline__ float16v mma(const half8 a, const half8 b, const float16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

// out[i,:] = sum_r X[i,r] Y[r,:] for the 64 rows i of a block: X is m, or its transpose (TRANS).  64 of r at a time go through LDS,
// the next 64 on their way in registers; two waves share 32 rows and halve the contraction, so that a fragment of X serves all of
// Y's column tiles.  Columns come out of LDS two bytes a lane.
template <int DT, bool TRANS, bool WEIGHTS>
__device__ __forceinline__ void tall_product(const AttnGradArgs& a, const HeadView& yv, const HeadView& ov, const int z, const int i0, unsigned char* smem)
{
    constexpr int D = DT * 32, YROW = D + 8, UNITS = D / 8;
    __half* const xs = reinterpret_cast<__half*>(smem);
    __half* const ys = xs + 64 * AG_ROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c = lane & 31, it = wave & 1, part = wave >> 1;
    const int rows = TRANS ? a.M : a.N, len = TRANS ? a.N : a.M;
    const __half* const x = a.m + (int64_t)z * a.N * a.M;
    const __half* const y = head_at(yv, z, a.inner);
    const int xr = tid >> 2, xc = (tid & 3) * 16;

    uint4 xreg[2], yreg[DT];
    auto load = [&](const int r0) {
        const int row = (TRANS ? r0 : i0) + xr;
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int col = (TRANS ? i0 : r0) + xc + 8 * p;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (row < a.N) {
                const __half* const from = x + (int64_t)row * a.M + col;
                if (col + 8 <= a.M) {
                    __builtin_memcpy(&v, from, 16);
                    if constexpr (WEIGHTS) v = make_uint4(weight_pair(v.x), weight_pair(v.y), weight_pair(v.z), weight_pair(v.w));
                } else {
                    unsigned d[4] = {0, 0, 0, 0};
#pragma unroll
                    for (int e = 0; e < 7; e++)
                        if (col + e < a.M) {
                            const unsigned b = __half_as_ushort(from[e]);
                            d[e >> 1] |= (WEIGHTS ? weight_pair(b) & 0xffffu : b) << (16 * (e & 1));
                        }
                    v = make_uint4(d[0], d[1], d[2], d[3]);
                }
            }
            xreg[p] = v;
        }
#pragma unroll
        for (int j = 0; j < DT; j++) {
            const int u = tid + 256 * j, r = r0 + u / UNITS;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (r < len) v = *reinterpret_cast<const uint4*>(y + r * yv.row + u % UNITS * 8);
            yreg[j] = v;
        }
    };

    float16v acc[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.f;
    load(0);
#pragma unroll 1
    for (int r0 = 0; r0 < len; r0 += 64) {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 2; p++) *reinterpret_cast<uint4*>(xs + xr * AG_ROW + xc + 8 * p) = xreg[p];
#pragma unroll
        for (int j = 0; j < DT; j++) {
            const int u = tid + 256 * j;
            *reinterpret_cast<uint4*>(ys + u / UNITS * YROW + u % UNITS * 8) = WEIGHTS ? yreg[j] : sign8(yreg[j]);
        }
        __syncthreads();
        if (r0 + 64 < len) load(r0 + 64);
        const _Float16* const xf = reinterpret_cast<const _Float16*>(xs);
        const _Float16* const yf = reinterpret_cast<const _Float16*>(ys);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int r = part * 32 + s * 16 + 8 * h;
            half8 xv;
            if constexpr (TRANS) {
#pragma unroll
                for (int e = 0; e < 8; e++) xv[e] = xf[(r + e) * AG_ROW + it * 32 + c];
            } else xv = *reinterpret_cast<const half8*>(xf + (it * 32 + c) * AG_ROW + r);
#pragma unroll
            for (int t = 0; t < DT; t++) {
                half8 yv8;
#pragma unroll
                for (int e = 0; e < 8; e++) yv8[e] = yf[(r + e) * YROW + t * 32 + c];
                acc[t] = mma(yv8, xv, acc[t]);
            }
        }
    }
    __syncthreads();
    float* const meet = reinterpret_cast<float*>(smem) + it * (DT * 1024) + lane;
    if (part)
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) meet[(t * 16 + v) * 64] = acc[t][v];
    __syncthreads();
    const int i = i0 + it * 32 + c;
    if (part || i >= rows) return;
    __half* const out = head_at(ov, z, a.inner) + i * ov.row;
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            union { __half x[4]; uint2 u; } pk;
#pragma unroll
            for (int e = 0; e < 4; e++) pk.x[e] = __float2half_rn(acc[t][4 * g + e] + meet[(t * 16 + 4 * g + e) * 64]);
            *reinterpret_cast<uint2*>(out + t * 32 + 8 * g + 4 * h) = pk.u;
        }
}

// 64 x 64 of grad_P: the operands are fragments as they lie, the result goes through LDS so that it leaves in pieces of 16 bytes.
template <int DT>
__device__ __forceinline__ void probs_tile(const AttnGradArgs& a, const int z, const int n0, const int m0, unsigned char* smem)
{
    __half* const stage = reinterpret_cast<__half*>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c = lane & 31, nt = wave & 1, mt = wave >> 1;
    const __half* const g = head_at(a.a, z, a.inner) + min(n0 + nt * 32 + c, a.N - 1) * a.a.row + 8 * h;
    const __half* const v = head_at(a.b, z, a.inner) + min(m0 + mt * 32 + c, a.M - 1) * a.b.row + 8 * h;
    float16v acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.f;
#pragma unroll
    for (int s = 0; s < 2 * DT; s++) {
        const uint4 x = sign8(*reinterpret_cast<const uint4*>(v + 16 * s));
        half8 vf;
        __builtin_memcpy(&vf, &x, 16);
        acc = mma(vf, *reinterpret_cast<const half8*>(g + 16 * s), acc);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        union { __half x[4]; uint2 u; } pk;
#pragma unroll
        for (int e = 0; e < 4; e++) pk.x[e] = __float2half_rn(__half2float(__float2half_rn(acc[4 * q + e])) * 0.5f);
        *reinterpret_cast<uint2*>(stage + (nt * 32 + c) * AG_ROW + mt * 32 + 8 * q + 4 * h) = pk.u;
    }
    __syncthreads();
    const int n = n0 + (tid >> 2);
    if (n >= a.N) return;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int at = (tid & 3) * 16 + 8 * p, m = m0 + at;
        __half* const to = a.gp + ((int64_t)z * a.N + n) * a.M + m;
        const __half* const from = stage + (tid >> 2) * AG_ROW + at;
        if (m + 8 <= a.M) __builtin_memcpy(to, from, 16);
        else
#pragma unroll
            for (int e = 0; e < 7; e++)
                if (m + e < a.M) to[e] = from[e];
    }
}

template <int DT> constexpr int ag_lds() { return (64 * AG_ROW + 64 * (DT * 32 + 8)) * 2 > DT * 8192 ? (64 * AG_ROW + 64 * (DT * 32 + 8)) * 2 : DT * 8192; }

// A matrix's blocks are neighbours: its second reading finds it in the caches.
template <int DT>
__global__ __launch_bounds__(256) void scores_grad_kernel(const AttnGradArgs a)
{
    __shared__ __align__(16) unsigned char smem[ag_lds<DT>()];
    const int z = blockIdx.x / a.per_batch, t = blockIdx.x % a.per_batch;
    if (t < a.first) tall_product<DT, false, false>(a, a.b, a.ga, z, t * 64, smem);
    else tall_product<DT, true, false>(a, a.a, a.gb, z, (t - a.first) * 64, smem);
}

template <int DT>
__global__ __launch_bounds__(256) void context_grad_kernel(const AttnGradArgs a)
{
    __shared__ __align__(16) unsigned char smem[ag_lds<DT>()];
    const int z = blockIdx.x / a.per_batch, t = blockIdx.x % a.per_batch;
    if (t < a.first) return tall_product<DT, true, true>(a, a.a, a.gb, z, t * 64, smem);
    const int mb = (a.M + 63) / 64, u = t - a.first;
    probs_tile<DT>(a, z, u / mb * 64, u % mb * 64, smem);
}

}  // namespace bgemm

using namespace bgemm;

// strides: outer, inner and row stride, in elements, of a, b, grad_a and grad_b.
static int attention_backward(const char* who, const bool context, const void* m, const void* a, const void* b, const int64_t* strides, const int64_t batch,
                              const int64_t inner, const int64_t N, const int64_t M, const int64_t D, void* grad_a, void* grad_b, void* grad_p, void* stream)
{
    if (batch < 1 || inner < 1 || batch % inner || N < 1 || M < 1 || N > (1 << 24) || M > (1 << 24) || D < 32 || D > 128 || D % 32)
        return fail(BGEMM_EINVAL, "%s: %lld (%lld) matrices of %lld x %lld, %lld columns", who, (long long)batch, (long long)inner, (long long)N,
                    (long long)M, (long long)D);
    if (!a || !b || !strides || (!context && !m) || (context && grad_b && !m)) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)grad_a | (uintptr_t)grad_b) & 15 || ((uintptr_t)m | (uintptr_t)grad_p) & 1)
        return fail(BGEMM_EALIGN, "%s: operands must be 16-byte aligned", who);
    for (int i = 0; i < 12; i++)
        if (strides[i] % 8) return fail(BGEMM_EALIGN, "%s: strides must be multiples of 8", who);
    const int64_t nb = cdiv(N, 64), mb = cdiv(M, 64);
    AttnGradArgs g = {};
    auto view = [&](const void* p, const int i) { return HeadView{(const __half*)p, strides[3 * i], strides[3 * i + 1], strides[3 * i + 2]}; };
    g.m = (const __half*)m; g.a = view(a, 0); g.b = view(b, 1); g.ga = view(grad_a, 2); g.gb = view(grad_b, 3); g.gp = (__half*)grad_p;
    g.N = (int)N; g.M = (int)M; g.inner = (int)inner;
    const int64_t first = context ? (grad_b ? mb : 0) : (grad_a ? nb : 0), second = context ? (grad_p ? nb * mb : 0) : (grad_b ? mb : 0);
    if (first + second == 0) return BGEMM_OK;
    if (batch > 0x7fffffffLL / (first + second)) return fail(BGEMM_EINVAL, "%s: too many blocks", who);
    g.first = (int)first; g.per_batch = (int)(first + second);
    const dim3 grid((unsigned)(batch * g.per_batch)), block(256);
    const hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto scores, auto ctx) {
        if (context) hipLaunchKernelGGL(ctx, grid, block, 0, st, g);
        else hipLaunchKernelGGL(scores, grid, block, 0, st, g);
    };
    switch (D / 32) {
    case 1: go(scores_grad_kernel<1>, context_grad_kernel<1>); break;
    case 2: go(scores_grad_kernel<2>, context_grad_kernel<2>); break;
    case 3: go(scores_grad_kernel<3>, context_grad_kernel<3>); break;
    default: go(scores_grad_kernel<4>, context_grad_kernel<4>); break;
    }
    return check_launch(who);
}

extern "C" int bgemm_scores_backward(const void* grad_scores, const void* a, const void* b, const int64_t* strides, int64_t batch, int64_t inner,
                                     int64_t N, int64_t M, int64_t D, void* grad_a, void* grad_b, void* stream)
{
    return attention_backward("bgemm_scores_backward", false, grad_scores, a, b, strides, batch, inner, N, M, D, grad_a, grad_b, nullptr, stream);
}

extern "C" int bgemm_context_backward(const void* probs, const void* grad_context, const void* value, const int64_t* strides, int64_t batch, int64_t inner,
                                      int64_t N, int64_t M, int64_t D, void* grad_probs, void* grad_value, void* stream)
{
    return attention_backward("bgemm_context_backward", true, probs, grad_context, value, strides, batch, inner, N, M, D, nullptr, grad_value, grad_probs,
                              stream);
}
