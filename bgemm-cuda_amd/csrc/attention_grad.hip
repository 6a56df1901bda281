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
// the matrix cores could do in the time.  48 matrices of 512 x 512, D = 64, launches in turn: scores 18.9 -> 12.0 us, context 28.8 -> 13.8, the
// latter's two halves 8.8 (25 MB written) and 8.6 (25 MB read) alone.  Blocks of a matrix on one XCD: dealt round robin, an XCD reads the
// same eighth of every row, from few of its L2's channels, and the scores' second reading comes from beyond its L2 (192 matrices: 43 and 51
// us for 63 and 59; a few long ones are the same).  Fragments that lie across the rows come out of LDS by transposing reads (two-byte ones: 96 for
// 24), and grad_P leaves from registers, 128 bytes of a row a half-wave.  A block's steps are a chain: loads, signs or weights, LDS, products.  So
// signs are seven instructions a word (is_signed; with packed minima, which the compiler takes apart into compares and selects, twice as
// many: 4 x 2048^2, D = 64, scores 34.9 for 29.3), and weights are formed on the way into LDS, not where they are loaded (V's gradient alone
// 45.9 for 32.5).  Waves still wait for 43 (scores) and 48 % of their cycles, vector units are busy for 23 and 21 %, the matrix cores 6.  Not ahead: stretches of 128 rows, two of them in flight, eight waves a block with stretches of their own and no barrier
// before the sums meet.
#include "common.h"
#include <type_traits>

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
    int batch, chunks;                // 64 columns of grad_P each, a block
};

__device__ __forceinline__ __half* head_at(const HeadView& v, const int z, const int inner)
{
    return const_cast<__half*>(v.p) + (z / inner) * v.so + (z % inner) * v.si;
}

// Two fp16 numbers at a time: bit 15 of each where it is neither zero nor NaN.  (Sums that stay within their halves: 1 .. 0x7c00 are those
// that 0x7fff carries into bit 15 and 0x3ff does not.)
__device__ __forceinline__ unsigned is_signed(const unsigned x)
{
    const unsigned m = x & 0x7fff7fffu;
    return (m + 0x7fff7fffu) & ~(m + 0x03ff03ffu) & 0x80008000u;
}
// Their signs; zeros and NaN give 0.
__device__ __forceinline__ unsigned sign_pair(const unsigned x) { return (is_signed(x) >> 15) * 0x3c00u | (x & 0x80008000u); }
// Two entries of P -> their weights.
__device__ __forceinline__ unsigned weight_pair(const unsigned x) { return 0x38003800u + (is_signed(x) >> 5); }
__device__ __forceinline__ uint4 sign8(const uint4 x) { return make_uint4(sign_pair(x.x), sign_pair(x.y), sign_pair(x.z), sign_pair(x.w)); }
__device__ __forceinline__ uint4 weight8(const uint4 x) { return make_uint4(weight_pair(x.x), weight_pair(x.y), weight_pair(x.z), weight_pair(x.w)); }
// Eight rows of a column each: lane (c, h) gets rows row0 + 8 h .. + 7 of column col0 + c of a staged matrix, by two reads that transpose 4 x 4
// elements among sixteen lanes (lane i of sixteen names row i / 4 and the four columns from 4 (i % 4) on, and gets column i).
typedef short short4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ half8 column8(const _Float16* const staged, const int stride, const int row0, const int col0, const int lane)
{
    typedef __attribute__((address_space(3))) short4v* lds4;
    const int i = lane & 15, g = lane >> 4;
    const _Float16* const at = staged + (row0 + 8 * (g >> 1) + (i >> 2)) * stride + col0 + 16 * (g & 1) + 4 * (i & 3);
    union { short4v s[2]; half8 h; } u;
#pragma unroll
    for (int k = 0; k < 2; k++) u.s[k] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(__attribute__((address_space(3))) void*)(at + 4 * k * stride));
    return u.h;
}
__device__ __forceinline__ float16v mma(const half8 a, const half8 b, const float16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

// out[i,:] = sum_r X[i,r] Y[r,:] for the 64 rows i of a block: X is m, or its transpose (TRANS).  64 of r at a time go through LDS,
// the next 64 on their way in registers; two waves share 32 rows and halve the contraction, so that a fragment of X serves all of
// Y's column tiles.  What lies across the rows comes out of LDS by reads that transpose.
constexpr int AG_STEP = 64;
template <int DT, bool TRANS, bool WEIGHTS>
__device__ __forceinline__ void tall_product(const AttnGradArgs& a, const HeadView& yv, const HeadView& ov, const int z, const int i0, unsigned char* smem)
{
    constexpr int D = DT * 32, YROW = D + 8, UNITS = D / 8;
    constexpr int XW = TRANS ? 8 : AG_STEP / 8, XROW = XW * 8 + 8, XLOADS = AG_STEP * 64 / 8 / 256, YLOADS = AG_STEP * UNITS / 256;      // 16-byte units of a staged row of X
    __half* const xs = reinterpret_cast<__half*>(smem);
    __half* const ys = xs + (TRANS ? AG_STEP : 64) * XROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c = lane & 31, it = wave & 1, part = wave >> 1;
    const int rows = TRANS ? a.M : a.N, len = TRANS ? a.N : a.M;
    const __half* const x = a.m + (int64_t)z * a.N * a.M;
    const __half* const y = head_at(yv, z, a.inner);

    uint4 xreg[XLOADS], yreg[YLOADS];
    auto load = [&](const int r0) {
#pragma unroll
        for (int p = 0; p < XLOADS; p++) {
            const int u = tid + 256 * p, row = (TRANS ? r0 : i0) + u / XW, col = (TRANS ? i0 : r0) + u % XW * 8;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (row < a.N && col < a.M) {
                const __half* const from = x + (int64_t)row * a.M + col;
                if (col + 8 <= a.M) __builtin_memcpy(&v, from, 16);
                else if (a.M >= 8) {
                    // a row's last elements: its last eight, those before them shifted out
                    uint64_t d[2];
                    __builtin_memcpy(d, from - (col + 8 - a.M), 16);
                    const int bits = (col + 8 - a.M) * 16;
                    d[0] = bits < 64 ? d[0] >> bits | d[1] << (64 - bits) : d[1] >> (bits - 64);
                    d[1] = bits < 64 ? d[1] >> bits : 0;
                    __builtin_memcpy(&v, d, 16);
                } else {
                    unsigned d[4] = {0, 0, 0, 0};
#pragma unroll
                    for (int e = 0; e < 7; e++)
                        if (col + e < a.M) d[e >> 1] |= (unsigned)__half_as_ushort(from[e]) << (16 * (e & 1));
                    v = make_uint4(d[0], d[1], d[2], d[3]);
                }
            }
            xreg[p] = v;
        }
#pragma unroll
        for (int j = 0; j < YLOADS; j++) {
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
    for (int r0 = 0; r0 < len; r0 += AG_STEP) {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < XLOADS; p++) {
            // (weights here and not where they are loaded, which would wait for each load; entries that do not exist weigh something, in rows
            // of the output that do not exist either or against zeros of Y)
            const int u = tid + 256 * p;
            *reinterpret_cast<uint4*>(xs + u / XW * XROW + u % XW * 8) = WEIGHTS ? weight8(xreg[p]) : xreg[p];
        }
#pragma unroll
        for (int j = 0; j < YLOADS; j++) {
            const int u = tid + 256 * j;
            *reinterpret_cast<uint4*>(ys + u / UNITS * YROW + u % UNITS * 8) = WEIGHTS ? yreg[j] : sign8(yreg[j]);
        }
        __syncthreads();
        if (r0 + AG_STEP < len) load(r0 + AG_STEP);
        const _Float16* const xf = reinterpret_cast<const _Float16*>(xs);
        const _Float16* const yf = reinterpret_cast<const _Float16*>(ys);
#pragma unroll
        for (int s = 0; s < AG_STEP / 32; s++) {
            const int r = 64 * (s >> 1) + part * 32 + (s & 1) * 16;
            const half8 xv = TRANS ? column8(xf, XROW, r, it * 32, lane) : *reinterpret_cast<const half8*>(xf + (it * 32 + c) * XROW + r + 8 * h);
#pragma unroll
            for (int t = 0; t < DT; t++) acc[t] = mma(column8(yf, YROW, r, t * 32, lane), xv, acc[t]);
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

// grad_P of 128 rows, a wave 32 of them, and `a.chunks` times 64 columns: the signs of V go through LDS, G's rows are operands as they lie.  The
// columns are dealt to two operands as even and odd ones, so that a lane has pairs of neighbours: a half-wave stores a line.
template <int DT>
__device__ __forceinline__ void probs_strip(const AttnGradArgs& a, const int z, const int n0, const int m0, unsigned char* smem)
{
    constexpr int D = DT * 32, VROW = D + 8, UNITS = D / 8, LOADS = 64 * UNITS / 256;
    typedef _Float16 half2v __attribute__((ext_vector_type(2)));
    typedef float float2v __attribute__((ext_vector_type(2)));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5, c = lane & 31, nw = n0 + wave * 32;
    const __half* const g = head_at(a.a, z, a.inner) + min(nw + c, a.N - 1) * a.a.row + 8 * h;
    const __half* const v = head_at(a.b, z, a.inner);
    __half* const vs = reinterpret_cast<__half*>(smem);
    uint4 vreg[LOADS];
    auto load = [&](const int m) {
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const int u = tid + 256 * j;
            vreg[j] = *reinterpret_cast<const uint4*>(v + min(m + u / UNITS, a.M - 1) * a.b.row + u % UNITS * 8);
        }
    };
    load(m0);
    half8 gf[2 * DT];
#pragma unroll
    for (int s = 0; s < 2 * DT; s++) gf[s] = *reinterpret_cast<const half8*>(g + 16 * s);
    __half* const out = a.gp + ((int64_t)z * a.N + nw + 4 * h) * a.M;
#pragma unroll 1
    for (int k = 0; k < a.chunks; k++) {
        const int m1 = m0 + 64 * k;
        if (m1 >= a.M) break;
        if (k) __syncthreads();
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const int u = tid + 256 * j;
            *reinterpret_cast<uint4*>(vs + u / UNITS * VROW + u % UNITS * 8) = sign8(vreg[j]);
        }
        __syncthreads();
        if (k + 1 < a.chunks) load(m1 + 64);
        float16v acc[2];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[j][i] = 0.f;
#pragma unroll
        for (int s = 0; s < 2 * DT; s++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                acc[j] = mma(gf[s], *reinterpret_cast<const half8*>(reinterpret_cast<const _Float16*>(vs) + (2 * c + j) * VROW + 16 * s + 8 * h), acc[j]);
        const int m = m1 + 2 * c;
        auto rows_out = [&](auto whole_c) {
            constexpr bool WHOLE = decltype(whole_c)::value;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int r = 8 * (i >> 2) + (i & 3);
                const half2v half = {(_Float16)0.5f, (_Float16)0.5f};
                const float2v two = {acc[0][i], acc[1][i]};
                const half2v p = __builtin_convertvector(two, half2v) * half;
                __half* const to = out + (int64_t)r * a.M + m;
                if (WHOLE) __builtin_memcpy(to, &p, 4);
                else if (nw + 4 * h + r < a.N) {
                    if (m < a.M) reinterpret_cast<_Float16*>(to)[0] = p[0];
                    if (m + 1 < a.M) reinterpret_cast<_Float16*>(to)[1] = p[1];
                }
            }
        };
        if (nw + 32 <= a.N && m1 + 64 <= a.M) rows_out(std::true_type{});
        else rows_out(std::false_type{});
    }
}

// (TRANS, or 64 rows of AG_STEP: about the same)
template <int DT> constexpr int ag_lds()
{
    constexpr int x = (AG_STEP * 72 > 64 * (AG_STEP + 8) ? AG_STEP * 72 : 64 * (AG_STEP + 8)) * 2, y = AG_STEP * (DT * 32 + 8) * 2;
    return x + y > DT * 8192 ? x + y : DT * 8192;
}

// A matrix's blocks are neighbours: its second reading finds it in the caches.
template <int DT>
__global__ __launch_bounds__(256) void scores_grad_kernel(const AttnGradArgs a)
{
    __shared__ __align__(16) unsigned char smem[ag_lds<DT>()];
    const unsigned id = xcd_contiguous_id(blockIdx.x, gridDim.x);
    const int z = id / a.per_batch, t = id % a.per_batch;
    if (t < a.first) tall_product<DT, false, false>(a, a.b, a.ga, z, t * 64, smem);
    else tall_product<DT, true, false>(a, a.a, a.gb, z, (t - a.first) * 64, smem);
}

// Both halves share the registers of the larger, the strips: 4, 3, 3 and 2 waves a SIMD at D = 32 .. 128, where P's half by itself has one or two more.
// Both gradients take the same time either way; V's alone would gain where the chip is full (64 x 1024^2 D = 64 31.6 -> 26.4 us, 768 x 512^2 D = 128
// 173 -> 155) and nothing where it is not (48 x 512^2 8.8 -> 8.5).
template <int DT>
__global__ __launch_bounds__(256) void context_grad_kernel(const AttnGradArgs a)
{
    __shared__ __align__(16) unsigned char smem[ag_lds<DT>()];
    // (the longer blocks first)
    const int tall = a.batch * a.first;
    if ((int)blockIdx.x < tall) {
        const unsigned id = xcd_contiguous_id(blockIdx.x, tall);
        return tall_product<DT, true, true>(a, a.a, a.gb, id / a.first, id % a.first * 64, smem);
    }
    const unsigned id = xcd_contiguous_id(blockIdx.x - tall, gridDim.x - tall), strips = a.per_batch - a.first;
    const int u = id % strips;
    const int mb = (a.M + 64 * a.chunks - 1) / (64 * a.chunks);
    probs_strip<DT>(a, id / strips, u / mb * 128, u % mb * 64 * a.chunks, smem);
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
    // A strip's columns: more of them read G's rows once, while there are eight blocks a compute unit.  grad_P alone, us with 64 columns, up to 128,
    // 256 and 512: 192 x 512^2 D = 64 25.5, 22.3, D = 128 48.6, 35.8; 64 x 1024^2 D = 64 33.8, 28.0, 25.0, D = 128 62.7, 45.7, 37.2; 768 x 512^2 D = 64 147,
    // 132, 112, 107, D = 128 262, 190, 154, 144.  D = 32 hardly cares (64 x 1024^2 22.5, 22.8, 22.9).  From half as many blocks on: D = 128 faster,
    // 35.5 -> 29.5, but 64 x 1024^2 D = 64 25.8 -> 27.3.
    int64_t chunks = 1;
    while (chunks < 8 && batch * cdiv(N, 128) * cdiv(M, 128 * chunks) >= 2048) chunks *= 2;
    const int64_t strips = cdiv(N, 128) * cdiv(M, 64 * chunks);
    AttnGradArgs g = {};
    auto view = [&](const void* p, const int i) { return HeadView{(const __half*)p, strides[3 * i], strides[3 * i + 1], strides[3 * i + 2]}; };
    g.m = (const __half*)m; g.a = view(a, 0); g.b = view(b, 1); g.ga = view(grad_a, 2); g.gb = view(grad_b, 3); g.gp = (__half*)grad_p;
    g.N = (int)N; g.M = (int)M; g.inner = (int)inner;
    const int64_t first = context ? (grad_b ? mb : 0) : (grad_a ? nb : 0), second = context ? (grad_p ? strips : 0) : (grad_b ? mb : 0);
    if (first + second == 0) return BGEMM_OK;
    if (batch > 0x7fffffffLL / (first + second)) return fail(BGEMM_EINVAL, "%s: too many blocks", who);
    g.first = (int)first; g.per_batch = (int)(first + second); g.batch = (int)batch; g.chunks = (int)chunks;
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
