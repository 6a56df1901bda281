// Both products of binary attention on fp16 operands where they lie, one launch each (tests/python/bert/bert.py:245-259 on sign bits,
// tests/python/bgemm_linear.py:9-61), for the passes whose scores and probabilities torch works on in between:
//
//   scores[n,m]  = sum_c sign(A)[n,c] sign(B)[m,c]     or the number of columns where both are negative
//   context[n,:] = sum over the m with P[n,m] >= 0 (sign bit clear) of sign(V)[m,:]
//
// on a batch of matrices, A, B and V of D = 32 .. 128 columns.  As two packs and a GEMM each a product was three launches, half of whose
// time went by between them, and P's bits and the transposed ones of V crossed memory on the way: 48 matrices of 512 x 512, D = 64,
// 14.5 and 20.5 us.  Here a block makes the bits it needs in LDS, those of its keys or values again for every 128 or 256 rows: 7.0 us
// (25 MB written, 4.9 us of a large copy's rate and the launch) and 10.8 (25 MB read; the time to V's bits, during which P's first groups
// are on their way, is what is left).
#include "common.h"
#include "attention_bits.h"

namespace bgemm {

struct AttnView { const __half* p; int64_t so, si, row; };      // [outer][inner][rows][..], the last dimension dense

struct AttnProductArgs {
    AttnView a, b;                    // scores: A, B.  context: P, V
    __half* out;                      // [batch][N][M] or [batch][N][D], dense
    int N, M, inner, nblocks, mblocks, both_negative, past;
    int one_xcd;                      // scores: a matrix's blocks on one XCD
};

constexpr int AP_COLS = 256;      // of a block of the scores

__device__ __forceinline__ const __half* view_at(const AttnView& v, const int z, const int inner) { return v.p + (z / inner) * v.so + (z % inner) * v.si; }

// Sign bits of `rows` rows of D halves from row r0 on (rows past `end` as its last) into words [W][rows] of LDS, eight elements a lane and step.
template <int W, int ROWS, int THREADS>
struct RowBits {
    static constexpr int PER_ROW = W * 4, STEPS = ROWS * PER_ROW / THREADS;
    uint4 raw[STEPS];
    __device__ __forceinline__ void load(const __half* base, const int64_t stride, const int r0, const int end)
    {
#pragma unroll
        for (int i = 0; i < STEPS; i++) {
            const int u = threadIdx.x + i * THREADS, r = min(r0 + u / PER_ROW, end - 1);
            __builtin_memcpy(&raw[i], base + r * stride + u % PER_ROW * 8, 16);
        }
    }
    __device__ __forceinline__ void store(uint32_t* words) const
    {
#pragma unroll
        for (int i = 0; i < STEPS; i++) {
            const int u = threadIdx.x + i * THREADS, r = u / PER_ROW, ch = u % PER_ROW;
            uint32_t sg, nz;
            bits8(raw[i], sg, nz);
            reinterpret_cast<unsigned char*>(words)[((ch >> 2) * ROWS + r) * 4 + 3 - (ch & 3)] = (unsigned char)sg;
        }
    }
};

// Queries are columns of the MFMA and keys its rows, in an order that gives a lane 32 consecutive keys of its query (see attention.hip).
template <int W, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void scores_kernel(const AttnProductArgs a)
{
    constexpr int D = W * 32, CH = (W + 1) / 2, THREADS = WAVES * 64, AP_ROWS = WAVES * 32;
    __shared__ uint32_t qb[W * AP_ROWS], kb[W * AP_COLS];
    __shared__ __align__(16) unsigned char stages[WAVES][32 * ATTN_STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, c = lane & 31;
    const unsigned id = a.one_xcd ? xcd_contiguous_id(blockIdx.x, gridDim.x) : blockIdx.x, per = a.nblocks * a.mblocks;
    const int z = id / per, t = id % per;
    const int n0 = t / a.mblocks * AP_ROWS, m0 = t % a.mblocks * AP_COLS;
    {
        RowBits<W, AP_COLS, THREADS> kr;
        RowBits<W, AP_ROWS, THREADS> qr;
        kr.load(view_at(a.b, z, a.inner), a.b.row, m0, a.M);
        qr.load(view_at(a.a, z, a.inner), a.a.row, n0, a.N);
        kr.store(kb);
        qr.store(qb);
    }
    __syncthreads();
    const int q0 = n0 + wave * 32;
    if (q0 >= a.N) return;
    unsigned qf[CH][4];
    int ones = 0;
#pragma unroll
    for (int ch = 0; ch < CH; ch++) {
        const int w = 2 * ch + h;
        const unsigned x = w < W ? qb[w * AP_ROWS + wave * 32 + c] : 0u;
        ones += __popc(x);
#pragma unroll
        for (int s = 0; s < 4; s++) qf[ch][s] = a.both_negative ? attn_one(x, s) : attn_sign(~x, s);
    }
    ones += __shfl_xor(ones, 32);
    EngF4::Acc start;
#pragma unroll
    for (int v = 0; v < 16; v++) start[v] = a.both_negative ? 0.f : (float)(D - 2 * ones);
    const int row_key = 32 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
    auto tile = [&](const int grp, const int j) {
        EngF4::Acc acc;
#pragma unroll
        for (int ch = 0; ch < CH; ch++) {
            const int w = 2 * ch + h;
            unsigned x = kb[(w < W ? w : 0) * AP_COLS + grp * 64 + 16 * j + row_key];
            if (W % 2 && ch == CH - 1 && h) x = 0;
            unsigned kf[4];
#pragma unroll
            for (int s = 0; s < 4; s++) kf[s] = attn_bit(x, s);
            acc = EngF4::mma(EngF4::make(kf), EngF4::make(qf[ch]), ch == 0 ? start : acc);
        }
        return acc;
    };
    unsigned char* const stage = stages[wave];
    const int r8 = lane >> 3, c8 = lane & 7;
    __half* const matrix = a.out + (int64_t)z * a.N * a.M;
    // (whole groups leave through a buffer that ends with the matrix: rows past the last one are dropped)
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(matrix, 0, (int)(a.N * a.M * 2), 0x00020000);
    int voff[4];
#pragma unroll
    for (int i = 0; i < 4; i++) voff[i] = ((q0 + r8 + 8 * i) * a.M + m0 + c8 * 8) * 2;
    const int groups = min(AP_COLS / 64, (a.M - m0 + 63) / 64);
    EngF4::Acc even = tile(0, 0), odd;
#pragma unroll 1
    for (int grp = 0; grp < groups; grp++) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (j == 0) odd = tile(grp, 1);
            else even = tile(min(grp + 1, groups - 1), 0);
            const EngF4::Acc& acc = j == 0 ? even : odd;
            unsigned hs[8];
#pragma unroll
            for (int p = 0; p < 8; p++) hs[p] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(acc[2 * p], acc[2 * p + 1]));      // (small integers: exact)
            uint4* const to = reinterpret_cast<uint4*>(stage + c * ATTN_STAGE + 64 * h + 32 * j);
            to[0] = make_uint4(hs[0], hs[1], hs[2], hs[3]);
            to[1] = make_uint4(hs[4], hs[5], hs[6], hs[7]);
        }
        attn_wave_sync();
        const bool whole = m0 + grp * 64 + 64 <= a.M;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint4 x = *reinterpret_cast<const uint4*>(stage + (r8 + 8 * i) * ATTN_STAGE + c8 * 16);
            if (whole) {
                const v4i v = {(int)x.x, (int)x.y, (int)x.z, (int)x.w};
                if (a.past) __builtin_amdgcn_raw_buffer_store_b128(v, rs, voff[i], grp * 128, 2);
                else __builtin_amdgcn_raw_buffer_store_b128(v, rs, voff[i], grp * 128, 0);
            } else if (q0 + r8 + 8 * i < a.N) {
                const unsigned d[4] = {x.x, x.y, x.z, x.w};
                __half* const to = matrix + (int64_t)(q0 + r8 + 8 * i) * a.M + m0 + grp * 64 + c8 * 8;
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (m0 + grp * 64 + c8 * 8 + e < a.M) to[e] = __ushort_as_half((uint16_t)(d[e >> 1] >> (16 * (e & 1))));
            }
        }
        attn_wave_sync();
    }
}

// A wave takes 32 rows of P and all of its columns or one half of them, 64 at a time and two groups requested ahead; a lane's eight
// elements become a byte, and the bytes of a row, through LDS, the word that is the product's operand.  A block's rows are CTX_ROWS.
constexpr int CTX_ROWS = 128;

// (blocks of at most 512 threads; the registers of four waves a SIMD are enough up to D = 96, which takes 124)
template <int W>
__global__ __launch_bounds__(512, W == 4 ? 2 : 4) void context_kernel(const AttnProductArgs a)
{
    constexpr int D = W * 32;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5, c = lane & 31;
    const int groups = (a.M + 63) / 64, S64 = groups * 64, waves = blockDim.x >> 6, part = wave >> 2, parts = waves >> 2;
    uint32_t* const vb = reinterpret_cast<uint32_t*>(smem);      // [W][S64]: words of a row of V
    uint32_t* const vt = vb + W * S64;                           // [2 groups][D]: words of 32 rows
    unsigned char* const stage = reinterpret_cast<unsigned char*>(vt + W * S64) + wave * 256;
    // (a matrix's blocks on one XCD: 48 x 512^2, D = 64, 10.7 -> 9.8 us from a graph, 192 x 512^2 28.5 -> 24.9, few matrices level)
    const int id = (int)xcd_contiguous_id(blockIdx.x, gridDim.x), z = id / a.nblocks, q0 = id % a.nblocks * CTX_ROWS + (wave & 3) * 32;
    const int first = groups * part / parts, end = q0 < a.N ? groups * (part + 1) / parts : first;
    const __half* v = view_at(a.b, z, a.inner);
    const __half* p = view_at(a.a, z, a.inner);
    // P's first groups are on their way while V is packed
    const int r8 = lane >> 3, c8 = lane & 7;
    const __half* row[4];
#pragma unroll
    for (int i = 0; i < 4; i++) row[i] = p + (int64_t)min(q0 + r8 + 8 * i, a.N - 1) * a.a.row;
    const int last8 = a.M - 8;                                   // (a row's last chunk is read as its last eight elements, the bits shifted into place)
    auto request = [&](uint4 (&raw)[4], const int grp) {
        const int at = min(min(grp, groups - 1) * 64 + c8 * 8, last8);
#pragma unroll
        for (int i = 0; i < 4; i++) __builtin_memcpy(&raw[i], row[i] + at, 16);
    };
    uint4 ra[4], rb[4], rc[4];
    request(ra, first);
    request(rb, first + 1);
    {
        constexpr int PER_ROW = W * 4, AHEAD = 4;
        const int step = blockDim.x;
        for (int u0 = threadIdx.x; u0 < S64 * PER_ROW; u0 += step * AHEAD) {
            uint4 raw[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                const int u = u0 + i * step;
                __builtin_memcpy(&raw[i], v + (int64_t)min(u / PER_ROW, a.M - 1) * a.b.row + u % PER_ROW * 8, 16);
            }
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                const int u = u0 + i * step, r = u / PER_ROW, ch = u % PER_ROW;
                uint32_t sg, nz;
                bits8(raw[i], sg, nz);
                if (r < S64) reinterpret_cast<unsigned char*>(vb)[((ch >> 2) * S64 + r) * 4 + 3 - (ch & 3)] = (unsigned char)sg;
            }
        }
    }
    __syncthreads();
    for (int u0 = wave * 2; u0 < groups * 2 * W; u0 += 2 * waves) {
        const int u = u0 + h, kw = u / W, w = u % W;             // (an even number of units)
        const unsigned t = transpose32(__brev(vb[w * S64 + kw * 32 + c]), lane);
        vt[kw * D + w * 32 + c] = __brev(t);
    }
    __syncthreads();
    const int row_col = 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
    EngF4::Acc ctx[W];
#pragma unroll
    for (int t = 0; t < W; t++)
#pragma unroll
        for (int i = 0; i < 16; i++) ctx[t][i] = 0.f;
    int counted = 0;
    auto step = [&](const uint4 (&raw)[4], const int grp) {
        const int shift = min(max(grp * 64 + c8 * 8 - last8, 0), 8);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t sg, nz;
            bits8(raw[i], sg, nz);
            // (elements past the row's end count as negative ones, which add nothing)
            stage[(r8 + 8 * i) * 8 + (c8 & 4) + 3 - (c8 & 3)] = (unsigned char)(sg << shift | (0xffu >> (8 - shift)));
        }
        attn_wave_sync();
        const unsigned counts = ~reinterpret_cast<const uint32_t*>(stage)[c * 2 + h];
        attn_wave_sync();
        counted += __popc(counts);
        unsigned pf[4];
#pragma unroll
        for (int s = 0; s < 4; s++) pf[s] = attn_one(counts, s);
#pragma unroll
        for (int t = 0; t < W; t++) {
            const unsigned x = vt[(2 * grp + h) * D + t * 32 + row_col];
            unsigned vf[4];
#pragma unroll
            for (int s = 0; s < 4; s++) vf[s] = attn_bit(x, s);
            ctx[t] = EngF4::mma(EngF4::make(vf), EngF4::make(pf), ctx[t]);
        }
    };
#pragma unroll 1
    for (int grp = first; grp < end;) {
        request(rc, grp + 2);
        step(ra, grp);
        if (++grp >= end) break;
        request(ra, grp + 2);
        step(rb, grp);
        if (++grp >= end) break;
        request(rb, grp + 2);
        step(rc, grp);
        ++grp;
    }
    counted += __shfl_xor(counted, 32);
    // The halves' sums, whole numbers of at most M <= 4096, meet in 16 bits where V's words were.
    if (parts == 2) {
        uint32_t* const to = reinterpret_cast<uint32_t*>(smem) + (wave & 3) * (W * 8 + 1) * 64 + lane;
        __syncthreads();
        if (part) {
#pragma unroll
            for (int t = 0; t < W; t++)
#pragma unroll
                for (int i = 0; i < 8; i++) to[(t * 8 + i) * 64] = (uint32_t)ctx[t][2 * i] | (uint32_t)ctx[t][2 * i + 1] << 16;
            to[W * 8 * 64] = (uint32_t)counted;
        }
        __syncthreads();
        if (!part) {
#pragma unroll
            for (int t = 0; t < W; t++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint32_t x = to[(t * 8 + i) * 64];
                    ctx[t][2 * i] += (float)(x & 0xffffu);
                    ctx[t][2 * i + 1] += (float)(x >> 16);
                }
            counted += (int)to[W * 8 * 64];
        }
    }
    if (part || q0 + c >= a.N) return;
    __half* const out = a.out + ((int64_t)z * a.N + q0 + c) * D + 16 * h;
#pragma unroll
    for (int t = 0; t < W; t++) {
        union { __half x[16]; uint4 u[2]; } pk;
#pragma unroll
        for (int i = 0; i < 16; i++) pk.x[i] = __float2half_rn(fmaf(-2.f, ctx[t][i], (float)counted));
        uint4* const to = reinterpret_cast<uint4*>(out + t * 32);
        to[0] = pk.u[0]; to[1] = pk.u[1];
    }
}

}  // namespace bgemm

using namespace bgemm;

static bool product_fits(int64_t batch, int64_t inner, int64_t N, int64_t M, int64_t D)
{
    return batch >= 1 && inner >= 1 && batch % inner == 0 && N >= 1 && M >= 1 && N <= (1 << 20) && M <= (1 << 20) && (D == 32 || D == 64 || D == 96 || D == 128);
}

// strides: outer, inner and row stride, in elements, of the two operands.
static void product_args(AttnProductArgs& g, const void* a, const void* b, const int64_t* strides, int64_t inner, int64_t N, int64_t M, void* out)
{
    g.a = {(const __half*)a, strides[0], strides[1], strides[2]};
    g.b = {(const __half*)b, strides[3], strides[4], strides[5]};
    g.out = (__half*)out;
    g.N = (int)N; g.M = (int)M; g.inner = (int)inner;
}

extern "C" int bgemm_scores_forward(int mode, const void* a, const void* b, const int64_t* strides, int64_t batch, int64_t inner, int64_t N, int64_t M, int64_t D,
                                    void* out, void* stream)
{
    const char* who = "bgemm_scores_forward";
    if ((mode != BGEMM_MODE_XOR && mode != BGEMM_MODE_AND) || !product_fits(batch, inner, N, M, D) || N * M * 2 > 0x7fffffffLL)
        return fail(BGEMM_EINVAL, "%s: mode %d, %lld (%lld) matrices of %lld x %lld, %lld columns", who, mode, (long long)batch, (long long)inner, (long long)N, (long long)M,
                    (long long)D);
    if (!a || !b || !strides || !out) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (((uintptr_t)a | (uintptr_t)b | (uintptr_t)out) & 1) return fail(BGEMM_EALIGN, "%s: an operand is not aligned", who);
    AttnProductArgs g = {};
    product_args(g, a, b, strides, inner, N, M, out);
    // 256 rows a block read the keys half as often (192 x 512^2: D = 128 38.7 -> 30.5 us, D = 64 27.2 -> 23.4), where no more of them is
    // past the end than with 128 (48 x 300^2: 7.6 -> 8.2), the chip stays filled (2 x 512^2: 4.8 -> 5.1) and keys are long enough
    // (16 x 2048^2, D = 32: 25.8 -> 27.3).
    const int waves = D >= 64 && cdiv(N, 256) * 2 == cdiv(N, 128) && batch * cdiv(N, 256) * cdiv(M, AP_COLS) >= 192 ? 8 : 4;
    g.nblocks = (int)cdiv(N, waves * 32); g.mblocks = (int)cdiv(M, AP_COLS);
    g.both_negative = mode == BGEMM_MODE_AND;
    g.past = M % 32 == 0 && ((uintptr_t)out & 63) == 0;
    // Blocks of a matrix go to one XCD, which reads its operands once, where an L2 does not hold the operands of all matrices anyway, and where
    // lines that two blocks share would be written by two XCDs.  From a graph, us, round robin / one XCD: 192 x 512^2 D = 64 23.4 / 20.1, 64 x 1024^2
    // 30.7 / 25.9, 128 x 512^2 D = 128 20.6 / 16.8, 96 x 512^2 D = 32 (6 MB of operands) 11.4 / 10.6, 16 x 1000^2 13.3 / 11.9; but 32 x 1024^2 D = 32 (4 MB)
    // 13.8 / 15.0, 16 x 1024^2 7.9 / 8.5, and 64 x 1024^2 26.8 / 27.6.  Short rows: 192 x 256^2 D = 32 6.9 / 7.7, 400 x 256^2 D = 128 15.5 / 17.3, 48 x 384 x 400 D = 64 8.1 / 8.4.
    g.one_xcd = M >= 500 && (M % 64 != 0 || (batch * (N + M) * D * 2 >= 6 << 20 && (D > 32 || M <= 512)));
    const int64_t blocks = batch * g.nblocks * g.mblocks;
    if (blocks > 0x7fffffffLL) return fail(BGEMM_EINVAL, "%s: too many blocks", who);
    const dim3 grid((unsigned)blocks), block(waves * 64);
    const hipStream_t st = (hipStream_t)stream;
#define SCORES(W) (waves == 4 ? scores_kernel<W, 4> : scores_kernel<W, 8>)
    switch (D / 32) {
    case 1: hipLaunchKernelGGL(SCORES(1), grid, block, 0, st, g); break;
    case 2: hipLaunchKernelGGL(SCORES(2), grid, block, 0, st, g); break;
    case 3: hipLaunchKernelGGL(SCORES(3), grid, block, 0, st, g); break;
    default: hipLaunchKernelGGL(SCORES(4), grid, block, 0, st, g); break;
    }
#undef SCORES
    return check_launch(who);
}

extern "C" int bgemm_context_forward(const void* probs, const void* value, const int64_t* strides, int64_t batch, int64_t inner, int64_t N, int64_t M, int64_t D, void* out,
                                     void* stream)
{
    const char* who = "bgemm_context_forward";
    if (!product_fits(batch, inner, N, M, D) || M < 8 || M * D > (1 << 17))
        return fail(BGEMM_EINVAL, "%s: %lld (%lld) matrices of %lld x %lld, %lld columns", who, (long long)batch, (long long)inner, (long long)N, (long long)M, (long long)D);
    if (!probs || !value || !strides || !out) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (((uintptr_t)probs | (uintptr_t)value) & 1 || (uintptr_t)out & 15) return fail(BGEMM_EALIGN, "%s: an operand is not aligned", who);
    AttnProductArgs g = {};
    product_args(g, probs, value, strides, inner, N, M, out);
    g.nblocks = (int)cdiv(N, CTX_ROWS);
    const int64_t blocks = batch * g.nblocks;
    if (blocks > 0x7fffffffLL) return fail(BGEMM_EINVAL, "%s: too many blocks", who);
    // Two waves to a row fill the chip (48 x 512^2, D = 64: 13.5 -> 10.8 us; 2 x 512^2: 11.9 -> 9.1) unless the blocks already do
    // (192 x 512^2: 28.6 -> 31.6) or a row is short (16 x 128^2: 5.4 -> 5.9).  Four were never ahead of two by more than 2 us.
    const int parts = M < 256 || blocks > 512 ? 1 : 2;
    const size_t words = (size_t)2 * (D / 32) * cdiv(M, 64) * 64 * 4 + (size_t)parts * 4 * 256, sums = (size_t)(parts - 1) * 4 * (D / 32 * 8 + 1) * 256;
    const size_t lds = words > sums ? words : sums;
    const dim3 grid((unsigned)blocks), block(parts * 256);
    const hipStream_t st = (hipStream_t)stream;
    switch (D / 32) {
    case 1: hipLaunchKernelGGL(context_kernel<1>, grid, block, lds, st, g); break;
    case 2: hipLaunchKernelGGL(context_kernel<2>, grid, block, lds, st, g); break;
    case 3: hipLaunchKernelGGL(context_kernel<3>, grid, block, lds, st, g); break;
    default: hipLaunchKernelGGL(context_kernel<4>, grid, block, lds, st, g); break;
    }
    return check_launch(who);
}
