// Binary self-attention without a gradient, one launch: what tests/python/bert/bert.py:245-259 does with dense matrices, on sign bits.
//
//   scores[q,k] = half(half(sum_c sign(Q)[q,c] sign(K)[k,c]) / sqrt(D))              stored: the block returns them
//   p[q,k]      = half(softmax_k(scores[q,:]))                                       never stored
//   context[q,c] = half(sum over the k with p[q,k] >= 1/S of sign(V)[k,c])           stored in the layer's own order, heads merged
//
// As separate kernels (a GEMM, the division, the softmax, the shift by 1/S, a pack, the second GEMM, and packs and copies of
// head-split views around them) the probabilities cross memory seven times: 12 heads of 64, 16 x 512 tokens 225 us, of which the one
// pass over the scores that is needed takes 20.  A score is one of D + 1 numbers (matching bits, 0 .. D), so everything the softmax
// needs of it comes from a table of D + 1 entries in LDS (exponential and rounded score), shifted by the largest score there can
// be instead of the row's: no pass for the maximum, and the table is the same for every row.  The probabilities rise with the
// score, so the bits of a row are a comparison with one number, found by bisection with the very division and rounding.
//
// A wave owns 32 queries.  Keys are the rows of the MFMA and queries its columns: a lane then holds one query's scores, row sums
// stay in the lane, and the order of the keys in a fragment is chosen such that a lane holds 32 consecutive ones: its bits are a
// word, and that word, four ways shifted, is the second product's operand as it stands.  The scores are multiplied twice, once for
// the sums and once for the bits: one MFMA per 32 x 32 tile and 64 of D, cheaper than keeping S of them a lane.
// 16 x 512 tokens, 12 heads of 64: 100 MB of scores written in 30.7 us (3.3 TB/s; three waves a SIMD, vector units half busy, the rest of a
// wave's time its chain of MFMA, table, LDS and store).  37 us with the table's index in two instructions, sums that were set to their
// start tile by tile, operands of +-1 on both sides (11 vector instructions a word of keys instead of 5), and every wave waiting for
// each word that a block prepares; the last also where there are few waves: 4 x 512 tokens 36 -> 16.4, 8 x 256 20 -> 10.2.  With a whole
// group's sums on their way (210 registers, two waves a SIMD) 36.9.  A head's blocks are on one XCD: 30.9 -> 30.1, and what the launch behind it
// takes 13.6 -> 12.3 (bits of neighbouring heads written into one cache): the whole block 58.6 -> 57.0 from a graph, also where the kernel alone is
// not ahead (4 x 512 tokens 18.2 -> 18.6, the block 33.6 -> 33.1; 8 x 256 12.5 and 12.5, 27.7 -> 26.8; 1 x 1024, 16 heads, 29.2 -> 29.6, 45.9 -> 45.6).
#include "common.h"
#include "attention_bits.h"
#include <math.h>
#include <type_traits>

namespace bgemm {

struct AttnArgs {
    const uint32_t* q; const uint32_t* k; const uint32_t* v;      // sign bits [batch * S][heads * D], tiled
    __half* scores; void* context;    // context: numbers, or the tiled operand of their signs after *zp is subtracted
    const void* zp;
    int64_t KT;                       // of the operands
    int S, heads, groups, qblocks, f32, past;      // past: scores are stored past the caches
    float scale, level;               // 1 / sqrt(D), 1 / S
};

// W: words a head (D = 32 W).  BITS: the context leaves as the next binary layer's operand.
template <int W, bool BITS>
__global__ __launch_bounds__(512) void attention_kernel(const AttnArgs a)
{
    constexpr int D = W * 32, CH = (W + 1) / 2;       // chunks of 64 bits, the last half a one if W is odd
    // a sum comes out as 2^23 + 2 * (matching bits): its bit pattern is an index
    constexpr unsigned BASE = 0x4b000000u;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int h = lane >> 5, c = lane & 31;
    const int S = a.S, S64 = a.groups * 64;
    unsigned char* const stage = smem + wave * (32 * ATTN_STAGE);
    uint2* const tbl = reinterpret_cast<uint2*>(smem + waves * (32 * ATTN_STAGE));           // [D + 2]
    uint32_t* const kb = reinterpret_cast<uint32_t*>(tbl + D + 2);                           // [W][S64]
    uint32_t* const vt = kb + W * S64;                                                       // [2 groups][D]: words of 32 keys

    const unsigned id = xcd_contiguous_id(blockIdx.x, gridDim.x);
    const int bh = id / a.qblocks, qb = id % a.qblocks, b = bh / a.heads, head = bh % a.heads;
    const int64_t row0 = (int64_t)b * S;
    auto word = [&](const uint32_t* p, const int row, const int w) { return p[tiled_word_offset(row0 + row, head * W + w, a.KT)]; };

    // ---- the block's shared operands: table, key bits, value bits transposed -----------------------------------------------------
    auto score16 = [&](const int idx) { return __float2half_rn((float)(2 * idx - D) * a.scale); };
    for (int i = threadIdx.x; i <= D; i += blockDim.x) {
        const __half s = score16(i);
        tbl[i] = make_uint2(__float_as_uint(expf(__half2float(s) - __half2float(score16(D)))), __half_as_ushort(s));
    }
    // (a stretch of loads before its first use: one trip to the caches for several words, where each of a few waves would wait for its own)
    constexpr int AHEAD = 4;
    for (int key0 = threadIdx.x; key0 < S64; key0 += AHEAD * blockDim.x) {
        uint32_t x[AHEAD][W];
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
#pragma unroll
            for (int w = 0; w < W; w++) x[i][w] = word(a.k, min(key0 + i * (int)blockDim.x, S - 1), w);
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int key = key0 + i * blockDim.x;
            if (key < S64)
#pragma unroll
                for (int w = 0; w < W; w++) kb[w * S64 + key] = key < S ? x[i][w] : 0u;
        }
    }
    for (int u0 = wave * 2; u0 < a.groups * 2 * W; u0 += waves * 2 * AHEAD) {
        uint32_t x[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int u = min(u0 + i * waves * 2 + h, a.groups * 2 * W - 1), kw = u / W, key = kw * 32 + c;
            x[i] = word(a.v, min(key, S - 1), u % W);
        }
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int u = u0 + i * waves * 2 + h, kw = u / W, w = u % W;
            if (u0 + i * waves * 2 >= a.groups * 2 * W) break;
            const unsigned t = transpose32(__brev(kw * 32 + c < S ? x[i] : 0u), lane);       // bit r: key r of the lane's column
            if (u < a.groups * 2 * W) vt[kw * D + w * 32 + c] = __brev(t);
        }
    }
    const int q0 = (qb * waves + wave) * 32;
    unsigned qw[CH];
#pragma unroll
    for (int ch = 0; ch < CH; ch++) {
        const int w = 2 * ch + h;
        qw[ch] = word(a.q, min(q0 + c, S - 1), w < W ? w : 0);
    }
    __syncthreads();
    if (q0 >= S) return;
    unsigned qf[CH][4];
    int ones = 0;
#pragma unroll
    for (int ch = 0; ch < CH; ch++) {
        if (2 * ch + h < W) ones += __popc(qw[ch]);
#pragma unroll
        for (int s = 0; s < 4; s++) qf[ch][s] = attn_sign(~qw[ch], s);
    }
    ones += __shfl_xor(ones, 32);
    // 2 * (matching bits) = D + (sum over the query's x of x (1 - 2 b)): what the sums start from
    const float both = (float)(2 * D - 2 * ones);
    EngF4::Acc start;
#pragma unroll
    for (int v = 0; v < 16; v++) start[v] = 8388608.f + both;
    // MFMA row r = 8 g + 4 half + i of tile j is key 32 half + 16 j + 4 g + i of the group's 64: register v of a lane is then key
    // 32 h + 16 j + v.  (The second product's rows, columns of V, likewise: register v is column 16 h + v.)
    const int row_key = 32 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3), row_col = 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
    auto tile = [&](const int grp, const int j) {
        EngF4::Acc acc;
#pragma unroll
        for (int ch = 0; ch < CH; ch++) {
            const int w = 2 * ch + h;
            unsigned x = kb[(w < W ? w : 0) * S64 + grp * 64 + 16 * j + row_key];
            if (W % 2 && ch == CH - 1 && h) x = 0;
            unsigned kf[4];
#pragma unroll
            for (int s = 0; s < 4; s++) kf[s] = attn_bit(x, s);
            acc = EngF4::mma(EngF4::make(kf), EngF4::make(qf[ch]), ch == 0 ? start : acc);
        }
        return acc;
    };
    // ---- scores out, sums of the exponentials --------------------------------------------------------------------------------------
    float s0 = 0.f, s1 = 0.f;
    const int r8 = lane >> 3, c8 = lane & 7;
    __half* const matrix = a.scores + (int64_t)bh * S * S;
    __half* const srow = matrix + (int64_t)(q0 + r8) * S + c8 * 8;
    // (whole groups leave through a buffer that ends with the matrix: rows past the last one are dropped)
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(matrix, 0, S * S * 2, 0x00020000);
    int voff[4];
#pragma unroll
    for (int i = 0; i < 4; i++) voff[i] = ((q0 + r8 + 8 * i) * S + c8 * 8) * 2;
    // (an entry's address in LDS straight from the sum's bits: one instruction)
    typedef unsigned pair_of __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(3))) pair_of* lds_pair;
    const uint32_t entry0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)tbl - (BASE << 2);
    auto entry = [&](const float sum) { return *(lds_pair)(uintptr_t)(entry0 + (__float_as_uint(sum) << 2)); };
    // (a tile's sums are on their way while the one before it is looked up)
    EngF4::Acc even = tile(0, 0), odd;
    auto group_scores = [&](const int grp, auto tail_c) {
        constexpr bool TAIL = decltype(tail_c)::value;       // some of the group's keys do not exist
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (j == 0) odd = tile(grp, 1);
            else even = tile(min(grp + 1, a.groups - 1), 0);
            const EngF4::Acc& acc = j == 0 ? even : odd;
            unsigned hs[8];
#pragma unroll
            for (int p = 0; p < 8; p++) {
                const pair_of e0 = entry(acc[2 * p]), e1 = entry(acc[2 * p + 1]);
                const int key = grp * 64 + 32 * h + 16 * j + 2 * p;
                s0 += !TAIL || key < S ? __uint_as_float(e0.x) : 0.f;
                s1 += !TAIL || key + 1 < S ? __uint_as_float(e1.x) : 0.f;
                hs[p] = __builtin_amdgcn_perm(e1.y, e0.y, 0x05040100u);
            }
            uint4* const to = reinterpret_cast<uint4*>(stage + c * ATTN_STAGE + 64 * h + 32 * j);
            to[0] = make_uint4(hs[0], hs[1], hs[2], hs[3]);
            to[1] = make_uint4(hs[4], hs[5], hs[6], hs[7]);
        }
        attn_wave_sync();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint4 x = *reinterpret_cast<const uint4*>(stage + (r8 + 8 * i) * ATTN_STAGE + c8 * 16);
            if constexpr (!TAIL) {
                const v4i v = {(int)x.x, (int)x.y, (int)x.z, (int)x.w};
                if (a.past) __builtin_amdgcn_raw_buffer_store_b128(v, rs, voff[i], grp * 128, 2);
                else __builtin_amdgcn_raw_buffer_store_b128(v, rs, voff[i], grp * 128, 0);
            } else {
                __half* const to = srow + (int64_t)(8 * i) * S + grp * 64;
                if (q0 + r8 + 8 * i < S) {
                    if (grp * 64 + c8 * 8 + 8 <= S) __builtin_memcpy(to, &x, 16);
                    else {
                        const unsigned d[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                        for (int e = 0; e < 7; e++)
                            if (grp * 64 + c8 * 8 + e < S) to[e] = __ushort_as_half((uint16_t)(d[e >> 1] >> (16 * (e & 1))));
                    }
                }
            }
        }
        attn_wave_sync();
    };
    const int whole = S / 64;
#pragma unroll 1
    for (int grp = 0; grp < whole; grp++) group_scores(grp, std::false_type{});
    if (whole < a.groups) group_scores(whole, std::true_type{});
    float total = s0 + s1;
    total += __shfl_xor(total, 32);

    // the fewest matching bits whose probability, rounded to fp16, reaches the level (D + 1: none does)
    int lo = 0, hi = D + 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (__half2float(__float2half_rn(__fdiv_rn(__uint_as_float(tbl[mid].x), total))) >= a.level) hi = mid;
        else lo = mid + 1;
    }
    // the sums less that level: negative where a probability counts as 0
#pragma unroll
    for (int v = 0; v < 16; v++) start[v] = both - (float)(2 * lo);

    // ---- bits of the probabilities, context --------------------------------------------------------------------------------------
    // ctx: keys that count and whose sign of V is negative
    EngF4::Acc ctx[W];
#pragma unroll
    for (int t = 0; t < W; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) ctx[t][v] = 0.f;
    int counted = 0;
    even = tile(0, 0);
#pragma unroll 1
    for (int grp = 0; grp < a.groups; grp++) {
        unsigned below = 0;               // key 32 h + r of the group at bit 31 - r: set where its probability counts as 0
        odd = tile(grp, 1);
#pragma unroll
        for (int v = 0; v < 16; v++) below = __builtin_amdgcn_alignbit(below, __float_as_uint(even[v]), 31);
        even = tile(min(grp + 1, a.groups - 1), 0);
#pragma unroll
        for (int v = 0; v < 16; v++) below = __builtin_amdgcn_alignbit(below, __float_as_uint(odd[v]), 31);
        const int left = S - (grp * 64 + 32 * h);
        if (left < 32) below |= left <= 0 ? 0xffffffffu : 0xffffffffu >> left;
        const unsigned counts = ~below;
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
    }
    counted += __shfl_xor(counted, 32);
    // the sum of the signs
#pragma unroll
    for (int t = 0; t < W; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) ctx[t][v] = fmaf(-2.f, ctx[t][v], (float)counted);
    if constexpr (BITS) {
        // a lane's 16 columns of its query, joined with the other half's: a word a head and 32 columns
        const float zp = !a.zp ? 0.f : a.f32 ? *reinterpret_cast<const float*>(a.zp) : __half2float(*reinterpret_cast<const __half*>(a.zp));
        uint32_t* const out = reinterpret_cast<uint32_t*>(a.context);
#pragma unroll
        for (int t = 0; t < W; t++) {
            unsigned w = 0;
#pragma unroll
            for (int v = 0; v < 16; v++) w = __builtin_amdgcn_alignbit(w, __float_as_uint(__fsub_rn(__half2float(__float2half_rn(ctx[t][v])), zp)), 31);
            w = w << 16 | __shfl_xor(w, 32);
            if (h == 0 && q0 + c < S) out[tiled_word_offset(row0 + q0 + c, head * W + t, a.KT)] = w;
        }
        if (head == a.heads - 1 && q0 + c < S)
            for (int64_t w = a.heads * W + h; w < a.KT * 8; w += 2) out[tiled_word_offset(row0 + q0 + c, w, a.KT)] = 0u;
        return;
    }
    if (q0 + c < S) {
        const int64_t at = ((row0 + q0 + c) * a.heads + head) * D + 16 * h;
#pragma unroll
        for (int t = 0; t < W; t++) {
            if (a.f32) {
                float4* const to = reinterpret_cast<float4*>(reinterpret_cast<float*>(a.context) + at + t * 32);
                auto f = [&](const int v) { return __half2float(__float2half_rn(ctx[t][v])); };
#pragma unroll
                for (int g = 0; g < 4; g++) to[g] = make_float4(f(4 * g), f(4 * g + 1), f(4 * g + 2), f(4 * g + 3));
            } else {
                union { __half x[16]; uint4 u[2]; } pk;
#pragma unroll
                for (int v = 0; v < 16; v++) pk.x[v] = __float2half_rn(ctx[t][v]);
                uint4* const to = reinterpret_cast<uint4*>(reinterpret_cast<__half*>(a.context) + at + t * 32);
                to[0] = pk.u[0]; to[1] = pk.u[1];
            }
        }
    }
}

}  // namespace bgemm

using namespace bgemm;

// Heads of 32, 64, 96 or 128 (whole words), and as many keys as leave a block's key and value bits within 32 KiB of LDS.
extern "C" int bgemm_attention_supported(int64_t batch, int64_t seq, int64_t heads, int64_t head_size)
{
    return batch >= 1 && seq >= 1 && heads >= 1 && head_size >= 32 && head_size <= 128 && head_size % 32 == 0 && seq * head_size <= (1 << 17) &&
           heads <= (1 << 17) && batch <= (1 << 24) && batch * heads * cdiv(seq, 32) <= 0x7fffffffLL && batch * seq <= 0x7fffffffLL;
}

static int attention(const char* who, const void* q, const void* k, const void* v, int64_t batch, int64_t seq, int64_t heads, int64_t head_size,
                     void* scores, void* context, const void* zero_point, bool bits, int context_type, void* stream)
{
    if (context_type != BGEMM_SRC_F16 && context_type != BGEMM_SRC_F32) return fail(BGEMM_EINVAL, "%s: context type %d", who, context_type);
    if (!bgemm_attention_supported(batch, seq, heads, head_size))
        return fail(BGEMM_EINVAL, "%s: %lld x %lld tokens, %lld heads of %lld", who, (long long)batch, (long long)seq, (long long)heads,
                    (long long)head_size);
    if (!q || !k || !v || !scores || !context) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)context) & 15 || (uintptr_t)scores & 1 ||
        (uintptr_t)zero_point & (context_type == BGEMM_SRC_F32 ? 3 : 1))
        return fail(BGEMM_EALIGN, "%s: operands and context must be 16-byte aligned", who);
    const int W = (int)head_size / 32;
    AttnArgs a = {(const uint32_t*)q, (const uint32_t*)k, (const uint32_t*)v, (__half*)scores, context, zero_point, k_tiles(heads * head_size)};
    a.S = (int)seq; a.heads = (int)heads; a.groups = (int)cdiv(seq, 64); a.f32 = context_type == BGEMM_SRC_F32; a.past = seq % 32 == 0 && ((uintptr_t)scores & 63) == 0;
    a.scale = 1.0f / (float)sqrt((double)head_size);
    a.level = (float)(1.0 / (double)seq);
    // Four waves share a block's operands, or eight where that needs no more rounds of waves a compute unit: what a block prepares is a
    // chain of its own, as long as a few groups of keys (us, heads of 64, 1 / 2 / 4 / 8 waves: 12 heads 4 x 512 tokens 33.7 / 27.2 / 19.6 /
    // 20.3, 8 x 512 39.5 / 28.7 / 24.2 / 20.8, 16 x 512 73.6 / 41.9 / 33.9 / 36.2, 4 heads 64 tokens 7.3 / 6.4 / 6.3 / 6.4).
    auto rounds = [&](const int w) { return cdiv(batch * heads * cdiv(seq, 32 * w), 256) * w; };
    auto lds_bytes = [&](const int w) { return (size_t)w * 32 * ATTN_STAGE + (head_size + 2) * 8 + (size_t)2 * W * a.groups * 64 * 4; };
    const int waves = rounds(8) <= rounds(4) && lds_bytes(8) <= (64 << 10) ? 8 : 4;
    a.qblocks = (int)cdiv(seq, 32 * waves);
    const size_t lds = lds_bytes(waves);
    const dim3 grid((unsigned)(batch * heads * a.qblocks)), block(waves * 64);
    const hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto numbers, auto as_bits) {
        if (bits) hipLaunchKernelGGL(as_bits, grid, block, lds, st, a);
        else hipLaunchKernelGGL(numbers, grid, block, lds, st, a);
    };
    switch (W) {
    case 1: go(attention_kernel<1, false>, attention_kernel<1, true>); break;
    case 2: go(attention_kernel<2, false>, attention_kernel<2, true>); break;
    case 3: go(attention_kernel<3, false>, attention_kernel<3, true>); break;
    default: go(attention_kernel<4, false>, attention_kernel<4, true>); break;
    }
    return check_launch(who);
}

extern "C" int bgemm_attention_forward(const void* q, const void* k, const void* v, int64_t batch, int64_t seq, int64_t heads, int64_t head_size,
                                       void* scores, void* context, int context_type, void* stream)
{
    return attention("bgemm_attention_forward", q, k, v, batch, seq, heads, head_size, scores, context, nullptr, false, context_type, stream);
}

extern "C" int bgemm_attention_forward_bits(const void* q, const void* k, const void* v, int64_t batch, int64_t seq, int64_t heads, int64_t head_size,
                                            void* scores, void* context_bits, const void* zero_point, int context_type, void* stream)
{
    return attention("bgemm_attention_forward_bits", q, k, v, batch, seq, heads, head_size, scores, context_bits, zero_point, true, context_type, stream);
}
