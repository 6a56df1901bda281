// Scaled binary Linear layers without a gradient in one launch, activations as they come: what tests/python/bgemm_linear.py:479-484 does
// in a centring pass, a pack, a GEMM and three elementwise passes.
//
//   y_l[n,m] = half(sum_k sign(x - zp_l)[n,k] sign(w_l)[m,k]) * sw_l[m] * sa_l (+ bias_l[m])          for up to three layers l of one input
//
// stored as numbers, with a residual added or not, or as the next layer's operand, the sign bits of y - next zero point.
#include "common.h"
#include "mfma_engines.h"
#include "pack_bits.h"
#include <type_traits>

namespace bgemm {

struct RowsLayer { const uint32_t* W; const void* zp; const void* sw; const void* sa; const void* bias; const void* next_zp; void* out; };

struct RowsArgs {
    RowsLayer l[3];
    const void* x; int64_t ld;        // unpacked rows (element stride), or one tiled operand of sign bits
    const void* residual;             // [N][M], or null
    int N, M, K, KT, MT, layers;
    int groups, splits, own;          // column groups of a layer, blocks a row tile, groups of a block (neighbours)
    int nt;                           // stores past the caches
    int first_lds;                    // bytes of the first area
    int gather;                       // bits of a whole row tile leave together: column tiles of the output, to the end of its last K-tile; else 0
};

enum { ROWS_BITS_F32 = 0, ROWS_BITS_F16 = 1, ROWS_F32 = 2, ROWS_F16 = 3 };
enum { ROWS_SRC_PACKED = 0, ROWS_SRC_F32 = 1, ROWS_SRC_F16 = 2 };
constexpr int ROWS_MAX_WAVES = 16;
constexpr int ROWS_MAX_K = 2048;      // up to here a sum is exact in fp16, and the rounding to it that the layer does is none

// fp4 operands whose products are -2 x where the weight's bit is set and 0 elsewhere, x = +-1, so that a sum that starts from the row's
// sum of x is the layer's: sum x (1 - 2 b).  The weight's bit stays where it is (0.5, 1, 2; at step 3 it moves to 1.0), five vector
// instructions a word; the activation is the sign over 2 / that value, from the inverted word.
__device__ __forceinline__ unsigned rows_w(const unsigned w, const int s) { return s == 3 ? (w >> 2) & 0x22222222u : w & (0x11111111u << s); }
__device__ __forceinline__ unsigned rows_x(const unsigned inverted, const int s)
{
    return ((inverted << (3 - s)) & 0x88888888u) | (s == 0 ? 0x66666666u : s == 2 ? 0x22222222u : 0x44444444u);
}

// A block owns one row tile of 32 activation rows.  Its waves turn them into sign bits in LDS, each layer's with that layer's zero
// point, then into matrix-core operands there (once: every column tile needs them), and take groups of CT column tiles in turn,
// whose weights come straight from the caches into registers, two K-tiles ahead.  The accumulators leave without a detour: a lane holds a
// column of sixteen rows (numbers: a half-wave stores a whole line; fp16 in pairs of columns), or with the operands exchanged sixteen
// columns of a row (bits: one instruction collects a sign, and whole 16-byte pieces of the output's tiles leave behind a barrier).
// What bounds it: numbers on many rows the stores, 8192 x 768 x 3072 fp32 25.3 us in place of 34.1 in two launches (101 MB of stores and
// 25 of reads, 5.0 TB/s; from and to memory, sets of buffers in turn, 26.5 for 37.8; fp16 17.7 for 26.7); bits the vector units, half of
// them the scaling: three layers 8192 x 768 x 768 14 us where three packs and three GEMMs took 46.7, each reading x and passing its outputs
// through LDS and a ballot a row; with a residual and a packed operand 8192 x 768 x 768 8.4 for 24.3 with the addition as its own pass.
// Few rows: the chain of one row tile, 64 x 512 x 512 4.5 for 7.6.
template <int SRC, int KIND, int CT>
__global__ __launch_bounds__(ROWS_MAX_WAVES * 64) void linear_rows_kernel(const RowsArgs a)
{
    constexpr bool BITS = KIND == ROWS_BITS_F32 || KIND == ROWS_BITS_F16, F32P = KIND == ROWS_BITS_F32 || KIND == ROWS_F32;
    static_assert(KIND != ROWS_F16 || CT % 2 == 0, "fp16 outputs leave in pairs of columns of two tiles");
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int h = lane >> 5, c = lane & 31;
    const unsigned id = xcd_contiguous_id(blockIdx.x, gridDim.x);
    const int rt = id / a.splits, part = id % a.splits;
    const int KT = a.KT, tiles_x = (SRC == ROWS_SRC_PACKED ? 1 : a.layers) * KT;
    uint4* const raw_bits = reinterpret_cast<uint4*>(smem);                 // [layer][K-tile][64]
    uint32_t* const words = reinterpret_cast<uint32_t*>(smem);              // BITS, in the same place later: [layer][column tile][row], tiles to the end of K-tiles
    uint4* const operands = reinterpret_cast<uint4*>(smem + a.first_lds);   // [layer][K-tile][step][64]
    float* const cols = reinterpret_cast<float*>(operands + tiles_x * 4 * TILE_U4);      // BITS: the block's columns' parameters, [layer][sw | bias][own * CT * 32]
    [[maybe_unused]] float* const xsums = cols + wave * 32;                 // else: the wave's row sums
    auto par = [](const void* p, const int64_t i) {
        if constexpr (F32P) return reinterpret_cast<const float*>(p)[i];
        else return __half2float(reinterpret_cast<const __half*>(p)[i]);
    };

    // ---- a wave's weights ----------------------------------------------------------------------------------------------------------
    const int g0 = part * a.own, g1 = min(a.groups, g0 + a.own), cols_n = a.own * CT * 32;
    // a wave works for one layer
    const int per_layer = waves / a.layers, l = wave / per_layer, wl = wave - l * per_layer, lx = SRC == ROWS_SRC_PACKED ? 0 : l;
    const RowsLayer& L = a.l[l];
    int gg = g0 + wl, kt = 0, rg = gg, rkt = 0;                       // the group that is multiplied, and the one whose weights are requested next
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(L.W), 0, a.MT * KT * 1024, 0x00020000);
    // which weight row a lane multiplies: bits: MFMA row 8 q + 4 half + i is column 16 half + 4 q + i, so that a lane ends up with 16
    // neighbouring columns of its row; fp16: the even rows of a pair of tiles, then the odd ones; else the lane's own
    const int own = BITS ? 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3) : c;
    auto request = [&](v4i (&w)[CT]) {
        const int mt0 = rg * CT;
#pragma unroll
        for (int j = 0; j < CT; j++) {
            if constexpr (KIND == ROWS_F16) {
                const int r = 2 * c + (j & 1), mt = min(mt0 + (j & ~1) + (r >> 5), a.MT - 1);
                w[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, mt * KT * 1024 + h * 512 + (r & 31) * 16, rkt * 1024, 0);
            } else
                w[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, h * 512 + own * 16, (min(mt0 + j, a.MT - 1) * KT + rkt) * 1024, 0);
        }
        if (++rkt == KT) {
            rkt = 0;
            rg += per_layer;                                           // (past the last one: the last tile again, nobody multiplies it)
        }
    };
    // Those of the first two K-tiles are on their way while the bits are made, where bits leave and little else fills that time (us:
    // 8192 x 768 x (3 x 768) 15.9 -> 15.4, 2048 x 768 x (3 x 768) 8.4 -> 8.0, 128 x 784 x 4096 7.2 -> 7.1; numbers, which have stores to
    // wait for: on packed rows 8192 x 768 x 3072 23.3 -> 23.7, fp16 4096 x 1024 x 1024 8.2 -> 8.3).
    v4i w0[CT], w1[CT], w2[CT];
    if constexpr (BITS) {
        request(w0);
        request(w1);
    }

    // ---- the rows' bits ----------------------------------------------------------------------------------------------------------
    if constexpr (SRC == ROWS_SRC_PACKED) {
        const uint4* const x = reinterpret_cast<const uint4*>(a.x) + (int64_t)rt * KT * TILE_U4;
        for (int i = threadIdx.x; i < KT * TILE_U4; i += waves * 64) raw_bits[i] = x[i];
    } else {
        constexpr bool F32 = SRC == ROWS_SRC_F32;
        typedef typename std::conditional<F32, uint32_t, uint16_t>::type E;
        const int last_row = min(a.N - rt * 32, 32) - 1;
        const E* const src = reinterpret_cast<const E*>(a.x) + (int64_t)rt * 32 * a.ld;
        float zf[3] = {0.f, 0.f, 0.f};
        for (int l = 0; l < a.layers; l++)
            if (a.l[l].zp) zf[l] = F32 ? *reinterpret_cast<const float*>(a.l[l].zp) : __half2float(*reinterpret_cast<const __half*>(a.l[l].zp));
        // a unit is two rows of a K-tile, a chunk of eight elements a lane; four of them requested at once
        // (K >= 8: a row's last chunk is read as its last eight elements, and the bits shifted into place)
        constexpr int AHEAD = 4;
        for (int u0 = wave; u0 < 16 * KT; u0 += waves * AHEAD) {
            Raw8<F32> raw[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                const int u = min(u0 + i * waves, 16 * KT - 1), r = (u & 15) * 2 + h;
                raw[i] = load_raw8<F32>(src + (int64_t)(r < last_row ? r : last_row) * a.ld, min((u >> 4) * TILE_KBITS + 8 * c, a.K - 8));
            }
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                const int u = min(u0 + i * waves, 16 * KT - 1), kt = u >> 4;           // (the last unit twice or more: the same bits)
                const int shift = min(max(kt * TILE_KBITS + 8 * c - (a.K - 8), 0), 8);
                unsigned char* const at = smem + kt * 1024 + tile_byte_of_chunk(c) + 16 * ((u & 15) * 2 + h);
                float f[8];
                centre8<F32>(raw[i], 0.f, f);
#pragma unroll
                for (int l = 0; l < 3; l++) {
                    if (l >= a.layers) break;
                    uint32_t sg = 0;
#pragma unroll
                    for (int e = 0; e < 8; e++) sg = __builtin_amdgcn_alignbit(sg, __float_as_uint(__fsub_rn(f[e], zf[l])), 31);
                    at[l * KT * 1024] = (unsigned char)(sg << shift);
                }
            }
        }
    }
    if constexpr (BITS) {
        for (int l = 0; l < a.layers; l++)
            for (int i = threadIdx.x; i < cols_n; i += waves * 64) {
                const int m = g0 * CT * 32 + i;
                cols[2 * l * cols_n + i] = m < a.M ? par(a.l[l].sw, m) : 0.f;
                cols[(2 * l + 1) * cols_n + i] = m < a.M && a.l[l].bias ? par(a.l[l].bias, m) : 0.f;
            }
    }
    __syncthreads();
    // the sum of the wave's x of row c
    int ones = 0;
#pragma unroll 1
    for (int t = 0; t < KT; t++) ones += popc4(raw_bits[(lx * KT + t) * TILE_U4 + lane]);
    ones += __shfl_xor(ones, 32);
    const float xsum = (float)(a.K - 2 * ones);
    for (int i = wave; i < tiles_x; i += waves) {
        const uint4 x = raw_bits[i * TILE_U4 + lane];
#pragma unroll
        for (int s = 0; s < 4; s++) operands[(i * 4 + s) * TILE_U4 + lane] = make_uint4(rows_x(~x.x, s), rows_x(~x.y, s), rows_x(~x.z, s), rows_x(~x.w, s));
    }
    __syncthreads();

    // ---- the products --------------------------------------------------------------------------------------------------------------
    const float sa = par(L.sa, 0), next = BITS && L.next_zp ? par(L.next_zp, 0) : 0.f;
    const bool has_bias = L.bias != nullptr, has_next = L.next_zp != nullptr;
    // the sums of x that the accumulators start from: BITS: the lane's row's, else those of its sixteen rows
    v16f acc[CT], start;
    if constexpr (BITS) {
#pragma unroll
        for (int v = 0; v < 16; v++) start[v] = xsum;
    } else {
        xsums[c] = xsum;                        // (both halves the same; the wave's own, LDS keeps its order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 s = *reinterpret_cast<const float4*>(xsums + 8 * q + 4 * h);
            start[4 * q] = s.x; start[4 * q + 1] = s.y; start[4 * q + 2] = s.z; start[4 * q + 3] = s.w;
        }
    }
    // numbers leave, and a residual comes, through buffers that end with the last row: what lies past it is dropped (and read as 0)
    constexpr int ESZ = F32P ? 4 : 2;
    const int row_b = a.M * ESZ, rows_b = min(a.N - rt * 32, 32) * row_b;
    auto rows_of = [&](const void* p) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(p)) + (int64_t)rt * 32 * row_b, 0, rows_b, 0x00020000);
    };
    auto store_group = [&] {
        const int mt0 = gg * CT;
        if constexpr (BITS) {
            const int n = rt * 32 + c;
#pragma unroll
            for (int j = 0; j < CT; j++) {
                const int mt = mt0 + j;
                if (mt >= a.MT) break;
                const float* const ps = cols + 2 * l * cols_n + (mt - g0 * CT) * 32 + 16 * h;
                const float* const pb = ps + cols_n;
                unsigned bits = 0;
                auto collect = [&](auto bias_c, auto next_c) {
                    constexpr bool BIAS = decltype(bias_c)::value, NEXT = decltype(next_c)::value;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float4 s4 = *reinterpret_cast<const float4*>(ps + 4 * q), b4 = BIAS ? *reinterpret_cast<const float4*>(pb + 4 * q) : float4{};
                        const float s[4] = {s4.x, s4.y, s4.z, s4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
                        for (int e = 0; e < 4; e++) {
#pragma clang fp contract(off)      // every step rounds by itself, as torch's separate kernels do
                            float y;
                            if constexpr (F32P) {
                                y = acc[j][4 * q + e] * s[e];
                                y = y * sa;
                                if (BIAS) y = y + b[e];
                            } else {
                                _Float16 r = (_Float16)acc[j][4 * q + e] * (_Float16)s[e];
                                r = r * (_Float16)sa;
                                if (BIAS) r = r + (_Float16)b[e];
                                y = (float)r;
                            }
                            bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(NEXT ? y - next : y), 31);
                        }
                    }
                };
                if (!has_bias) collect(std::false_type{}, std::true_type{});
                else if (has_next) collect(std::true_type{}, std::true_type{});
                else collect(std::true_type{}, std::false_type{});
                const unsigned other = __shfl_xor(bits, 32);
                unsigned word = bits << 16 | other;
                if ((mt + 1) * 32 > a.M) word &= 0xffffffffu << ((mt + 1) * 32 - a.M);
                if (a.gather) {
                    if (h == 0) words[(l * a.gather + mt) * 32 + c] = word;
                } else if (h == 0 && n < a.N) reinterpret_cast<uint32_t*>(L.out)[tiled_word_offset(n, mt, k_tiles(a.M))] = word;
            }
        } else if constexpr (KIND == ROWS_F32) {
            const __amdgpu_buffer_rsrc_t ro = rows_of(L.out), rr = rows_of(a.residual);
#pragma unroll
            for (int j = 0; j < CT; j++) {
                const int mt = mt0 + j, m = mt * 32 + c;
                if (mt >= a.MT) break;
                const int mc = m < a.M ? m : a.M - 1, voff = m < a.M ? 4 * h * row_b + m * 4 : 0x7ffffff0;
                const float s = par(L.sw, mc), b = has_bias ? par(L.bias, mc) : 0.f;
                float y[16], res[16];
                if (a.residual)
#pragma unroll
                    for (int v = 0; v < 16; v++) res[v] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr, voff, (8 * (v >> 2) + (v & 3)) * row_b, 0));
#pragma unroll
                for (int v = 0; v < 16; v++) {
#pragma clang fp contract(off)      // every step rounds by itself, as torch's separate kernels do
                    y[v] = acc[j][v] * s;
                    y[v] = y[v] * sa;
                }
                if (has_bias)
#pragma unroll
                    for (int v = 0; v < 16; v++) y[v] = __fadd_rn(y[v], b);
                if (a.residual)
#pragma unroll
                    for (int v = 0; v < 16; v++) y[v] = __fadd_rn(y[v], res[v]);
                if (a.nt) {
#pragma unroll
                    for (int v = 0; v < 16; v++) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[v]), ro, voff, (8 * (v >> 2) + (v & 3)) * row_b, 2);
                } else {
#pragma unroll
                    for (int v = 0; v < 16; v++) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[v]), ro, voff, (8 * (v >> 2) + (v & 3)) * row_b, 0);
                }
            }
        } else {
            const __amdgpu_buffer_rsrc_t ro = rows_of(L.out), rr = rows_of(a.residual);
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int p = 0; p < CT / 2; p++) {
                const int mt = mt0 + 2 * p, m = mt * 32 + 2 * c;
                if (mt >= a.MT) break;
                // (the last column of an odd number stands alone)
                const bool pair = m + 1 < a.M, single = m + 1 == a.M;
                const int voff = pair ? 4 * h * row_b + m * 2 : 0x7ffffff0, voff1 = single ? 4 * h * row_b + m * 2 : 0x7ffffff0;
                h2 s = {(_Float16)0.f, (_Float16)0.f}, b = s;
                if (pair || single) {
                    s[0] = reinterpret_cast<const _Float16*>(L.sw)[m];
                    s[1] = reinterpret_cast<const _Float16*>(L.sw)[pair ? m + 1 : m];
                    if (has_bias) {
                        b[0] = reinterpret_cast<const _Float16*>(L.bias)[m];
                        b[1] = reinterpret_cast<const _Float16*>(L.bias)[pair ? m + 1 : m];
                    }
                }
                const h2 sah = {(_Float16)sa, (_Float16)sa};
                h2 y[16];
                unsigned res[16];
                if (a.residual)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const int o = (8 * (v >> 2) + (v & 3)) * row_b;
                        res[v] = __builtin_amdgcn_raw_buffer_load_b32(rr, voff, o, 0);
                        if (a.M & 1) res[v] |= __builtin_amdgcn_raw_buffer_load_b16(rr, voff1, o, 0);
                    }
#pragma unroll
                for (int v = 0; v < 16; v++) {
#pragma clang fp contract(off)
                    y[v][0] = (_Float16)acc[2 * p][v];
                    y[v][1] = (_Float16)acc[2 * p + 1][v];
                    y[v] = y[v] * s;
                    y[v] = y[v] * sah;
                }
                if (has_bias)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
#pragma clang fp contract(off)
                        y[v] = y[v] + b;
                    }
                if (a.residual)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
#pragma clang fp contract(off)
                        y[v] = y[v] + __builtin_bit_cast(h2, res[v]);
                    }
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int o = (8 * (v >> 2) + (v & 3)) * row_b;
                    const unsigned u = __builtin_bit_cast(unsigned, y[v]);
                    if (a.nt) __builtin_amdgcn_raw_buffer_store_b32(u, ro, voff, o, 2);
                    else __builtin_amdgcn_raw_buffer_store_b32(u, ro, voff, o, 0);
                    if (a.M & 1) __builtin_amdgcn_raw_buffer_store_b16((unsigned short)u, ro, voff1, o, 0);
                }
            }
        }
    };
    auto step = [&](const v4i (&w)[CT]) {
        const uint4* const op = operands + (lx * KT + kt) * 4 * TILE_U4 + lane;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const uint4 x = op[s * TILE_U4];
            const unsigned fx[4] = {x.x, x.y, x.z, x.w};
            unsigned fw[CT][4];
#pragma unroll
            for (int j = 0; j < CT; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) fw[j][q] = rows_w((unsigned)w[j][q], s);
            auto multiply = [&](auto first_c) {
#pragma unroll
                for (int j = 0; j < CT; j++) {
                    const v16f& from = decltype(first_c)::value ? start : acc[j];
                    if constexpr (BITS) acc[j] = EngF4::mma(EngF4::make(fw[j]), EngF4::make(fx), from);
                    else acc[j] = EngF4::mma(EngF4::make(fx), EngF4::make(fw[j]), from);
                }
            };
            if (s == 0 && kt == 0) multiply(std::true_type{});
            else multiply(std::false_type{});
        }
        if (++kt == KT) {
            store_group();
            kt = 0;
            gg += per_layer;
        }
    };
    if (gg < g1) {
        if constexpr (!BITS) {
            request(w0);
            request(w1);
        }
        for (;;) {
            request(w2);
            step(w0);
            if (gg >= g1) break;
            request(w0);
            step(w1);
            if (gg >= g1) break;
            request(w1);
            step(w2);
            if (gg >= g1) break;
        }
    }
    if (BITS && !a.gather && a.MT % 8 && g1 == a.groups) {
        // the block with the rows' last words ends them
        for (int i = threadIdx.x; i < a.layers * 32; i += waves * 64)
            if (rt * 32 + i % 32 < a.N) end_bits_row(reinterpret_cast<uint32_t*>(a.l[i / 32].out), rt * 32 + i % 32, a.M);
    }
    if (BITS && a.gather) {
        // whole tiles of the output, their padding of zeros included
        for (int i = threadIdx.x; i < a.layers * (a.gather - a.MT) * 32; i += waves * 64) words[(i / ((a.gather - a.MT) * 32) * a.gather + a.MT) * 32 + i % ((a.gather - a.MT) * 32)] = 0u;
        __syncthreads();
        for (int i = threadIdx.x; i < a.layers * a.gather * 8; i += waves * 64) {
            const int l = i / (a.gather * 8), j = i - l * a.gather * 8, r = j & 31, q4 = j >> 5;      // words 4 q4 .. of row r
            const uint32_t* const from = words + (l * a.gather + 4 * q4) * 32 + r;
            if (rt * 32 + r < a.N)
                *reinterpret_cast<uint4*>(reinterpret_cast<uint32_t*>(a.l[l].out) + ((int64_t)rt * (a.gather / 8) * TILE_U4 + j) * 4) = make_uint4(from[0], from[32], from[64], from[96]);
        }
    }
}

// A layer of packed rows whose fp32 outputs, plus a residual, go through a layer norm: as the numbers kernel above, but a block keeps all
// columns of its rows in registers, a wave CT column tiles, until their mean and deviation are known, so that they are stored once.
struct RowsNorm { const float* gamma; const float* beta; double eps, share; };      // (either pointer may be null; share: 1 / M)
constexpr int NORM_MAX_KT = 4, NORM_MAX_M = ROWS_MAX_WAVES * 64;

// Rows' mean, then the mean square of what is left (two passes over registers: nothing cancels), each a sum over 32 lanes and the waves.
// What bounds it: reading the residual and storing, one block a compute unit; the residual and all weights are requested before the
// bits are there.  8192 x 768 x 768 27.0 us with the layer norm as a launch of its own (25 MB written and read again), 11.9 here (50 MB
// of residual and stores, 4.2 TB/s); its relative error to 64 bits 4.0e-8 where that of the separate one is 4.6e-8.
template <int CT>
__global__ __launch_bounds__(ROWS_MAX_WAVES * 64) void rows_norm_kernel(const RowsArgs a, const RowsNorm norm)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int h = lane >> 5, c = lane & 31;
    const int rt = xcd_contiguous_id(blockIdx.x, gridDim.x), KT = a.KT, mt0 = wave * CT;
    uint4* const raw_bits = reinterpret_cast<uint4*>(smem);                 // [K-tile][64]
    uint4* const operands = raw_bits + KT * TILE_U4;                        // [K-tile][step][64]
    float* const shares = reinterpret_cast<float*>(operands + KT * 4 * TILE_U4);      // [2][wave][row]: the waves' shares of the sums
    float* const mine = shares + (2 * waves + wave) * 32;                   // a value a row, for the wave's lanes
    const RowsLayer& L = a.l[0];
    const uint4* const x = reinterpret_cast<const uint4*>(a.x) + (int64_t)rt * KT * TILE_U4;
    for (int i = threadIdx.x; i < KT * TILE_U4; i += waves * 64) raw_bits[i] = x[i];
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(L.W), 0, a.MT * KT * 1024, 0x00020000);
    v4i w[NORM_MAX_KT][CT];
#pragma unroll
    for (int kt = 0; kt < NORM_MAX_KT; kt++)
#pragma unroll
        for (int j = 0; j < CT; j++)
            w[kt][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, h * 512 + c * 16, (min(mt0 + j, a.MT - 1) * KT + min(kt, KT - 1)) * 1024, 0);
    const int row_b = a.M * 4, rows_b = min(a.N - rt * 32, 32) * row_b;
    auto rows_of = [&](const void* p) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(p)) + (int64_t)rt * 32 * row_b, 0, rows_b, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ro = rows_of(L.out), rr = rows_of(a.residual);
    int voff[CT];                                                           // (columns past the last one: past the buffer's end)
    float y[CT][16];
#pragma unroll
    for (int j = 0; j < CT; j++) {
        const int m = (mt0 + j) * 32 + c;
        voff[j] = m < a.M ? 4 * h * row_b + m * 4 : 0x7ffffff0;
#pragma unroll
        for (int v = 0; v < 16; v++) y[j][v] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr, voff[j], (8 * (v >> 2) + (v & 3)) * row_b, 0));
    }
    __syncthreads();
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // the wave's values a row, as the lane's sixteen rows have them
    auto of_rows = [&](const float value, float (&to)[16]) {
        wave_sync();
        mine[c] = value;                        // (both halves the same)
        wave_sync();
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 s = *reinterpret_cast<const float4*>(mine + 8 * q + 4 * h);
            to[4 * q] = s.x; to[4 * q + 1] = s.y; to[4 * q + 2] = s.z; to[4 * q + 3] = s.w;
        }
    };
    int ones = 0;
    for (int t = 0; t < KT; t++) ones += popc4(raw_bits[t * TILE_U4 + lane]);
    ones += __shfl_xor(ones, 32);
    for (int i = wave; i < KT; i += waves) {
        const uint4 b = raw_bits[i * TILE_U4 + lane];
#pragma unroll
        for (int s = 0; s < 4; s++) operands[(i * 4 + s) * TILE_U4 + lane] = make_uint4(rows_x(~b.x, s), rows_x(~b.y, s), rows_x(~b.z, s), rows_x(~b.w, s));
    }
    float start[16];
    of_rows((float)(a.K - 2 * ones), start);
    v16f acc[CT];
#pragma unroll
    for (int j = 0; j < CT; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[j][v] = start[v];
    __syncthreads();
#pragma unroll
    for (int kt = 0; kt < NORM_MAX_KT; kt++) {
        if (kt >= KT) break;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const uint4 b = operands[(kt * 4 + s) * TILE_U4 + lane];
            const unsigned fx[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int j = 0; j < CT; j++) {
                unsigned fw[4];
#pragma unroll
                for (int q = 0; q < 4; q++) fw[q] = rows_w((unsigned)w[kt][j][q], s);
                acc[j] = EngF4::mma(EngF4::make(fx), EngF4::make(fw), acc[j]);
            }
        }
    }
    const float sa = *reinterpret_cast<const float*>(L.sa);
#pragma unroll
    for (int j = 0; j < CT; j++) {
        const int m = min((mt0 + j) * 32 + c, a.M - 1);
        const float s = reinterpret_cast<const float*>(L.sw)[m], b = L.bias ? reinterpret_cast<const float*>(L.bias)[m] : 0.f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
#pragma clang fp contract(off)      // every step rounds by itself, as torch's separate kernels do
            float t = acc[j][v] * s;
            t = t * sa;
            if (L.bias) t = t + b;
            y[j][v] = t + y[j][v];
        }
    }
    // the sum of a lane's sixteen values over the block's columns, of row c
    auto over_columns = [&](float (&s)[16], float* const area) {
        // lanes d apart share the work: each keeps one half of the values (v = c >> 1 in the end)
        auto halve = [&](auto d_c) {
            constexpr int d = decltype(d_c)::value;
            const bool upper = c & d;
#pragma unroll
            for (int i = 0; i < d / 2; i++) {
                const float keep = upper ? s[i + d / 2] : s[i], give = upper ? s[i] : s[i + d / 2];
                s[i] = keep + __shfl_xor(give, d);
            }
        };
        halve(std::integral_constant<int, 16>{});
        halve(std::integral_constant<int, 8>{});
        halve(std::integral_constant<int, 4>{});
        halve(std::integral_constant<int, 2>{});
        s[0] += __shfl_xor(s[0], 1);
        const int v = c >> 1;
        if (!(c & 1)) area[wave * 32 + 8 * (v >> 2) + 4 * h + (v & 3)] = s[0];
        __syncthreads();
        double t = 0.;                          // (a value a lane: in 64 bits, as what follows from it, for nothing)
#pragma unroll 4
        for (int i = 0; i < waves; i++) t += (double)area[i * 32 + c];
        return t;
    };
    float sum[16], of[16];
#pragma unroll
    for (int v = 0; v < 16; v++) {
        sum[v] = 0.f;
#pragma unroll
        for (int j = 0; j < CT; j++) sum[v] += voff[j] == 0x7ffffff0 ? 0.f : y[j][v];
    }
    of_rows((float)(over_columns(sum, shares) * norm.share), of);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        sum[v] = 0.f;
#pragma unroll
        for (int j = 0; j < CT; j++) {
            y[j][v] -= of[v];
            sum[v] += voff[j] == 0x7ffffff0 ? 0.f : y[j][v] * y[j][v];
        }
    }
    of_rows((float)rsqrt(over_columns(sum, shares + waves * 32) * norm.share + norm.eps), of);
#pragma unroll
    for (int j = 0; j < CT; j++) {
        const int m = min((mt0 + j) * 32 + c, a.M - 1);
        const float g = norm.gamma ? norm.gamma[m] : 1.f, b = norm.beta ? norm.beta[m] : 0.f;
#pragma unroll
        for (int v = 0; v < 16; v++) y[j][v] = y[j][v] * of[v] * g + b;
        if (a.nt) {
#pragma unroll
            for (int v = 0; v < 16; v++) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[j][v]), ro, voff[j], (8 * (v >> 2) + (v & 3)) * row_b, 2);
        } else {
#pragma unroll
            for (int v = 0; v < 16; v++) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[j][v]), ro, voff[j], (8 * (v >> 2) + (v & 3)) * row_b, 0);
        }
    }
}

// How a size is launched, and what a block keeps in LDS: the rows' bits, later those of the output, and operands for every layer, and where
// bits leave the parameters of its columns.
struct RowsPlan { int64_t ct, per_layer, splits, groups, own, first_lds, lds; };

static RowsPlan rows_plan(int64_t N, int64_t M, int64_t K, int layers, bool packed, int out_dtype, int shape)
{
    RowsPlan p;
    const bool bits = out_dtype == BGEMM_OUT_BITS_F32 || out_dtype == BGEMM_OUT_BITS_F16, f32 = out_dtype == BGEMM_OUT_BITS_F32 || out_dtype == BGEMM_OUT_F32_SCALED;
    const int64_t rt = row_tiles(N);
    // How many column tiles a wave multiplies at once, how many waves a layer has in a block, how many blocks share a row tile.
    // Numbers, one tile (fp16: a pair), eight waves, as many blocks as there are groups for up to two a compute unit, one storing while the
    // other makes its bits (us, 16 waves and one block / 8 and two, from and to memory, on a kernel that is 10 % faster now: fp32 8192 x 768 x 3072 29.0 / 28.9, x 1008 16.0 /
    // 14.9; fp16 20.3 / 19.3; 512 x 512 x 2048 7.1 / 5.7).  Beyond K = 1024 making them again costs more than that, fp32 rows of 16 KiB meet
    // on the same memory channels when more blocks store at a time (8192 x 256 x 4096 30.7 / 37.1), and bits have nothing to store: one
    // block a compute unit, of as many waves as give each a tile or two (2048 x 2048 x 2048 10.8, in two blocks of eight 13.7; 8192 x
    // 768 x (3 x 768) bits 14 and 20).  Two tiles at once share an operand's reads from LDS: bits from sixteen tiles a
    // compute unit on (8192 x 768 x (3 x 768) 15.3 -> 14.4, but 100 rows 7.2 -> 8.1).
    const int64_t tiles = rt * row_tiles(M);
    const bool f16_numbers = out_dtype == BGEMM_OUT_F16_SCALED, one_a_unit = bits || K > 1024 || (f32 && M >= 4096);
    p.ct = f16_numbers ? 2 : shape ? shape & 15 : bits && layers * tiles >= 4096 ? 2 : 1;
    p.groups = cdiv(row_tiles(M), p.ct);
    p.per_layer = 8 / layers;
    if (one_a_unit) {
        const int64_t want = cdiv(cdiv(rt * p.groups, 256), 4) * 4, most = layers == 3 ? 4 : ROWS_MAX_WAVES / layers;
        // (one layer at least eight: the waves make the bits of 32 rows together, on few rows four of them in as many trips to memory as
        // their products take: bits 128 x 784 x 4096 fp16 7.0 -> 5.7, fp32 5.9 -> 5.2; 512 x 1000 x 2048 6.1 -> 5.2; 40 x 1024 x 4096 7.0 ->
        // 5.6; 64 x 512 x 1024 4.4 -> 4.0; sixteen 5.8, 5.3, 5.6, 5.7, 4.1; three layers have twelve)
        const int64_t least = layers == 1 ? 8 : 4;
        p.per_layer = want < least ? least : want > most ? most : want;
    }
    if (shape) p.per_layer = shape >> 4 & 31;
    p.splits = cdiv(p.groups, p.per_layer);
    while (p.splits > 1 && rt * p.splits > (one_a_unit ? 256 : 512)) p.splits--;
    if (shape >> 12) p.splits = shape >> 12;
    p.own = cdiv(p.groups, p.splits);
    p.splits = cdiv(p.groups, p.own);
    const int planes = packed ? 1 : layers;
    const int64_t in = planes * k_tiles(K) * 1024, out = bits && p.splits == 1 ? layers * k_tiles(M) * 1024 : 0;
    p.first_lds = in > out ? in : out;
    p.lds = p.first_lds + planes * k_tiles(K) * 4096 + (bits ? layers * p.own * p.ct * 32 * 8 : ROWS_MAX_WAVES * 128);
    return p;
}

// fp32 numbers of which there are more than the caches take, on rows that share lines of 128 bytes and on a K so short that little but their
// stores is left: a GEMM's tiles finish such lines sooner than blocks that share a row tile (us, pack and GEMM / here: 16384 x 128 x 3000 51 / 65, x
// 768 64 / 73, but x 1024 69 / 71 and 16384 x 1024 x 4100 135 / 106; rows that share no 64 bytes 16384 x 128 x 6000 84 / 103, x 512 99 / 105, but x
// 768 112 / 104; half as many numbers 8192 x 128 x 4100 36.7 / 31.0).
bool linear_rows_past_caches(int64_t N, int64_t M, int64_t K, int out_dtype)
{
    return out_dtype == BGEMM_OUT_F32_SCALED && N * M > (40 << 20) && M % 32 && k_tiles(K) <= (M % 16 ? 3 : 2);
}

}  // namespace bgemm

using namespace bgemm;

extern "C" int bgemm_linear_rows_supported(int64_t N, int64_t M, int64_t K, int layers, int out_dtype)
{
    if (out_dtype != BGEMM_OUT_F32_SCALED && out_dtype != BGEMM_OUT_F16_SCALED && out_dtype != BGEMM_OUT_BITS_F32 && out_dtype != BGEMM_OUT_BITS_F16) return 0;
    if (N < 1 || N > (1 << 24) || M < 1 || M > (1 << 16) || K < 8 || K > ROWS_MAX_K || layers < 1 || layers > 3 ||
        rows_plan(N, M, K, layers, false, out_dtype, 0).lds > (64 << 10))
        return 0;
    // Against a pack and a GEMM (one layer, N = 5 .. 8192, M = 256 .. 22016, both types).  On few rows its time is that of one wave's walk
    // over K, which the decode kernels split among their waves: us, two launches / this one, fp32 32 x 512 x 4096 7.3 / 4.5, 32 x 1000 x
    // 4096 6.5 / 5.8 but 16 x 1000 x 1000 5.9 / 6.0, 128 x 1536 x 4096 7.4 / 7.7 and 512 x 1536 x 4096 10.1 / 7.8, 512 x 2048 x 1000 7.8 / 9.0
    // and 2048 x 2048 x 1000 12.4 / 10.9.  Beyond 16384 columns a few hundred rows are too few for a block a row tile to share them
    // (512 x 2048 x 22016 22.2 / 26.7, fp16 512 x 1000 x 22016 15.1 / 16.1).  Bits (one layer, fp32 32 x 512 x 4096 8.6 / 4.4, 1 x 512 x 512 5.2 /
    // 4.1, 512 x 1500 x 4096 10.0 / 7.2, 2048 x 2048 x 512 11.5 / 7.9) are ahead on fewer rows than that, already on 8 at three or four K-tiles and on 32 at six
    // (32 x 1024 x 512 7.2 / 5.3, 128 x 1500 x 512 7.5 / 6.6; 1 x 1500 x 512 5.3 / 6.3, 128 x 2048 x 512 6.8 / 7.7), never behind where this says 2.
    // Three layers' bits are ahead wherever they are taken (1 x 1024 x (3 x 1024) six launches 15.3, one 7.6), and a residual on a packed operand
    // beside a pack, a GEMM and the addition from two rows on (4 x 2048 x 2048 fp32 5.9 / 5.3, 256 rows 10.0 / 5.6; one row 4.9 / 5.3, four fp16 5.8 /
    // 7.0: no more than the launches that fall away cost the host).
    const int64_t KT = k_tiles(K), rows = KT <= 2 ? 1 : KT <= 4 ? 33 : KT <= 6 ? 512 : 2048;
    return N >= rows && (M <= 16384 || N < 256) && !linear_rows_past_caches(N, M, K, out_dtype) ? 2 : 1;
}

extern "C" int bgemm_linear_rows_forward(const void* x, int x_dtype, int64_t ldx, int64_t N, int64_t M, int64_t K, int layers,
                                         const bgemm_rows_layer* layer, int out_dtype, const void* residual, int shape, void* stream)
{
    const char* who = "bgemm_linear_rows_forward";
    const bool bits = out_dtype == BGEMM_OUT_BITS_F32 || out_dtype == BGEMM_OUT_BITS_F16;
    const bool f32 = out_dtype == BGEMM_OUT_BITS_F32 || out_dtype == BGEMM_OUT_F32_SCALED, packed = x_dtype == BGEMM_SRC_BITS;
    if (!bgemm_linear_rows_supported(N, M, K, layers, out_dtype))
        return fail(BGEMM_EINVAL, "%s: N=%lld M=%lld K=%lld, %d layers, output %d", who, (long long)N, (long long)M, (long long)K, layers, out_dtype);
    if (!packed && x_dtype != (f32 ? BGEMM_SRC_F32 : BGEMM_SRC_F16)) return fail(BGEMM_EINVAL, "%s: activations of type %d for that output", who, x_dtype);
    if (!packed && ldx < K) return fail(BGEMM_EINVAL, "%s: row stride %lld < K", who, (long long)ldx);
    if (residual && bits) return fail(BGEMM_EINVAL, "%s: a residual is added to numbers", who);
    if (shape && (shape < 0 || (shape & 15) < 1 || (shape & 15) > 2 || (shape >> 4 & 31) < 1 || (shape >> 4 & 31) * layers > ROWS_MAX_WAVES || shape >> 22))
        return fail(BGEMM_EINVAL, "%s: launch shape %d", who, shape);
    if (!x || !layer) return fail(BGEMM_ENULL, "%s: null pointer", who);
    const unsigned odd = f32 ? 3 : 1;
    if (((uintptr_t)x & (packed ? 15 : odd)) || ((uintptr_t)residual & odd)) return fail(BGEMM_EALIGN, "%s: an operand is not aligned", who);
    RowsArgs a = {};
    for (int l = 0; l < layers; l++) {
        const bgemm_rows_layer& s = layer[l];
        if (!s.W_tiled || !s.sw || !s.sa || !s.out) return fail(BGEMM_ENULL, "%s: layer %d: null pointer", who, l);
        if (((uintptr_t)s.W_tiled & 15) || ((uintptr_t)s.out & (bits ? 15 : odd)) || (((uintptr_t)s.sw | (uintptr_t)s.sa | (uintptr_t)s.bias | (uintptr_t)s.zero_point | (uintptr_t)s.next_zero_point) & odd))
            return fail(BGEMM_EALIGN, "%s: layer %d: an operand is not aligned", who, l);
        a.l[l] = {(const uint32_t*)s.W_tiled, packed ? nullptr : s.zero_point, s.sw, s.sa, s.bias, bits ? s.next_zero_point : nullptr, s.out};
    }
    a.x = x; a.ld = ldx; a.residual = residual;
    a.N = (int)N; a.M = (int)M; a.K = (int)K; a.KT = (int)k_tiles(K); a.MT = (int)row_tiles(M); a.layers = layers;
    const RowsPlan p = rows_plan(N, M, K, layers, packed, out_dtype, shape);
    if (p.lds > (64 << 10)) return fail(BGEMM_EINVAL, "%s: launch shape %d needs %lld bytes of LDS", who, shape, (long long)p.lds);
    a.groups = (int)p.groups; a.splits = (int)p.splits; a.own = (int)p.own;
    a.first_lds = (int)p.first_lds;
    a.gather = bits && p.splits == 1 ? (int)k_tiles(M) * 8 : 0;
    // Past the caches where no two blocks share a 64-byte piece of a row (from and to memory, on a kernel that is 10 % faster now: fp32 8192 x 768 x 3072 34.3 -> 28.9, 4096 x 1024 x 4096 26.6 ->
    // 19.7, fp16 8192 x 768 x 768 12.9 -> 11.0; rows of 4000 bytes 19.0 -> 20.3, of fp16 6176 26.5 -> 28.6).
    a.nt = M * (f32 ? 4 : 2) % 64 == 0;
    const size_t lds = (size_t)p.lds;
    const int ct = (int)p.ct;
    const dim3 grid((unsigned)(row_tiles(N) * p.splits)), block((unsigned)(layers * p.per_layer * 64));
    const hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto src, auto kind) {
        constexpr int SRC = decltype(src)::value, KIND = decltype(kind)::value;
        if constexpr (KIND != ROWS_F16) {
            if (ct == 1) hipLaunchKernelGGL((linear_rows_kernel<SRC, KIND, 1>), grid, block, lds, st, a);
        }
        if (ct == 2) hipLaunchKernelGGL((linear_rows_kernel<SRC, KIND, 2>), grid, block, lds, st, a);
    };
    auto kinds = [&](auto src32, auto src16) {
        if (out_dtype == BGEMM_OUT_BITS_F32) go(src32, std::integral_constant<int, ROWS_BITS_F32>{});
        else if (out_dtype == BGEMM_OUT_BITS_F16) go(src16, std::integral_constant<int, ROWS_BITS_F16>{});
        else if (out_dtype == BGEMM_OUT_F32_SCALED) go(src32, std::integral_constant<int, ROWS_F32>{});
        else go(src16, std::integral_constant<int, ROWS_F16>{});
    };
    typedef std::integral_constant<int, ROWS_SRC_PACKED> P;
    if (packed) kinds(P{}, P{});
    else kinds(std::integral_constant<int, ROWS_SRC_F32>{}, std::integral_constant<int, ROWS_SRC_F16>{});
    return check_launch(who);
}

extern "C" int bgemm_linear_rows_norm_supported(int64_t N, int64_t M, int64_t K)
{
    if (N < 1 || N > (1 << 24) || M < 1 || M > NORM_MAX_M || K < 1 || K > NORM_MAX_KT * TILE_KBITS) return 0;
    // Against the layer with its residual and the layer norm as a launch of its own (us, N x M x M, two launches / this one): 8192 x
    // 768 27.0 / 11.9, 2048 x 768 11.6 / 9.8, 1024 x 768 9.7 / 9.8, 512 x 768 8.4 / 9.7, 2048 x 1024 13.5 / 12.3, 1024 x 1024 10.6 / 12.3; 1024 x
    // 512 8.3 / 7.7, 512 x 512 7.8 / 7.6.  (512 x 64 6.6 / 4.0, but the call around so few rows is the host's time either way, and its sums
    // are in the separate one's order.)
    return N >= (M <= 512 ? 1024 : 2048) ? 2 : 1;
}

extern "C" int bgemm_linear_rows_norm_forward(const void* x_tiled, int64_t N, int64_t M, int64_t K, const bgemm_rows_layer* layer, const void* residual,
                                              const void* gamma, const void* beta, double eps, void* stream)
{
    const char* who = "bgemm_linear_rows_norm_forward";
    if (!bgemm_linear_rows_norm_supported(N, M, K)) return fail(BGEMM_EINVAL, "%s: N=%lld M=%lld K=%lld", who, (long long)N, (long long)M, (long long)K);
    if (!x_tiled || !layer || !residual) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (!layer->W_tiled || !layer->sw || !layer->sa || !layer->out) return fail(BGEMM_ENULL, "%s: the layer: null pointer", who);
    if ((((uintptr_t)x_tiled | (uintptr_t)layer->W_tiled) & 15) ||
        (((uintptr_t)residual | (uintptr_t)layer->sw | (uintptr_t)layer->sa | (uintptr_t)layer->bias | (uintptr_t)layer->out | (uintptr_t)gamma | (uintptr_t)beta) & 3))
        return fail(BGEMM_EALIGN, "%s: an operand is not aligned", who);
    RowsArgs a = {};
    a.l[0] = {(const uint32_t*)layer->W_tiled, nullptr, layer->sw, layer->sa, layer->bias, nullptr, layer->out};
    a.x = x_tiled; a.residual = residual;
    a.N = (int)N; a.M = (int)M; a.K = (int)K; a.KT = (int)k_tiles(K); a.MT = (int)row_tiles(M); a.layers = 1;
    a.nt = M % 16 == 0;                     // (as above)
    // one column tile a wave while sixteen waves are enough
    const int ct = a.MT <= ROWS_MAX_WAVES ? 1 : 2, waves = (a.MT + ct - 1) / ct;
    const size_t lds = (size_t)a.KT * 5 * 1024 + (size_t)3 * waves * 128;
    const RowsNorm norm = {(const float*)gamma, (const float*)beta, eps, 1. / (double)M};
    const dim3 grid((unsigned)row_tiles(N)), block(waves * 64);
    if (ct == 1) hipLaunchKernelGGL(rows_norm_kernel<1>, grid, block, lds, (hipStream_t)stream, a, norm);
    else hipLaunchKernelGGL(rows_norm_kernel<2>, grid, block, lds, (hipStream_t)stream, a, norm);
    return check_launch(who);
}
