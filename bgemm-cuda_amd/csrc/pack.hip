// fp16 / fp32 -> bit-plane packing and logical <-> tiled re-layout.  HBM-bound byte work.
// Tiled output: a wave packs 8, 16 or 32 rows of one 32-row x 256-bit tile, with all of its 16-byte loads in
// flight at once; each lane turns eight elements into a byte of sign (and nonzero) bits, the
// bytes are put in tile order through LDS, and the tile leaves as one 16-byte store per lane.
// Logical output (the reference's row-major words): a wave packs 512 elements of one row.
#include "common.h"
#include "pack_bits.h"
#include <type_traits>
#include <string.h>

namespace bgemm {

// One operand to pack.  mode bit3: tiled output written by the row-segment waves (small operands:
// many short waves); bit5 / bit6: by waves of 8 / 16 rows of a tile instead of all 32.  mode bit0: also write the (sign & nonzero) plane and make plane 0 the
// nonzero plane; mode bit4: plane 0 = sign, plane 1 = nonzero.  mode bit1: write the logical layout instead of the tiled one.  mode bit2: the
// source is fp32 (rounded to fp16 first, as the layers' `.to(torch.half)` does).  mode bit7 (with bit 0): the two planes are written as
// codes (ternary_codes); always by waves of whole tile rows.
// zp: device scalar of the source type subtracted before that rounding, or null.
// A job may hold nmat = outer x inner matrices of `rows` rows each (tiled output only): matrix (o, i) starts
// so * o + si * i elements into src and fills its own mtiles row tiles of the output, one matrix after the other.
struct PackJob {
    const void* src; int64_t rows, K, ld;
    uint32_t* dst0; uint32_t* dst1; int mode;
    const void* zp;
    // training packs: the zero point as a mean of the operand itself (fp32, `nparts` partial sums, up to 128, and 1 / elements), a
    // scalar that the centred values are divided by, or null, and where those values are kept for the backward pass, [rows][K], or null
    const float* parts; int nparts; float inv_n;
    const float* divisor; void* kept;
    int kept_half;                 // kept as fp16
    NonzeroRule nonzero;
    int64_t rows_out, nseg, KT, Kw, waves;
    int64_t nmat, inner, so, si, mtiles;
};

// Element offset of output row `row` in the source, or -1 for a row of padding.
__device__ __forceinline__ int64_t source_row(const PackJob& j, const int64_t row)
{
    if (j.nmat == 1) return row < j.rows ? row * j.ld : -1;
    const int64_t mpad = j.mtiles * TILE_ROWS, b = row / mpad, rl = row - b * mpad;
    if (rl >= j.rows) return -1;
    const int64_t o = b / j.inner, i = b - o * j.inner;
    return o * j.so + i * j.si + rl * j.ld;
}

// Elements k0 .. k0 + 7 of a source row, centred, those from K on as +0.0.
__device__ __forceinline__ void load8_as_float(const void* row, const bool f32, const int64_t k0, const int64_t K, const float zf, float (&f)[8])
{
#pragma unroll
    for (int e = 0; e < 8; e++) {
        f[e] = 0.f;
        if (k0 + e < K) {
            const float v = f32 ? reinterpret_cast<const float*>(row)[k0 + e] : __half2float(reinterpret_cast<const __half*>(row)[k0 + e]);
            f[e] = __fsub_rn(v, zf);
        }
    }
}

// Eight values of a training pack, as they come and centred, into the ones whose signs are packed, and those kept (n of them, the first
// at element `at` of the operand): what the layer's backward pass reads is what there was at the time of the forward pass.  The divisor d
// comes loaded: behind the stores here the compiler would have to load it again for every eight values (fp32 [2048 + 1024, 1024]
// 11.1 -> 10.6 us).
__device__ __forceinline__ void train8(const PackJob& j, const float d, const int64_t at, const int n, float (&f)[8])
{
    if (j.divisor) {
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] = __fdiv_rn(f[e], d);
    }
    if (!j.kept || n <= 0) return;
    if (j.kept_half) {
        __half* const to = reinterpret_cast<__half*>(j.kept) + at;
        __half v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = __float2half_rn(f[e]);
        if (n == 8) __builtin_memcpy(to, v, sizeof v);
        else
#pragma unroll
            for (int e = 0; e < 7; e++)
                if (e < n) to[e] = v[e];
        return;
    }
    float* const to = reinterpret_cast<float*>(j.kept) + at;
    if (n == 8) __builtin_memcpy(to, f, sizeof f);
    else
#pragma unroll
        for (int e = 0; e < 7; e++)
            if (e < n) to[e] = f[e];
}

// A few values copied beside the packing (2-byte units): a scale as it is now, for the backward pass.
struct PackCopy { const uint16_t* src; uint16_t* dst; int64_t n; };
constexpr int COPY_PER_BLOCK = 2048;

// The scalar an operand is centred by, and whether it is; wave-uniform.
template <bool TRAIN>
__device__ __forceinline__ float job_center(const PackJob& j, const bool f32, const int lane)
{
    if (TRAIN && j.parts) {
        float s = lane < j.nparts ? j.parts[lane] : 0.f;
        if (lane + 64 < j.nparts) s += j.parts[lane + 64];
#pragma unroll
        for (int d = 32; d; d >>= 1) s += __shfl_xor(s, d);
        return s * j.inv_n;
    }
    return !j.zp ? 0.f : f32 ? *reinterpret_cast<const float*>(j.zp) : __half2float(*reinterpret_cast<const __half*>(j.zp));
}
template <bool TRAIN>
__device__ __forceinline__ float job_divisor(const PackJob& j) { return TRAIN && j.divisor ? *j.divisor : 1.f; }
__device__ __forceinline__ bool job_centred(const PackJob& j) { return j.zp != nullptr || (j.mode & 16); }

// Logical output: one wave packs 512 consecutive K elements of one row (16 words).
template <bool TRAIN>
__device__ __forceinline__ void pack_wave(const PackJob& j, const int64_t gw, const int lane)
{
    const int64_t row = gw / j.nseg, seg = gw - row * j.nseg;
    if (row >= j.rows_out) return;        // whole wave leaves together
    const int64_t k0 = seg * 512 + 8 * lane;

    uint32_t sg = 0, nz = 0;              // elements past K stay +0.0
    const int64_t soff = source_row(j, row);
    const float zf = job_center<TRAIN>(j, j.mode & 4, lane);
    [[maybe_unused]] const float d = job_divisor<TRAIN>(j);
    if (soff >= 0 && k0 < j.K) {
        const bool f32 = j.mode & 4, centred = job_centred(j);
        const char* const src = reinterpret_cast<const char*>(j.src) + soff * (f32 ? 4 : 2);
        if (j.K >= 8) {
            // the row's last chunk is read as its last eight elements, and the bits shifted into place
            const int64_t kc = k0 + 8 <= j.K ? k0 : j.K - 8;
            if constexpr (TRAIN) {
                float f[8];
                if (f32) centre8(load_raw8<true>(src, kc), zf, f);
                else centre8(load_raw8<false>(src, kc), zf, f);
                train8(j, d, row * j.K + kc, 8, f);
                bits8(f, j.nonzero, sg, nz);
            } else if (f32) bits8(load_raw8<true>(src, kc), centred, zf, j.nonzero, sg, nz);
            else bits8(load_raw8<false>(src, kc), centred, zf, j.nonzero, sg, nz);
            sg = (sg << (k0 - kc)) & 0xffu;
            nz = (nz << (k0 - kc)) & 0xffu;
        } else {
            float f[8];
            load8_as_float(src, f32, k0, j.K, zf, f);
            if constexpr (TRAIN) train8(j, d, row * j.K + k0, (int)(j.K - k0), f);
            bits8(f, j.nonzero, sg, nz);
            sg &= 0xff00u >> (j.K - k0); nz &= 0xff00u >> (j.K - k0);
        }
    }
    const bool ternary = j.mode & (1 | 16);
    uint32_t p0 = j.mode & 1 ? nz : sg, p1 = j.mode & 16 ? nz : sg & nz;
    const int sh = 8 * (3 - (lane & 3));
    p0 <<= sh; p1 <<= sh;
    p0 |= __shfl_xor(p0, 1); p0 |= __shfl_xor(p0, 2);
    if (ternary) { p1 |= __shfl_xor(p1, 1); p1 |= __shfl_xor(p1, 2); }
    if (lane & 3) return;
    const int64_t jw = seg * 16 + (lane >> 2);
    if (j.mode & 2) {
        if (row < j.rows && jw < j.Kw) { j.dst0[row * j.Kw + jw] = p0; if (ternary) j.dst1[row * j.Kw + jw] = p1; }
    } else if (jw < j.KT * 8) {
        const int64_t o = tiled_word_offset(row, jw, j.KT);
        j.dst0[o] = p0;
        if (ternary) j.dst1[o] = p1;
    }
}

// One wave packs RW of the 32 rows of tile (rt, kt) = gw / (32 / RW) of the tiled layout.  The lanes are spread over as many 8-element chunks as the tile's
// rows have (8, 16 or 32), so that a short row does not leave most of the wave idle: CW lanes per row, 64 / CW rows per step.
// lds: RW * 64 bytes of this wave's own, the two K-halves' 16-byte slots of its rows (twice for two planes).
// What bounds it is the read of the source: every load of the wave is in flight before the first is used.  Rows at any address and of any length take the same vector loads: rows and chunks past the end read the last ones
// again (the last chunk as the row's last eight elements, its bits then shifted into place), so nothing branches.  With
// element loads for such rows, as it was, fp16 [8195 + 2053, 4345] took 82.9 us; 19.3 us = 4.6 TB/s now (aligned rows: 5.1).
template <bool F32, int RW, bool TRAIN>
__device__ __forceinline__ void pack_tile(const PackJob& j, const int64_t gw, const int lane, unsigned char* lds)
{
    constexpr int PARTS = TILE_ROWS / RW, PLANE = RW * 32;
    const uint32_t tile = (uint32_t)gw / PARTS, kt32 = tile % (uint32_t)j.KT;
    const int64_t rt = tile / (uint32_t)j.KT, kt = kt32;
    const int row0 = (int)((uint32_t)gw % PARTS) * RW;               // the wave's first row in the tile
    if (rt * TILE_ROWS >= j.rows_out) return;              // whole wave leaves together
    // where the tile's first row lies in the source, and how many source rows there are from it on
    int64_t off0 = rt * TILE_ROWS * j.ld, rows_left = j.rows - rt * TILE_ROWS;
    if (j.nmat > 1) {
        const int64_t b = rt / j.mtiles, rtl = rt - b * j.mtiles, o = b / j.inner, i = b - o * j.inner;
        off0 = o * j.so + i * j.si + rtl * TILE_ROWS * j.ld;
        rows_left = j.rows - rtl * TILE_ROWS;
    }
    const bool ternary = j.mode & (1 | 16), centred = job_centred(j);      // two planes are written
    const bool nz_first = j.mode & 1, nz_second = j.mode & 16;
    const float zf = job_center<TRAIN>(j, F32, lane);
    [[maybe_unused]] const float d = job_divisor<TRAIN>(j);
    const int64_t left = j.K - kt * TILE_KBITS;
    typedef typename std::conditional<F32, uint32_t, uint16_t>::type E;
    const E* const src = reinterpret_cast<const E*>(j.src) + off0;
    const int last_row = (int)(rows_left < TILE_ROWS ? rows_left : TILE_ROWS) - 1;
    auto slot_byte = [](const int c, const int r) { return (c >> 4) * (RW * 16) + r * 16 + ((c >> 2) & 3) * 4 + (3 - (c & 3)); };
    if (j.K >= 8) {
        auto rows_by = [&](auto cw_tag) {
            constexpr int CW = decltype(cw_tag)::value, RI = 64 / CW, STEPS = RW / RI, G = STEPS < (F32 ? 8 : 16) ? STEPS : (F32 ? 8 : 16);
            const int c = lane & (CW - 1), rs = lane / CW;
            const int64_t k0 = kt * TILE_KBITS + 8 * c, kc = k0 + 8 <= j.K ? k0 : j.K - 8;
            const int shift = k0 - kc < 8 ? (int)(k0 - kc) : 8;
            if (CW < 32)                           // the bytes of the chunks this tile does not have
                for (int i = lane; i < (ternary ? PLANE / 2 : PLANE / 4); i += 64) reinterpret_cast<uint32_t*>(lds)[i] = 0u;
#pragma unroll
            for (int g = 0; g < STEPS; g += G) {
                Raw8<F32> raw[G];
#pragma unroll
                for (int jj = 0; jj < G; jj++) {
                    const int r = row0 + RI * (g + jj) + rs;
                    raw[jj] = load_raw8<F32>(src + (int64_t)(r < last_row ? r : last_row) * j.ld, kc);
                }
#pragma unroll
                for (int jj = 0; jj < G; jj++) {
                    const int r = RI * (g + jj) + rs, at = slot_byte(c, r);
                    uint32_t sg, nz;
                    if constexpr (TRAIN) {
                        float f[8];
                        centre8(raw[jj], zf, f);
                        train8(j, d, (rt * TILE_ROWS + row0 + r) * j.K + kc, row0 + r <= last_row && k0 < j.K ? 8 : 0, f);
                        bits8(f, j.nonzero, sg, nz);
                    } else
                        bits8(raw[jj], centred, zf, j.nonzero, sg, nz);
                    const uint32_t keep = row0 + r <= last_row ? 0xffu : 0u;
                    sg = (sg << shift) & keep; nz = (nz << shift) & keep;
                    lds[at] = (unsigned char)(nz_first ? nz : sg);
                    if (ternary) lds[PLANE + at] = (unsigned char)(nz_second ? nz : sg & nz);
                }
            }
        };
        if (left <= 64) rows_by(std::integral_constant<int, 8>{});
        else if (left <= 128) rows_by(std::integral_constant<int, 16>{});
        else rows_by(std::integral_constant<int, 32>{});
    } else {
        // rows of fewer than eight elements
        const int c = lane & 31;
        for (int jj = 0; jj < RW / 2; jj++) {
            const int rl = 2 * jj + (lane >> 5), r = row0 + rl, at = slot_byte(c, rl);
            float f[8];
            uint32_t sg, nz;
            const int n = r <= last_row && c == 0 ? (int)j.K : 0;
            load8_as_float(src + (int64_t)(r < last_row ? r : last_row) * j.ld, F32, 8 * c, n ? j.K : 0, zf, f);
            if constexpr (TRAIN) train8(j, d, (rt * TILE_ROWS + r) * j.K, n, f);
            bits8(f, j.nonzero, sg, nz);
            sg &= 0xff00u >> n; nz &= 0xff00u >> n;
            lds[at] = (unsigned char)(nz_first ? nz : sg);
            if (ternary) lds[PLANE + at] = (unsigned char)(nz_second ? nz : sg & nz);
        }
    }
    __builtin_amdgcn_wave_barrier();       // the slots were written by this wave alone: LDS keeps its order
    if (lane < 2 * RW) {
        const int64_t at = (int64_t)tile * TILE_U4 + (lane / RW) * 32 + row0 + lane % RW;
        if constexpr (!TRAIN) {
            if (j.mode & 128) {
                const uint4 z = reinterpret_cast<const uint4*>(lds)[lane], zs = reinterpret_cast<const uint4*>(lds + PLANE)[lane];
                uint4 a, b;
                ternary_codes(z.x, zs.x, a.x, b.x); ternary_codes(z.y, zs.y, a.y, b.y);
                ternary_codes(z.z, zs.z, a.z, b.z); ternary_codes(z.w, zs.w, a.w, b.w);
                reinterpret_cast<uint4*>(j.dst0)[at] = a;
                reinterpret_cast<uint4*>(j.dst1)[at] = b;
                return;
            }
        }
        reinterpret_cast<uint4*>(j.dst0)[at] = reinterpret_cast<const uint4*>(lds)[lane];
        if (ternary) reinterpret_cast<uint4*>(j.dst1)[at] = reinterpret_cast<const uint4*>(lds + PLANE)[lane];
    }
}

// Up to two operands per launch (the fp16 entry point packs weights and activations together).
template <bool TRAIN>
__device__ __forceinline__ void pack_jobs(const PackJob& j0, const PackJob& j1, const unsigned block, unsigned char (*s_tile)[2048])
{
    // the wave index as a scalar: the tile's coordinates and addresses stay on the scalar unit
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t gw = (int64_t)block * 4 + wave;
    const bool first = gw < j0.waves;
    const PackJob& j = first ? j0 : j1;
    if (!first) gw -= j0.waves;
    if (gw >= j.waves) return;
    if (j.mode & (2 | 8)) pack_wave<TRAIN>(j, gw, lane);
    else if (j.mode & 64) {
        if (j.mode & 4) pack_tile<true, 16, TRAIN>(j, gw, lane, s_tile[wave]);
        else pack_tile<false, 16, TRAIN>(j, gw, lane, s_tile[wave]);
    } else if (j.mode & 32) {
        if (j.mode & 4) pack_tile<true, 8, TRAIN>(j, gw, lane, s_tile[wave]);
        else pack_tile<false, 8, TRAIN>(j, gw, lane, s_tile[wave]);
    } else if (j.mode & 4) pack_tile<true, 32, TRAIN>(j, gw, lane, s_tile[wave]);
    else pack_tile<false, 32, TRAIN>(j, gw, lane, s_tile[wave]);
}

__global__ __launch_bounds__(256) void pack_f16_kernel(const PackJob j0, const PackJob j1)
{
    __shared__ __align__(16) unsigned char s_tile[4][2048];
    pack_jobs<false>(j0, j1, blockIdx.x, s_tile);
}

// The same for a layer's training pass, with a copy in the blocks before the packing's (last, they would end alone).  TRAIN: means,
// divisors and kept values.  A stretch of loads and its stores then wait for each other (one counter serves both; all stores
// behind all loads spill), so operands without any of them, the scaled layer's, are packed without: fp32 [8192 + 3072, 768]
// 17.3 -> 13.8 us, as without the copy.
template <bool TRAIN>
__global__ __launch_bounds__(256, 4) void pack_train_kernel(const PackJob j0, const PackJob j1, const PackCopy c, const int copy_blocks)
{
    __shared__ __align__(16) unsigned char s_tile[4][2048];
    if ((int)blockIdx.x < copy_blocks) {
        const int64_t i0 = (int64_t)blockIdx.x * COPY_PER_BLOCK + threadIdx.x;
#pragma unroll
        for (int i = 0; i < COPY_PER_BLOCK; i += 256)
            if (i0 + i < c.n) c.dst[i0 + i] = c.src[i0 + i];
        return;
    }
    pack_jobs<TRAIN>(j0, j1, blockIdx.x - copy_blocks, s_tile);
}

// dir 0: logical -> tiled (zero padding), dir 1: tiled -> logical.  One thread per tiled word.
__global__ __launch_bounds__(256) void relayout_kernel(
    const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, int64_t rows, int64_t Kw,
    int64_t KT, int64_t total, int dir)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    // decode tiled word index i -> (row, jw)
    const int64_t q = i & 3, slot = (i >> 2) & 63, tile = i >> 8;
    const int64_t kt = tile % KT, rt = tile / KT;
    const int64_t row = rt * 32 + (slot & 31), jw = kt * 8 + (slot >> 5) * 4 + q;
    const bool real = row < rows && jw < Kw;
    if (dir == 0) dst[i] = real ? src[row * Kw + jw] : 0u;
    else if (real) dst[row * Kw + jw] = src[i];
}

static int make_job(PackJob* j, const void* src, int64_t rows, int64_t K, int64_t ld, void* d0, void* d1, int mode,
                    const void* zp, const char* who, int64_t outer = 1, int64_t inner = 1, int64_t so = 0, int64_t si = 0)
{
    if (rows < 0 || K < 0 || ld < K) return fail(BGEMM_EINVAL, "%s: bad shape rows=%lld K=%lld ld=%lld", who,
                                                 (long long)rows, (long long)K, (long long)ld);
    if (outer < 0 || inner < 0 || so < 0 || si < 0 || ((mode & 2) && outer * inner != 1))
        return fail(BGEMM_EINVAL, "%s: bad batch %lld x %lld, strides %lld, %lld", who, (long long)outer,
                    (long long)inner, (long long)so, (long long)si);
    memset(j, 0, sizeof *j);
    if (rows == 0 || K == 0 || outer * inner == 0) return BGEMM_OK;
    if (!src || !d0 || ((mode & (1 | 16)) && !d1)) return fail(BGEMM_ENULL, "%s: null pointer", who);
    if (((uintptr_t)d0 & 15) || ((uintptr_t)d1 & 15)) return fail(BGEMM_EALIGN, "%s: destination not 16-byte aligned", who);
    j->nonzero = mode & 16 ? nonzero_sign_half() : nonzero_half();
    j->src = src; j->zp = zp; j->rows = rows; j->K = K; j->ld = ld;
    j->dst0 = (uint32_t*)d0; j->dst1 = (uint32_t*)d1; j->mode = mode;
    j->KT = k_tiles(K); j->Kw = cdiv(K, 32);
    j->nmat = outer * inner; j->inner = inner; j->so = so; j->si = si; j->mtiles = row_tiles(rows);
    j->rows_out = (mode & 2) ? rows : j->nmat * j->mtiles * TILE_ROWS;
    j->nseg = cdiv(j->KT * TILE_KBITS, 512);
    // Rows of a tile a wave takes.  A read of this kind wants many waves with a few loads each: four loads a lane (eight 16-byte
    // ones, fp32) are 8 rows of a whole tile, 16 or 32 where K is so short that half or a quarter of the lanes' chunks hold any;
    // on large fp16 operands 16 rows, where half as many waves to start weighs more (us, 32 / 16 / 8 rows a wave: fp32
    // 8192^2 54.4 / 49.1 / 46.3, 8192 x 768 8.3 / 7.7 / 7.2; fp16 8192^2 28.8 / 26.5 / 28.2, 11008 x 4096 23.3 / 18.7 / 21.8,
    // 8192 x 768 6.3 / 5.9 / 5.4, 98304 x 64 5.6 / 6.4 / 7.7, 8192 x 64 3.2 / 2.8 / 2.7).  Below 160 tiles single-row waves
    // (128 x 4096 fp16 4.7 / 3.7 / 3.2 / 2.8 with one row).
    const int64_t tiles = j->nmat * j->mtiles * j->KT;
    int rows_per_wave = 8;
    if (tiles >= 2048) rows_per_wave = K <= 64 ? 32 : K <= 128 || !(mode & 4) ? 16 : 8;
    if (!(mode & 2)) j->mode |= tiles < 160 && !(mode & 128) ? 8 : rows_per_wave == 8 ? 32 : rows_per_wave == 16 ? 64 : 0;
    j->waves = (j->mode & (2 | 8)) ? j->rows_out * j->nseg : tiles * (TILE_ROWS / rows_per_wave);
    return BGEMM_OK;
}

static int launch_jobs(const PackJob& j0, const PackJob& j1, hipStream_t st, const char* who, const PackCopy* train = nullptr)
{
    const int64_t blocks = cdiv(j0.waves + j1.waves, 4);
    if (blocks == 0) return BGEMM_OK;
    if (blocks > 0x3fffffffLL) return fail(BGEMM_EINVAL, "%s: operand too large", who);      // (wave numbers are 32 bits wide)
    if (!train) {
        hipLaunchKernelGGL(pack_f16_kernel, dim3((unsigned)blocks), dim3(256), 0, st, j0, j1);
        return check_launch(who);
    }
    auto of_its_own = [](const PackJob& j) { return j.parts || j.divisor || j.kept; };
    const int copy_blocks = (int)cdiv(train->n, COPY_PER_BLOCK);
    const dim3 grid((unsigned)(blocks + copy_blocks));
    if (of_its_own(j0) || of_its_own(j1)) hipLaunchKernelGGL(pack_train_kernel<true>, grid, dim3(256), 0, st, j0, j1, *train, copy_blocks);
    else hipLaunchKernelGGL(pack_train_kernel<false>, grid, dim3(256), 0, st, j0, j1, *train, copy_blocks);
    return check_launch(who);
}

static int pack_common(const void* src, int64_t rows, int64_t K, int64_t ld, void* d0, void* d1,
                       int mode, const void* zp, hipStream_t st, const char* who,
                       int64_t outer = 1, int64_t inner = 1, int64_t so = 0, int64_t si = 0)
{
    PackJob j0, j1;
    memset(&j1, 0, sizeof j1);
    const int rc = make_job(&j0, src, rows, K, ld, d0, d1, mode, zp, who, outer, inner, so, si);
    return rc ? rc : launch_jobs(j0, j1, st, who);
}

int pack_activations(const void* src, bool f32, bool ternary, bool codes, const void* zero_point, int64_t rows, int64_t K, int64_t ld, void* d0, void* d1,
                     hipStream_t st, const char* who)
{
    PackJob j0, j1;
    memset(&j1, 0, sizeof j1);
    const int rc = make_job(&j0, src, rows, K, ld, d0, d1, (ternary ? 1 : 0) | (codes ? 128 : 0) | (f32 ? 4 : 0), zero_point, who);
    return rc ? rc : launch_jobs(j0, j1, st, who);
}

// Sign-packs two fp16 operands into their tiled buffers with one launch.
int pack_sign_pair(const void* srcA, int64_t rowsA, void* dstA, const void* srcB, int64_t rowsB, void* dstB,
                   int64_t K, hipStream_t st, const char* who)
{
    PackJob j0, j1;
    int rc = make_job(&j0, srcA, rowsA, K, K, dstA, nullptr, 0, nullptr, who);
    if (!rc) rc = make_job(&j1, srcB, rowsB, K, K, dstB, nullptr, 0, nullptr, who);
    return rc ? rc : launch_jobs(j0, j1, st, who);
}

// Sign and nonzero planes of the learned-scale layer's operands, centred by their own means (see common.h).
int pack_elastic_pair(const float* x, int64_t N, void* x_sign, void* x_nonzero, float* xs, const float* w, int64_t M, void* w_sign, void* w_nonzero,
                      float* ws, int64_t K, const float* parts, int nparts, const float* sa, hipStream_t st, const char* who)
{
    PackJob j0, j1;
    int rc = make_job(&j0, x, N, K, K, x_sign, x_nonzero, 16 | 4, nullptr, who);
    if (!rc) rc = make_job(&j1, w, M, K, K, w_sign, w_nonzero, 16 | 4, nullptr, who);
    if (rc) return rc;
    j0.parts = parts; j0.inv_n = 1.f / (float)(N * K); j0.divisor = sa; j0.kept = xs;
    j1.parts = parts + nparts; j1.inv_n = 1.f / (float)(M * K); j1.kept = ws;
    j0.nparts = j1.nparts = nparts;
    j0.nonzero = j1.nonzero = nonzero_sign_float();
    const PackCopy none = {nullptr, nullptr, 0};
    return launch_jobs(j0, j1, st, who, &none);
}

// Sign and nonzero planes of the scaled layer's operands (see common.h).
int pack_linear_pair(const LinearPack& a, hipStream_t st, const char* who)
{
    PackJob j0, j1;
    const int mode = 16 | (a.src_dtype == BGEMM_SRC_F32 ? 4 : 0);
    int rc = make_job(&j0, a.x, a.N, a.K, a.ldx, a.x_sign, a.x_nonzero, mode, a.zero_point_x, who);
    if (!rc) rc = make_job(&j1, a.w, a.M, a.K, a.ldw, a.w_sign, a.w_nonzero, mode, a.zero_point_w, who);
    j0.kept = a.centred_x; j0.kept_half = 1;
    const PackCopy copy = {(const uint16_t*)a.sw, (uint16_t*)a.sw_then, a.sw_then ? a.M * (a.src_dtype == BGEMM_SRC_F32 ? 2 : 1) : 0};
    return rc ? rc : launch_jobs(j0, j1, st, who, &copy);
}

}  // namespace bgemm

using namespace bgemm;

extern "C" int64_t bgemm_tiled_words(int64_t rows, int64_t K)
{
    if (rows <= 0 || K <= 0) return 0;
    return row_tiles(rows) * k_tiles(K) * TILE_WORDS;
}

extern "C" int bgemm_pack_sign_f16(const void* src, int64_t rows, int64_t K, int64_t ld,
                                   void* dst_tiled, void* stream)
{
    return pack_common(src, rows, K, ld, dst_tiled, nullptr, 0, nullptr, (hipStream_t)stream, "bgemm_pack_sign_f16");
}

extern "C" int bgemm_pack_sign_f16_logical(const void* src, int64_t rows, int64_t K, int64_t ld,
                                           uint32_t* dst_logical, void* stream)
{
    return pack_common(src, rows, K, ld, dst_logical, nullptr, 2, nullptr, (hipStream_t)stream, "bgemm_pack_sign_f16_logical");
}

extern "C" int bgemm_pack_ternary_f16(const void* src, int64_t rows, int64_t K, int64_t ld,
                                      void* nz_tiled, void* sg_tiled, void* stream)
{
    return pack_common(src, rows, K, ld, nz_tiled, sg_tiled, 1, nullptr, (hipStream_t)stream, "bgemm_pack_ternary_f16");
}

extern "C" int bgemm_pack_sign_centered(const void* src, int src_dtype, int64_t rows, int64_t K, int64_t ld,
                                        const void* zero_point, void* dst_tiled, void* stream)
{
    if (src_dtype != BGEMM_SRC_F16 && src_dtype != BGEMM_SRC_F32)
        return fail(BGEMM_EINVAL, "bgemm_pack_sign_centered: unknown source type %d", src_dtype);
    return pack_common(src, rows, K, ld, dst_tiled, nullptr, src_dtype == BGEMM_SRC_F32 ? 4 : 0, zero_point,
                       (hipStream_t)stream, "bgemm_pack_sign_centered");
}

extern "C" int bgemm_pack_batched(const void* src, int src_dtype, int ternary, const void* zero_point,
                                  int64_t batch_outer, int64_t batch_inner, int64_t rows, int64_t K, int64_t ld,
                                  int64_t stride_outer, int64_t stride_inner, void* dst0_tiled, void* dst1_tiled,
                                  void* stream)
{
    if (src_dtype != BGEMM_SRC_F16 && src_dtype != BGEMM_SRC_F32)
        return fail(BGEMM_EINVAL, "bgemm_pack_batched: unknown source type %d", src_dtype);
    if (ternary && zero_point) return fail(BGEMM_EINVAL, "bgemm_pack_batched: a zero point goes with the sign pack only");
    return pack_common(src, rows, K, ld, dst0_tiled, ternary ? dst1_tiled : nullptr,
                       (ternary ? 1 : 0) | (src_dtype == BGEMM_SRC_F32 ? 4 : 0), zero_point, (hipStream_t)stream,
                       "bgemm_pack_batched", batch_outer, batch_inner, stride_outer, stride_inner);
}

extern "C" int bgemm_pack_sign_nonzero_pair(const void* src_a, int64_t rows_a, int64_t ld_a, const void* zero_point_a, void* sign_a,
                                            void* nonzero_a, const void* src_b, int64_t rows_b, int64_t ld_b, const void* zero_point_b,
                                            void* sign_b, void* nonzero_b, int src_dtype, int64_t K, void* stream)
{
    const char* who = "bgemm_pack_sign_nonzero_pair";
    if (src_dtype != BGEMM_SRC_F16 && src_dtype != BGEMM_SRC_F32) return fail(BGEMM_EINVAL, "%s: unknown source type %d", who, src_dtype);
    const int mode = 16 | (src_dtype == BGEMM_SRC_F32 ? 4 : 0);
    PackJob j0, j1;
    int rc = make_job(&j0, src_a, rows_a, K, ld_a, sign_a, nonzero_a, mode, zero_point_a, who);
    if (!rc) rc = make_job(&j1, src_b, rows_b, K, ld_b, sign_b, nonzero_b, mode, zero_point_b, who);
    return rc ? rc : launch_jobs(j0, j1, (hipStream_t)stream, who);
}

namespace bgemm {

// Transposed source ([K][rows] in memory): a wave builds one 32-row x 256-bit tile.  For each of its
// four words, lane (h, k') reads the 32 consecutive fp16 of source row k = 256 kt + 128 h + 32 q + k'
// (four 16-byte loads when the source allows, all sixteen in flight), gathers their sign bits into a
// word (bit r = row r), and the 32 x 32 bit matrix held by the 32 lanes of a wave half is transposed
// in registers with five masked exchanges: lane r then holds the word of row r, bit k' = column k'.
template <bool F32>
__global__ __launch_bounds__(256) void pack_transposed_kernel(const void* __restrict__ src_, const int64_t rows,
                                                              const int64_t K, const int64_t ld, const int64_t inner,
                                                              const int64_t so, const int64_t si,
                                                              uint4* __restrict__ dst, const int64_t tiles_per_matrix,
                                                              const int64_t KT, const int64_t total_tiles)
{
    typedef typename std::conditional<F32, uint32_t, uint16_t>::type E;
    constexpr int EB = sizeof(E), NV = 32 * EB / 16;       // 16-byte loads per 32 elements
    const int lane = threadIdx.x & 63, h = lane >> 5, kk = lane & 31;
    const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile >= total_tiles) return;             // whole wave leaves together
    const int64_t b = tile / tiles_per_matrix, t = tile - b * tiles_per_matrix, rt = t / KT, kt = t - rt * KT;
    const int64_t o = b / inner, i = b - o * inner;
    const int64_t r0 = rt * 32, k0 = kt * TILE_KBITS + h * 128 + kk;
    const E* p = reinterpret_cast<const E*>(src_) + o * so + i * si + k0 * ld + r0;
    const bool vec = r0 + 32 <= rows &&
                     (((uintptr_t)src_ | (uintptr_t)(ld * EB) | (uintptr_t)(so * EB) | (uintptr_t)(si * EB)) & 15) == 0;
    unsigned w[4];
    if (vec) {
        uint4 raw[4][NV];
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int c = 0; c < NV; c++)
                raw[q][c] = k0 + q * 32 < K ? reinterpret_cast<const uint4*>(p + (int64_t)q * 32 * ld)[c] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            unsigned x = 0;
#pragma unroll
            for (int c = 0; c < NV; c++) {
                const unsigned d[4] = {raw[q][c].x, raw[q][c].y, raw[q][c].z, raw[q][c].w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (F32)
                        x |= (d[e] >> 31) << (4 * c + e);
                    else {
                        const unsigned sb = d[e] & 0x80008000u;          // sign bits of two halves
                        x |= (((sb >> 15) | (sb >> 30)) & 3u) << (8 * c + 2 * e);
                    }
                }
            }
            w[q] = x;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            unsigned x = 0;
            if (k0 + q * 32 < K)
                for (int r = 0; r < 32; r++)
                    if (r0 + r < rows) x |= (unsigned)(p[(int64_t)q * 32 * ld + r] >> (8 * EB - 1)) << r;
            w[q] = x;
        }
    }
    // lane r of each half now takes row r; element k' of a word goes to bit 31 - k'
#pragma unroll
    for (int q = 0; q < 4; q++) w[q] = __brev(transpose32(w[q], lane));
    dst[tile * TILE_U4 + lane] = make_uint4(w[0], w[1], w[2], w[3]);
}

}  // namespace bgemm

extern "C" int bgemm_pack_transposed_batched(const void* src, int src_dtype, int64_t batch_outer, int64_t batch_inner,
                                             int64_t rows, int64_t K, int64_t ld, int64_t stride_outer,
                                             int64_t stride_inner, void* dst_tiled, void* stream)
{
    const char* who = "bgemm_pack_transposed_batched";
    if (src_dtype != BGEMM_SRC_F16 && src_dtype != BGEMM_SRC_F32) return fail(BGEMM_EINVAL, "%s: unknown source type %d", who, src_dtype);
    if (batch_outer < 0 || batch_inner < 0 || rows < 0 || K < 0 || ld < rows || stride_outer < 0 || stride_inner < 0)
        return fail(BGEMM_EINVAL, "%s: bad shape batch=%lld x %lld rows=%lld K=%lld ld=%lld", who, (long long)batch_outer,
                    (long long)batch_inner, (long long)rows, (long long)K, (long long)ld);
    const int64_t batch = batch_outer * batch_inner;
    if (batch == 0 || rows == 0 || K == 0) return BGEMM_OK;
    if (!src || !dst_tiled) return fail(BGEMM_ENULL, "%s: null pointer", who);
    const bool f32 = src_dtype == BGEMM_SRC_F32;
    if (((uintptr_t)src & (f32 ? 3 : 1)) || ((uintptr_t)dst_tiled & 15))
        return fail(BGEMM_EALIGN, "%s: source must be aligned to its elements, destination to 16 bytes", who);
    const int64_t KT = k_tiles(K), per = row_tiles(rows) * KT, total = batch * per, blocks = cdiv(total, 4);
    if (blocks > 0x7fffffffLL) return fail(BGEMM_EINVAL, "%s: operand too large", who);
    if (f32)
        hipLaunchKernelGGL(pack_transposed_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, src, rows,
                           K, ld, batch_inner, stride_outer, stride_inner, reinterpret_cast<uint4*>(dst_tiled), per, KT, total);
    else
        hipLaunchKernelGGL(pack_transposed_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, src, rows,
                           K, ld, batch_inner, stride_outer, stride_inner, reinterpret_cast<uint4*>(dst_tiled), per, KT, total);
    return check_launch(who);
}

extern "C" int bgemm_pack_sign_f16_transposed(const void* src, int64_t batch, int64_t rows, int64_t K, int64_t ld,
                                              int64_t src_batch_stride, void* dst_tiled, void* stream)
{
    return bgemm_pack_transposed_batched(src, BGEMM_SRC_F16, 1, batch, rows, K, ld, 0, src_batch_stride, dst_tiled, stream);
}

static int relayout(const void* src, void* dst, int64_t rows, int64_t K, int dir, void* stream, const char* who)
{
    if (rows < 0 || K < 0) return fail(BGEMM_EINVAL, "%s: bad shape", who);
    if (rows == 0 || K == 0) return BGEMM_OK;
    if (!src || !dst) return fail(BGEMM_ENULL, "%s: null pointer", who);
    const int64_t total = bgemm_tiled_words(rows, K), blocks = cdiv(total, 256);
    if (blocks > 0x7fffffffLL) return fail(BGEMM_EINVAL, "%s: operand too large", who);
    hipLaunchKernelGGL(relayout_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const uint32_t*)src, (uint32_t*)dst, rows, cdiv(K, 32), k_tiles(K), total, dir);
    return check_launch(who);
}

// Row popcounts of a tiled operand: one block of sixteen waves per 32-row tile row, wave w takes K-tiles w, w + 16, ...
// (two 16-byte loads in flight a lane: a launch of this size is one memory round trip), lanes 0-31 and 32-63 of a
// wave hold the two K-halves of a row; the partial counts of a row meet in LDS.
__global__ __launch_bounds__(1024) void row_popcount_kernel(const uint4* __restrict__ tiled, int32_t* __restrict__ counts,
                                                            const int64_t rows, const int64_t KT, const int64_t stride_u4)
{
    __shared__ int part[1024];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t rt = blockIdx.x, b = blockIdx.y;
    const uint4* base = tiled + b * stride_u4 + rt * KT * TILE_U4 + lane;
    int n = 0;
    int64_t kt = wave;
    for (; kt + 16 < KT; kt += 32) {
        const uint4 v0 = base[kt * TILE_U4], v1 = base[(kt + 16) * TILE_U4];
        n += __popc(v0.x) + __popc(v0.y) + __popc(v0.z) + __popc(v0.w) + __popc(v1.x) + __popc(v1.y) + __popc(v1.z) + __popc(v1.w);
    }
    if (kt < KT) {
        const uint4 v = base[kt * TILE_U4];
        n += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
    }
    part[threadIdx.x] = n;
    __syncthreads();
    if (threadIdx.x < 32) {
        int t = 0;
#pragma unroll
        for (int w = 0; w < 32; w++) t += part[w * 32 + threadIdx.x];     // 16 waves x 2 K-halves
        const int64_t row = rt * 32 + threadIdx.x;
        if (row < rows) counts[b * rows + row] = t;
    }
}

extern "C" int bgemm_row_popcounts(const void* tiled, int64_t batch, int64_t rows, int64_t K, int64_t stride_words,
                                   void* counts, void* stream)
{
    if (batch < 0 || rows < 0 || K < 0 || K >= (1LL << 24) || stride_words < 0 || (stride_words & 3))
        return fail(BGEMM_EINVAL, "bgemm_row_popcounts: bad shape batch=%lld rows=%lld K=%lld stride=%lld", (long long)batch,
                    (long long)rows, (long long)K, (long long)stride_words);
    if (batch == 0 || rows == 0) return BGEMM_OK;
    if (!counts || (K > 0 && !tiled)) return fail(BGEMM_ENULL, "bgemm_row_popcounts: null pointer");
    if (((uintptr_t)tiled & 15) || ((uintptr_t)counts & 3)) return fail(BGEMM_EALIGN, "bgemm_row_popcounts: operand not aligned");
    if (batch > 65535 || row_tiles(rows) > 0x7fffffffLL) return fail(BGEMM_EINVAL, "bgemm_row_popcounts: operand too large");
    if (batch > 1 && stride_words < bgemm_tiled_words(rows, K))
        return fail(BGEMM_EINVAL, "bgemm_row_popcounts: stride %lld smaller than one operand", (long long)stride_words);
    hipLaunchKernelGGL(row_popcount_kernel, dim3((unsigned)row_tiles(rows), (unsigned)batch), dim3(1024), 0, (hipStream_t)stream,
                       (const uint4*)tiled, (int32_t*)counts, rows, k_tiles(K), stride_words / 4);
    return check_launch("bgemm_row_popcounts");
}

extern "C" int bgemm_tile_from_logical(const uint32_t* logical, int64_t rows, int64_t K,
                                       void* dst_tiled, void* stream)
{
    return relayout(logical, dst_tiled, rows, K, 0, stream, "bgemm_tile_from_logical");
}

extern "C" int bgemm_logical_from_tiled(const void* tiled, int64_t rows, int64_t K,
                                        uint32_t* dst_logical, void* stream)
{
    return relayout(tiled, dst_logical, rows, K, 1, stream, "bgemm_logical_from_tiled");
}
