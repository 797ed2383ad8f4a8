// BF16 / FP16 256x256 tile kernel: 8 waves in two groups that take turns at the matrix cores and at
// memory ("ping-pong"), operands staged into LDS by DMA (global_load_lds_dwordx4).  Device code only;
// kernels_half_dma_{bf16,fp16}.hip instantiate it, plain and grouped.
//
// d = alpha * (a @ b) + beta * c, the contract of the other 16-bit tiles (fp32 accumulation; c and d
// in fp32 or the input type; with a null c the beta term is dropped).  Applicability, checked on the
// host, is that of the DMA tiles of dma_tile.hpp (16-byte aligned a and b, leading dimensions
// multiples of 8 and below 2^23, those of c and d below 2^21, a's and b's contiguous extents multiples
// of 8); m, n and k are free otherwise.
//
// Workgroup: 8 waves, two per SIMD.  Wave w is in group wm = w / 4 and has column place wn = w % 4.
// The tile's rows come in two halves of 128, its columns too; a wave owns, of each of the four
// quarters (row half i, column half j), rows 64 wm .. + 63 and columns 32 wn .. + 31: 4 x 2 blocks
// of v_mfma_f32_16x16x32.  The MFMA takes b's fragment first and a's second, so it computes the
// transposed block and a lane ends up with 4 adjacent columns of one row:
//   a fragment: lane l holds A[row l % 16][k 8 (l / 16) .. + 7], b's the same of its column;
//   result    : lane l, register r holds D[row l % 16][column 4 (l / 16) + r].
//
// Stage = 64 k, as four half tiles of 16 KiB (A0, A1, B0, B1), two stages (128 KiB).  A stage is two
// phases, each a memory part (LDS reads into registers, 4 DMAs per wave) and a matrix part (32 MFMAs,
// one row half of the tile):
//   phase 0: read A0, B1      DMA A1 (stage + 1), B0 (stage + 2)    A0 x (B0, B1)
//   phase 1: read A1, B0(+1)  DMA A0, B1 (stage + 2)                A1 x (B0, B1)
// A barrier ends every part, and group 1 starts one barrier late, so on every SIMD one wave runs its
// matrix part while the other runs its memory part: the LDS latency, the waits and the address work
// of one group lie under the other's MFMAs.
//   A half tile is overwritten by DMAs issued one phase after both groups have read it: each wave
// waits for its reads before the barrier that ends its memory part.
//   A half tile is read 3 phases (3072 MFMA cycles) after its DMAs were issued; the wait (vmcnt) that
// ends a memory part leaves the DMAs of the last two phases in flight.
// A tile with at most 128 rows inside the matrix (the last one of a group, of any ragged m) is short:
// it needs no A1, so its stage is one phase (read A0, B0, B1; DMA A0, B0, B1 of stage + 2; 32 MFMAs)
// and three stages of 48 KiB fit.  Grouped 16384x14336x4096 over 64 experts of 102 to 410 rows, 2396 ->
// 2216 us (16-bit d, column-major weights 2329 -> 2117); over 8 experts 1503 -> 1473.
// The DMA is issued from inline assembly with M0 set in the same statement; every wait on it is an
// explicit vmcnt in this file, and the compiler has no other use of M0 here.
//
// What bounds it, and why this shape.  MFMA issue under the clock that the chip's power limit leaves:
// 4 waves of 128x128 (one per SIMD, 32x32x16 MFMAs, DMAs one stage ahead) interleaved their LDS
// reads, waits and DMA issue with their own MFMAs and lost 16-20% of the issue slots; two waves per
// SIMD that alternate lose almost none, 16x16x32 MFMAs draw less power per FLOP, and the longer DMA
// lead covers HBM, so a b larger than the last-level cache needs no prefetch.  Measured on MI355X
// against that tile, same box, bf16, us: 16384x14336x4096 with column-major b and 16-bit d 1577 ->
// 1256, 4096x4096x8200 with column-major a and fp32 c 219 -> 199, 2048x114688x4096 1526 -> 1411, grouped
// 16384x14336x4096 over 8 / 64 experts 1680 -> 1503 / 2599 -> 2396.  Phases of 16 MFMAs instead of 32
// (barriers twice as often, LDS reads and waits no longer covered) ran 10% slower (8192^3 826 against
// 757); raising the wave priority in the matrix part was 0.5% slower, DMAs before the reads the same.
// Bands (tile_of) of 4 rows: 8192^3 738 us against 743 (6), 778 (8), 835 (16).  Stores of fp32 d
// through L2 as usual 712-725 against 720-727 non-temporal; 16-bit d 16384x14336x4096 1255 against
// 1242 non-temporal.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "ft/gemm_kernels.hpp"

namespace ftrain::gemm::ppdev {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
using u16 = unsigned short;

constexpr int kStageK = 64;
constexpr unsigned kHalfTile = 16384;      // bytes of one half tile (128 rows or columns x 64 k)
constexpr unsigned kStage    = 4 * kHalfTile;
// A short tile's stage (A0, B0, B1); three of them are the larger of the two layouts (144 KiB).
constexpr unsigned kShortStage = 3 * kHalfTile;
static_assert(3 * kShortStage >= 2 * kStage, "LDS");
constexpr unsigned kA0 = 0, kA1 = kHalfTile, kB0 = 2 * kHalfTile, kB1 = 3 * kHalfTile;
// Word 3 of a raw buffer resource on gfx9 parts: 32-bit data format, range check on every access.
constexpr int kBufferConfig = 0x00020000;

template <bool BF16>
__device__ __forceinline__ floatx4 mfma(u32x4 b, u32x4 a, floatx4 acc) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b), __builtin_bit_cast(bf16x8, a),
                                                       acc, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, b), __builtin_bit_cast(halfx8, a),
                                                      acc, 0, 0, 0);
}

template <bool BF16>
__device__ __forceinline__ float to_float(u16 v) {
    if constexpr (BF16)
        return __builtin_bit_cast(float, static_cast<unsigned int>(v) << 16);
    else
        return static_cast<float>(__builtin_bit_cast(_Float16, v));
}

template <bool BF16>
__device__ __forceinline__ u16 from_float(float v) {
    if constexpr (BF16)
        return __builtin_bit_cast(u16, static_cast<__bf16>(v));
    else
        return __builtin_bit_cast(u16, static_cast<_Float16>(v));
}

template <bool BF16>
__device__ __forceinline__ unsigned pack2(float lo, float hi) {
    return static_cast<unsigned>(from_float<BF16>(lo)) | (static_cast<unsigned>(from_float<BF16>(hi)) << 16);
}

// 1 KiB DMA: lane l copies 16 bytes from sbase + voff(l) to LDS byte address lds + 16 l.
__device__ __forceinline__ void dma_1k(unsigned voff, const void* sbase, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(sbase)
                 : "memory", "m0");
}

// Output tile of workgroup `bid`: the 8 XCDs take contiguous runs of tile ids, walked in bands of
// `rows_per_band` tile rows.
__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn, int rows_per_band) {
    const int tiles = tiles_m * tiles_n;
    const int per   = tiles >> 3;
    int t           = bid;
    if (bid < (per << 3)) t = (bid & 7) * per + (bid >> 3);
    const int band_span = rows_per_band * tiles_n;
    const int band      = t / band_span;
    const int first_m   = band * rows_per_band;
    const int band_rows = min(tiles_m - first_m, rows_per_band);
    const int within    = t - band * band_span;
    tm                  = first_m + within % band_rows;
    tn                  = within / band_rows;
}

// One operand's staging.  A half tile takes 16 DMAs, two per wave (blocks wave and wave + 8).
//   k-contiguous operand (row-major a, column-major b): LDS [128 rows][64 k], a DMA covers 8 rows
//     (whole 128-byte lines); 16-byte chunk c of row r sits at slot c ^ ((r >> 1) & 7);
//   transposed operand (TR): LDS [64 k][128], a DMA covers 4 k rows of 256 bytes; chunk c of k row kr
//     sits at slot c ^ (2 ((kr & 3) + 4 ((kr >> 3) & 1))).
// Both keep the reads free of bank conflicts: the 16 lanes of a ds_read_b128 pass (16 rows, one
// chunk) cover 256 bytes of banks, and so do the 8 k rows x 32 bytes of a transposing read.
// Rows (columns) past the matrix are clamped onto its last row (last whole chunk: the extent of a
// transposed operand is a multiple of 8); they feed only outputs that are not stored.
template <bool TR>
struct Operand {
    const char* base;   // tile origin
    int64_t step;       // bytes from one stage to the next
    int64_t half_block; // TR: bytes from a wave's first block of a half tile to its second (32 k rows)
    unsigned voff[2][2];

    __device__ __forceinline__ void init(const u16* m, int64_t ld, int origin, int extent, int wave, int lane) {
        if constexpr (TR) {
            const int kr = 4 * wave + (lane >> 4);
            const int chunk = (lane & 15) ^ (2 * ((kr & 3) + 4 * ((kr >> 3) & 1)));
            base       = reinterpret_cast<const char*>(m + origin);
            step       = kStageK * ld * 2;
            half_block = 32 * ld * 2;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int col = min(origin + 128 * i + 8 * chunk, extent - 8) - origin;
                voff[i][0] = voff[i][1] = static_cast<unsigned>((kr * ld + col) * 2);
            }
        } else {
            const unsigned last = static_cast<unsigned>(min(extent - 1 - origin, 255));
            const unsigned ld2  = static_cast<unsigned>(2 * ld);
            base       = reinterpret_cast<const char*>(m + (size_t)origin * ld);
            step       = kStageK * 2;
            half_block = 0;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const unsigned r = 8 * (wave + 8 * j) + (lane >> 3);
                    voff[i][j] = min(128u * i + r, last) * ld2 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
                }
        }
    }
    // This wave's two DMAs of half tile i of the stage at `src` (base + stage * step).
    __device__ __forceinline__ void dma(const char* src, int i, unsigned lds, int wave) const {
        dma_1k(voff[i][0], src, lds + wave * 1024);
        dma_1k(voff[i][1], src + half_block, lds + (wave + 8) * 1024);
    }
    // What those DMAs would write, by ordinary loads, with zeros for k (within the stage) of k_left
    // or more: the partial last stage of a k tail.  Such lanes load nothing.
    __device__ __forceinline__ void fill(const char* src, int i, char* lds, int wave, int lane, int k_left) const {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r   = 8 * (wave + 8 * j) + (lane >> 3);
            const bool ok = TR ? 4 * (wave + 8 * j) + (lane >> 4) < k_left : 8 * ((lane & 7) ^ ((r >> 1) & 7)) < k_left;
            u32x4 v       = u32x4{0u, 0u, 0u, 0u};
            if (ok) v = *reinterpret_cast<const u32x4*>(src + (j ? half_block : 0) + voff[i][j]);
            *reinterpret_cast<u32x4*>(lds + (wave + 8 * j) * 1024 + 16 * lane) = v;
        }
    }
};

// What the pipeline reads when k holds no whole stage (its data is discarded): operands initialised
// on it with a leading dimension of 0 keep every lane's offset within 512 bytes.
static __device__ __attribute__((aligned(256))) u16 pp_dummy[512];

template <bool BF16, bool TA, bool TB>
__device__ __forceinline__ void half_gemm_pp_tile(const HalfGemmParams& p, int bid, int band) {
    constexpr bool A_TR = TA, B_TR = !TB;
    __shared__ __attribute__((aligned(1024))) char lds[3 * kShortStage];
    const int tid = threadIdx.x, lane = tid & 63, j16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    int tm, tn;
    tile_of(bid, p.tiles_m, p.tiles_n, tm, tn, band);
    const int m0 = tm * 256, n0 = tn * 256;
    const int M = p.m, N = p.n;
    const int nst = p.k / kStageK, k_tail = p.k - nst * kStageK;

    const u16* const pa = static_cast<const u16*>(p.a);
    const u16* const pb = static_cast<const u16*>(p.b);
    Operand<A_TR> opa;
    Operand<B_TR> opb;
    if (nst > 0) {
        opa.init(pa, p.lda, m0, M, wave, lane);
        opb.init(pb, p.ldb, n0, N, wave, lane);
    } else {
        opa.init(pp_dummy, 0, 0, 256, wave, lane);
        opb.init(pp_dummy, 0, 0, 256, wave, lane);
    }
    const int last_st   = nst > 0 ? nst - 1 : 0;
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds;

    // LDS read addresses: this lane's part of each operand's fragments, for either stage buffer (the
    // half tile, block row and k-step are added as constants).
    // k-contiguous: row x + 16 u + j16, chunk 4 ks + g; x is a multiple of 16, so the swizzle is that
    // of j16, and ks flips bit 2 of the slot (64 bytes).
    // Transposed: k row 32 ks + 8 g + 4 part + tr_k (tr_k = j16 / 4), elements 16 x16 + 4 (lane % 4) ..
    // + 3; the swizzle of those k rows is 2 (tr_k + 4 (g & 1)) chunks, so 16-element run x16 sits at
    // run x16 ^ (tr_k + 4 (g & 1)).
    const unsigned tr_swz = (j16 >> 2) + 4 * (g & 1);
    const unsigned tr_row = (8 * g + (j16 >> 2)) * 256 + 8 * (lane & 3);
    auto kc_lane = [&](int x, int ks) { return lds0 + (x + j16) * 128 + 16 * ((4 * ks + g) ^ (j16 >> 1)); };
    auto tr_lane = [&](int x16) { return lds0 + tr_row + (x16 ^ tr_swz) * 32; };
    unsigned ra[2][4], rb[2][2];  // [stage buffer][k-step, or 16-element run of a transposed operand]
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int u = 0; u < 4; ++u) ra[q][u] = q * kStage + (A_TR ? tr_lane(4 * wm + u) : kc_lane(64 * wm, u & 1));
#pragma unroll
        for (int v = 0; v < 2; ++v) rb[q][v] = q * kStage + (B_TR ? tr_lane(2 * wn + v) : kc_lane(32 * wn, v));
    }
    auto read_kc = [&](unsigned at) { return *(lds_u32x4*)(uintptr_t)at; };
    auto read_tr = [&](unsigned at) {
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(uintptr_t)at);
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(uintptr_t)(at + 4 * 256));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        return u32x4{l2[0], l2[1], h2[0], h2[1]};
    };

    floatx4 acc[2][2][4][2];  // row half, column half, block row, block column
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 2; ++v) acc[i][j][u][v] = floatx4{0.f, 0.f, 0.f, 0.f};
    u32x4 fa[4][2], f0[2][2], f1[2][2], g0[2][2];  // a: block row, k-step; b: block column, k-step

    // a's (b's) fragments of half tile `half` (kA0 ..) of stage buffer q.
    auto read_a = [&](int q, unsigned half) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                fa[u][ks] = A_TR ? read_tr(ra[q][u] + half + 32 * 256 * ks) : read_kc(ra[q][ks] + half + 2048 * u);
    };
    auto read_b = [&](int q, unsigned half, u32x4 (&f)[2][2]) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int v = 0; v < 2; ++v)
                f[v][ks] = B_TR ? read_tr(rb[q][v] + half + 32 * 256 * ks) : read_kc(rb[q][ks] + half + 2048 * v);
    };
    auto matrix = [&](floatx4 (&c)[4][2], u32x4 (&f)[2][2]) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 2; ++v) c[u][v] = mfma<BF16>(f[v][ks], fa[u][ks], c[u][v]);
    };
    // End of a memory part: this wave's LDS reads are done, its DMAs of 2 phases ago have landed.
#define FT_PP_MEM_END                                                                \
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");         \
    __builtin_amdgcn_sched_barrier(0);
#define FT_PP_MATRIX(I, F0)                      \
    matrix(acc[I][0], F0);                       \
    matrix(acc[I][1], f1);                       \
    __builtin_amdgcn_sched_barrier(0);           \
    asm volatile("s_barrier" ::: "memory");      \
    __builtin_amdgcn_sched_barrier(0);
    // Stage st in buffer Q: fragments of B0 in F0, those of the next stage's B0 into FN.  sa, sb point
    // at stage st + 1 (clamped to the last: nothing reads what is reloaded past it).
#define FT_PP_STAGE(Q, F0, FN, ST)                                  \
    read_a(Q, kA0);                                                 \
    read_b(Q, kB1, f1);                                             \
    opa.dma(sa, 1, lds0 + (1 - (Q)) * kStage + kA1, wave);          \
    if ((ST) + 2 <= last_st) {                                      \
        sa += opa.step;                                             \
        sb += opb.step;                                             \
    }                                                               \
    opb.dma(sb, 0, lds0 + (Q) * kStage + kB0, wave);                \
    FT_PP_MEM_END                                                   \
    FT_PP_MATRIX(0, F0)                                             \
    read_a(Q, kA1);                                                 \
    read_b(1 - (Q), kB0, FN);                                       \
    opa.dma(sa, 0, lds0 + (Q) * kStage + kA0, wave);                \
    opb.dma(sb, 1, lds0 + (Q) * kStage + kB1, wave);                \
    FT_PP_MEM_END                                                   \
    FT_PP_MATRIX(1, F0)

    const char *sa = opa.base, *sb = opb.base;
    if (M - m0 <= 128) {
        // Short tile.  Stages 0 and 1 in flight; stage st + 2 takes the slot that both groups finished
        // reading one phase ago.
        auto dma_stage = [&](unsigned at) {
            opa.dma(sa, 0, at, wave);
            opb.dma(sb, 0, at + kHalfTile, wave);
            opb.dma(sb, 1, at + 2 * kHalfTile, wave);
        };
        dma_stage(lds0);
        if (last_st >= 1) {
            sa += opa.step;
            sb += opb.step;
        }
        dma_stage(lds0 + kShortStage);
        asm volatile("s_waitcnt vmcnt(6)\n\ts_barrier" ::: "memory");
        if (wm == 1) asm volatile("s_barrier" ::: "memory");
        unsigned slot = 0, free = 2 * kShortStage;
        for (int st = 0; st < nst; ++st) {
            // read_a and read_b add kA0 = 0, or a half tile's offset, to the addresses of buffer 0.
            const unsigned keep_a[4] = {ra[0][0], ra[0][1], ra[0][2], ra[0][3]}, keep_b[2] = {rb[0][0], rb[0][1]};
#pragma unroll
            for (int u = 0; u < 4; ++u) ra[0][u] += slot;
#pragma unroll
            for (int v = 0; v < 2; ++v) rb[0][v] += slot;
            read_b(0, kHalfTile, f0);
            read_a(0, 0);
            read_b(0, 2 * kHalfTile, f1);
#pragma unroll
            for (int u = 0; u < 4; ++u) ra[0][u] = keep_a[u];
#pragma unroll
            for (int v = 0; v < 2; ++v) rb[0][v] = keep_b[v];
            if (st + 2 <= last_st) {
                sa += opa.step;
                sb += opb.step;
            }
            dma_stage(lds0 + free);
            asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            FT_PP_MATRIX(0, f0)
            free = slot;
            slot = slot == 2 * kShortStage ? 0 : slot + kShortStage;
        }
        if (wm == 0) asm volatile("s_barrier" ::: "memory");
    } else {
        // Stage 0 and, but for its A1, stage 1 in flight, in the order the phases read them; then B0 of
        // stage 0.
        opb.dma(sb, 0, lds0 + kB0, wave);
        opa.dma(sa, 0, lds0 + kA0, wave);
        opb.dma(sb, 1, lds0 + kB1, wave);
        opa.dma(sa, 1, lds0 + kA1, wave);
        if (last_st >= 1) {
            sa += opa.step;
            sb += opb.step;
        }
        opb.dma(sb, 0, lds0 + kStage + kB0, wave);
        opa.dma(sa, 0, lds0 + kStage + kA0, wave);
        opb.dma(sb, 1, lds0 + kStage + kB1, wave);
        // B0, A0 and B1 of stage 0 have landed.
        asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
        read_b(0, kB0, f0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (wm == 1) asm volatile("s_barrier" ::: "memory");

        int st = 0;
        for (; st + 1 < nst; st += 2) {
            FT_PP_STAGE(0, f0, g0, st)
            FT_PP_STAGE(1, g0, f0, st + 1)
        }
        if (st < nst) {
            FT_PP_STAGE(0, f0, g0, st)
        }
        if (wm == 0) asm volatile("s_barrier" ::: "memory");
    }
#undef FT_PP_STAGE
#undef FT_PP_MEM_END
#undef FT_PP_MATRIX
    // The workgroup's LDS must not be released, nor refilled, with a DMA still writing it.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // k tail: the partial last stage is staged by ordinary loads (zeros past k), then multiplied.
    if (k_tail > 0) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        opa.init(pa, p.lda, m0, M, wave, lane);
        opb.init(pb, p.ldb, n0, N, wave, lane);
        const char* const ta = opa.base + (size_t)nst * opa.step;
        const char* const tb = opb.base + (size_t)nst * opb.step;
        opa.fill(ta, 0, lds + kA0, wave, lane, k_tail);
        opa.fill(ta, 1, lds + kA1, wave, lane, k_tail);
        opb.fill(tb, 0, lds + kB0, wave, lane, k_tail);
        opb.fill(tb, 1, lds + kB1, wave, lane, k_tail);
        __syncthreads();
        read_b(0, kB0, f0);
        read_b(0, kB1, f1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            read_a(0, i ? kA1 : kA0);
            matrix(acc[i][0], f0);
            matrix(acc[i][1], f1);
        }
    }

    // Epilogue.  Lane (j16, g) holds row j16, columns 4 g .. 4 g + 3 of every 16x16 block; stored from
    // there, every access would touch 16 rows.  One row half of the tile at a time is therefore turned
    // over through LDS (128 rows of 1 KiB, 16-byte chunk c of row r at slot c ^ (r & 15): neither side
    // has bank conflicts), after which a wave owns 16 whole rows: an access covers one row of 1 KiB in
    // fp32, two of 512 bytes in 16 bits.  c is loaded in that layout, a row half ahead of its use.
    //   Buffer accesses relative to the tile's corner: the lane part of the offset in the VGPR offset, the
    // row in the scalar offset.  An element outside the matrix gets the lane offset 2^31, past the
    // buffer's size (at most 2^31 - 1 bytes), so its c load returns 0 and its store is dropped; ldc and
    // ldd below 2^21 keep every sum below 2^32.  A buffer access of 16 bytes needs an address aligned to 4:
    // 16-bit c and d whose rows are not (!WIDE) take global accesses, which need no alignment.  The chunk
    // across the last column, if there is one, goes element by element.
    //   Measured against stores from the MFMA layout (16 rows of 64 bytes per access; element by element
    // where n, ldc or ldd were not multiples of 16 bytes), fp16, us: 9216x2827x2112 with a column-major b
    // and 16-bit d 275 -> 115; bf16 with c, 8192x8192x256 114 -> 92, 3584x6272x512 (fp32 c) 69 -> 60.
    const float alpha = p.alpha, beta = p.beta;
    const unsigned ldd = static_cast<unsigned>(p.ldd), ldc = static_cast<unsigned>(p.ldc);
    const int rows_left = M - m0, cols_left = N - n0;
    constexpr unsigned kOut = 0x80000000u;
    auto epilogue = [&](auto c_tag, auto half_tag, auto wide_tag) {
        constexpr bool HAS_C = decltype(c_tag)::value, HALF = decltype(half_tag)::value, WIDE = decltype(wide_tag)::value;
        constexpr unsigned ES = HALF ? 2 : 4;
        constexpr int EPL = HALF ? 8 : 4, RPA = HALF ? 2 : 1;  // elements per lane, rows per access
        constexpr int NA = 16 / RPA;                           // accesses of a wave per row half
        // 16-bit d is stored non-temporal (2), fp32 d is not (0): measured, above.
        constexpr int kPolicy = HALF ? 2 : 0;
        typedef u32x4 u32x4_any __attribute__((aligned(2)));
        const int er = HALF ? lane >> 5 : 0, ec = EPL * (HALF ? lane & 31 : lane);
        const bool full = ec + EPL <= cols_left, cut = ec < cols_left && !full;
        const bool any_cut = cols_left < 256 && cols_left % EPL != 0;
        auto span = [&](uint64_t ld) {
            const uint64_t b = ((uint64_t)(rows_left - 1) * ld + (uint64_t)cols_left) * ES;
            return static_cast<int>(b < 0x7FFFFFFFull ? b : 0x7FFFFFFFull);
        };
        char* const dcorner = static_cast<char*>(p.d) + ((size_t)m0 * p.ldd + n0) * ES;
        const __amdgpu_buffer_rsrc_t dres = __builtin_amdgcn_make_buffer_rsrc(dcorner, 0, span(p.ldd), kBufferConfig);
        const char* ccorner         = nullptr;
        __amdgpu_buffer_rsrc_t cres = dres;
        if constexpr (HAS_C) {
            ccorner = static_cast<const char*>(p.c) + ((size_t)m0 * p.ldc + n0) * ES;
            cres    = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(ccorner), 0, span(p.ldc), kBufferConfig);
        }
        const unsigned lane_d = (er * ldd + ec) * ES, lane_c = (er * ldc + ec) * ES;
        auto row_of = [&](int i, int t) { return 128 * i + 16 * wave + RPA * t; };  // wave-uniform
        u32x4 cv[HAS_C ? NA : 1];
        auto load_c = [&](int i, int t) {
            if constexpr (HAS_C) {
                const int row0 = row_of(i, t);
                const bool ok  = full && row0 + er < rows_left;
                if constexpr (HALF && !WIDE) {
                    cv[t] = u32x4{0u, 0u, 0u, 0u};
                    if (ok) cv[t] = *reinterpret_cast<const u32x4_any*>(ccorner + (size_t)(row0 * ldc) * ES + lane_c);
                } else {
                    cv[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                          cres, ok ? lane_c : kOut, static_cast<int>(row0 * ldc * ES), 0));
                }
            }
        };
        auto element = [&](const u32x4& w, int e) {
            if constexpr (HALF)
                return to_float<BF16>(static_cast<u16>(w[e >> 1] >> (16 * (e & 1))));
            else
                return __builtin_bit_cast(floatx4, w)[e];
        };
#pragma unroll
        for (int t = 0; t < NA; ++t) load_c(0, t);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (128 * i >= rows_left) break;
            // The other waves are done with what LDS held.
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int v = 0; v < 2; ++v)
                        *reinterpret_cast<floatx4*>(lds + (64 * wm + 16 * u + j16) * 1024 +
                                                    16 * ((32 * j + 8 * wn + 4 * v + g) ^ j16)) = alpha * acc[i][j][u][v];
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int t = 0; t < NA; ++t) {
                const int row0 = row_of(i, t), r = 16 * wave + RPA * t + er;
                float out[EPL];
#pragma unroll
                for (int q = 0; q < EPL / 4; ++q) {
                    const floatx4 f = *reinterpret_cast<const floatx4*>(lds + r * 1024 + 16 * ((ec / 4 + q) ^ (r & 15)));
#pragma unroll
                    for (int e = 0; e < 4; ++e) out[4 * q + e] = f[e];
                }
                if (any_cut) {
                    if (cut && row0 + er < rows_left) {
                        const size_t at_d = ((size_t)(row0 + er) * ldd + ec) * ES, at_c = ((size_t)(row0 + er) * ldc + ec) * ES;
#pragma unroll
                        for (int e = 0; e < EPL - 1; ++e) {
                            if (ec + e >= cols_left) break;
                            float x = out[e];
                            if constexpr (HALF) {
                                if constexpr (HAS_C) x += beta * to_float<BF16>(reinterpret_cast<const u16*>(ccorner + at_c)[e]);
                                reinterpret_cast<u16*>(dcorner + at_d)[e] = from_float<BF16>(x);
                            } else {
                                if constexpr (HAS_C) x += beta * reinterpret_cast<const float*>(ccorner + at_c)[e];
                                reinterpret_cast<float*>(dcorner + at_d)[e] = x;
                            }
                        }
                    }
                }
                if constexpr (HAS_C) {
#pragma unroll
                    for (int e = 0; e < EPL; ++e) out[e] += beta * element(cv[t], e);
                    if (i == 0) load_c(1, t);
                }
                u32x4 w;
                if constexpr (HALF)
                    w = u32x4{pack2<BF16>(out[0], out[1]), pack2<BF16>(out[2], out[3]), pack2<BF16>(out[4], out[5]),
                              pack2<BF16>(out[6], out[7])};
                else
                    w = __builtin_bit_cast(u32x4, floatx4{out[0], out[1], out[2], out[3]});
                const bool ok = full && row0 + er < rows_left;
                if constexpr (HALF && !WIDE) {
                    if (ok) *reinterpret_cast<u32x4_any*>(dcorner + (size_t)(row0 * ldd) * ES + lane_d) = w;
                } else {
                    __builtin_amdgcn_raw_buffer_store_b128(w, dres, ok ? lane_d : kOut, static_cast<int>(row0 * ldd * ES), kPolicy);
                    // The data registers stay unwritten for two wait states after the store (a VALU write
                    // right after it has replaced its first dword).
                    asm volatile("s_nop 1" ::"v"(w) : "memory");
                }
            }
        }
    };
    auto with_half = [&](auto c_tag) {
        if (!p.cd_half) {
            epilogue(c_tag, std::false_type{}, std::true_type{});
            return;
        }
        // Every row of c and d on a 4-byte address.
        const bool wide = ldd % 2 == 0 && (uintptr_t)p.d % 4 == 0 &&
                          (p.c == nullptr || (ldc % 2 == 0 && (uintptr_t)p.c % 4 == 0));
        if (wide)
            epilogue(c_tag, std::true_type{}, std::true_type{});
        else
            epilogue(c_tag, std::true_type{}, std::false_type{});
    };
    if (p.c != nullptr)
        with_half(std::true_type{});
    else
        with_half(std::false_type{});
}

// Tile rows walked as one band (tile_of).
constexpr int kBand = 4;

template <bool BF16, bool TA, bool TB>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void half_gemm_pp(
    HalfGemmParams p) {
    half_gemm_pp_tile<BF16, TA, TB>(p, blockIdx.x, kBand);
}

// Grouped GEMM over a device table of per-group parameters: the workgroup's group is the last one
// whose first tile id is at most its own.  Group starts are multiples of 8, so the group-local id
// keeps the hardware id's XCD; ids past the group's tiles are padding and exit at once (before any
// barrier, the whole workgroup).
template <bool BF16, bool TA, bool TB>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2))) void grouped_half_gemm_pp(
    GroupedHalfArgs g) {
    const int bid = blockIdx.x;
    int lo = 0, hi = g.groups - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (g.tile_start[mid] <= bid)
            lo = mid;
        else
            hi = mid - 1;
    }
    const HalfGemmParams p = g.params[lo];
    const int local        = bid - g.tile_start[lo];
    if (local >= p.tiles_m * p.tiles_n) return;
    half_gemm_pp_tile<BF16, TA, TB>(p, local, kBand);
}

// Kernel for one input type and operand orientation (ta: column-major a, tb: column-major b).
template <bool BF16>
const void* ppKernel(bool ta, bool tb) {
    if (ta) return tb ? reinterpret_cast<const void*>(&half_gemm_pp<BF16, true, true>)
                      : reinterpret_cast<const void*>(&half_gemm_pp<BF16, true, false>);
    return tb ? reinterpret_cast<const void*>(&half_gemm_pp<BF16, false, true>)
              : reinterpret_cast<const void*>(&half_gemm_pp<BF16, false, false>);
}
template <bool BF16>
const void* groupedPpKernel(bool ta, bool tb) {
    if (ta) return tb ? reinterpret_cast<const void*>(&grouped_half_gemm_pp<BF16, true, true>)
                      : reinterpret_cast<const void*>(&grouped_half_gemm_pp<BF16, true, false>);
    return tb ? reinterpret_cast<const void*>(&grouped_half_gemm_pp<BF16, false, true>)
              : reinterpret_cast<const void*>(&grouped_half_gemm_pp<BF16, false, false>);
}

}  // namespace ftrain::gemm::ppdev
