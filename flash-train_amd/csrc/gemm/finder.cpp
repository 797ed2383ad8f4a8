// ShapeCost Finder: ranks the kernel catalog by a roofline cost model.
//
// The reference ships only a placeholder Finder that expresses no preference
// (src/include/flash_train/family/gemm/finder.hpp:21-26); selection then falls
// back to registration order.  This Finder estimates each variant's time on
// the problem's shape and returns the variants best-first; the engine drops
// the ones whose applicability check fails (alignment, size limits) and
// caches the surviving order per problem key.
//
// Model, per variant (microseconds):
//   compute: workgroups = tiles * splits; each CU runs ceil(wgs / CUs) of
//            them back to back at the variant's sustained fraction of its
//            MFMA FLOP/clk/CU at 2.4 GHz (interpolated down to the variant's
//            single-workgroup fraction while fewer than its resident count
//            are available), plus a fixed cost per round of resident
//            workgroups.
//   memory : algorithmic bytes (a, b, d, optional c) at 80% of 8 TB/s, plus
//            the partial tiles (written and read once) for split-k; scaled
//            by the share of CUs the launch's workgroups occupy when there
//            are fewer workgroups than CUs.
//   time   = max(compute, memory) + the reduction's pass over the partial
//            tiles (split-k) + launch latency (one more for split-k).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <limits>
#include <numeric>

#include <hip/hip_runtime_api.h>

#include "ft/gemm.hpp"

namespace ftrain {
namespace gemm {

namespace {
constexpr double kClockPerMicro = 2.4e3;  // peak engine clock (MHz)
constexpr double kHbmBytesPerMicro = 8.0e6 * 0.8;  // sustained HBM bytes per microsecond
constexpr double kLaunchMicros = 1.23;
constexpr double kPoolMicros      = 3.48;  // dependency gap before the reduction kernel (fitted)
// The reduction kernel's pass over the partial tiles, relative to HBM time (fitted).
constexpr double kReduceFactor    = 1.206;
// The deep-k kernel (SplitKind::kFused): ramp of its single round, and the
// tile's last workgroup storing, counting and gathering the partial tiles
// (measured on MI355X: 3.7 us at 4 splits, 11-12 us at 16; the per-split
// figure is set so that the kernel loses to the split-k tiles at 16 splits,
// as measured: 64x1024x16384 33.9 against 31.1 us, 256x256x65536 89.8
// against 80.0).
constexpr double kFusedRampMicros     = 1.5;
constexpr double kFusedGatherMicros   = 2.2;
constexpr double kFusedPerSplitMicros = 0.9;
constexpr double kFusedStoreMicros    = 2.0;  // per round: a split workgroup's partial store and count
// Fixed cost per round of resident workgroups (operand prologue, epilogue
// stores, the ramp of the first stages); fitted with the catalog efficiencies.
constexpr double kRoundMicros     = 3.35;
constexpr double kThinRoundMicros = 7.0;  // a second round on few CUs, see modelMicros
constexpr double kTieWeight       = 1e-3;
// The whole-k form of the fp32 64x64 split tile, see modelMicros: its rate on rows of part lines, and of one
// workgroup per CU on operands larger than the L2s (8 of 4 MiB).
constexpr double kWholePartLines = 0.95;
constexpr double kWholeStreaming = 0.72;
constexpr double kL2Bytes        = 32.0 * 1048576.0;
// Whole-k 16-bit tiles on few workgroups, see modelMicros: MFMA time on rows of part lines, and a 16-bit c
// on a 128-row tile.
constexpr double kHalfPartLines = 1.4;
constexpr double kHalfCMicros   = 9.0;
// The skinny kernel for a column-major b with five rows or more: bytes per microsecond over its rounds of
// one workgroup per CU, and a fixed cost.
constexpr double kGemvManyRowsRate   = 5.9e6;
constexpr double kGemvManyRowsMicros = 9.0;
constexpr double kCuBytesPerMicro = 6.4e4;  // one CU's sustained load rate (about 27 bytes per clock)
// A DMA tile stages a partial last stage (k not a multiple of its stage) by ordinary loads once its
// pipeline has drained: per tile, the drain, the loads' latency and a barrier (bf16 8192x8192x8200 819 us
// on the 256x256 tile).  A smaller tile stages as much less: fp32 127x97x33 (one stage and a tail) takes
// 4.6 us in all on the 64x64 tile.  Grouped 16-bit launches have their own figures (groupedTerms).
constexpr double kDmaTailMicros = 3.0;  // of a 256x256 tile
// Rate of a lone workgroup of the 16-bit 128x128 DMA tiles in their form for two per CU.
constexpr double kPairedSoloEfficiency = 0.37;
constexpr uint64_t kMinSplitDepth = 256;  // reduction depth worth one split-k workgroup
constexpr uint64_t kMinGemvDepth  = 64;

uint64_t ceilDiv(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// The 16-bit 64x128 split tile (m of at most 64).
bool half64x128(const VariantInfo& vi) {
    return vi.input != FTRAIN_NUMERIC_TYPE_FP32 && vi.bm == 64 && vi.bn == 128 && vi.split == SplitKind::kPartial;
}

bool half128Dma(const VariantInfo& vi) {
    return vi.input != FTRAIN_NUMERIC_TYPE_FP32 && vi.bm == 128 && std::strstr(vi.name, "_Dma") != nullptr;
}

bool half256Dma(const VariantInfo& vi) {
    return vi.input != FTRAIN_NUMERIC_TYPE_FP32 && vi.bm == 256 && std::strstr(vi.name, "_Dma") != nullptr;
}

// Rows of a problem in tile rows of vi.  The 16-bit 256x256 DMA tile runs a last tile row of at most
// 128 rows with half the MFMAs, in 70% of the time beside other tiles (fitted with groupedTerms).
double tileRows(const VariantInfo& vi, uint64_t m) {
    const uint64_t rows = ceilDiv(m, vi.bm), left = m - (rows ? rows - 1 : 0) * vi.bm;
    return half256Dma(vi) && left <= 128 ? double(rows) - 0.3 : double(rows);
}

// Whether variant vi runs a k tail through the separate pass of the DMA tiles (stages of 32 k for
// fp32, 64 for 16-bit inputs).
bool dmaTail(const VariantInfo& vi, uint64_t k) {
    return std::strstr(vi.name, "_Dma") != nullptr && k % (vi.input == FTRAIN_NUMERIC_TYPE_FP32 ? 32 : 64) != 0;
}

double tailMicros(const VariantInfo& vi) { return kDmaTailMicros * std::min(1.0, vi.bm * vi.bn / 65536.0); }
}  // namespace

int computeUnits(FTrainDeviceId device) {
    static std::atomic<int> cached[64] = {};
    const int slot = device >= 0 && device < 64 ? device : -1;
    if (slot >= 0) {
        const int v = cached[slot].load(std::memory_order_relaxed);
        if (v > 0) return v;
    }
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        n = 256;
    }
    if (slot >= 0) cached[slot].store(n, std::memory_order_relaxed);
    return n;
}

namespace {

// Sustained fraction of the MFMA rate when a CU holds `per_cu` of the
// launch's workgroups: interpolated between one resident workgroup and the
// variant's full occupancy.
double residentEfficiency(const VariantInfo& vi, uint64_t per_cu) {
    if (vi.occupancy <= 1) return vi.efficiency;
    const double resident = double(std::min<uint64_t>(std::max<uint64_t>(per_cu, 1), uint64_t(vi.occupancy)));
    return vi.solo_efficiency + (vi.efficiency - vi.solo_efficiency) * (resident - 1.0) / double(vi.occupancy - 1);
}

// Modelled time of variant `v` with a given split count (1 = no split).
double modelMicros(const VariantInfo& vi, const GemmShape& s, bool has_c, int cus, uint64_t splits,
                   const OperandForm& o = {}) {
    const double m = double(s.m), n = double(s.n), k = double(s.k);
    // a and b in the variant's input type; c and d counted at the same size.
    const double eb   = vi.input == FTRAIN_NUMERIC_TYPE_FP32 ? 4.0 : 2.0;
    double bytes      = eb * (m * k + k * n + m * n * (has_c ? 2.0 : 1.0));
    double launch     = kLaunchMicros;
    double serial_us  = 0.0;  // work in a second kernel that cannot overlap the first
    if (vi.split == SplitKind::kPartial && (splits > 1 || vi.gemv)) {
        // The GEMM kernel writes splits partial tiles instead of d; the
        // reduction kernel then reads them (and c) and writes d.
        bytes += 4.0 * m * n * (double(splits) - 1.0 - (has_c ? 1.0 : 0.0));
        serial_us = kReduceFactor * 4.0 * m * n * (double(splits) + (has_c ? 2.0 : 1.0)) / kHbmBytesPerMicro;
        launch += kLaunchMicros + kPoolMicros;
    }
    if (vi.split == SplitKind::kFused && splits > 1) {
        // Partial tiles written and read once, plus the last workgroup's
        // store / count / gather, after the tile's other workgroups.
        const double tiles = double(ceilDiv(s.m, vi.bm) * ceilDiv(s.n, vi.bn));
        bytes += 2.0 * 4.0 * tiles * vi.bm * vi.bn * double(splits);
        serial_us = kFusedGatherMicros + kFusedPerSplitMicros * (double(splits) - 1.0);
    }
    if (vi.gemv) {
        // Too few waves cannot reach the HBM peak; about four per CU do
        // (measured with the one-pass kernel: 1024 waves over 256 CUs stream
        // 5.4-6.3 TB/s, 256 waves lose to split-k).
        // A CU also loads at a bounded rate, so a launch of few workgroups is bound by the bytes each
        // one reads (bf16 1x4096x4096, 64 workgroups of 512 KiB: 9.0 us).
        const int threads = vi.split == SplitKind::kNone ? gemvPassThreads(int(std::max<uint64_t>(s.m, 1)), o.tb) : vi.threads;
        const double wgs  = double(ceilDiv(std::max<uint64_t>(s.n, 1), uint64_t(vi.bn)) * splits);
        const double fill = std::min(1.0, wgs * (threads / 64) / (double(cus) * 4.0));
        const double per_cu = std::ceil(wgs / double(cus)) * bytes / wgs;
        // From five rows on, the form for a column-major b has room for one workgroup per CU: a last round
        // on few CUs takes as long as a full one (us, against the best split tile: 8x8192x8192, 256
        // workgroups, 58.7 / 74.9; 7x12768x4600, 399, 50 / 64; 5x8824x13680, 276, 183 / 127; 6x11688x12376,
        // 366, 174 / 147; 6x11440x6728, 358, 96 / 84; 8x9616x1416, 301, 27.6 / 23.2).
        if (o.tb && vi.split == SplitKind::kNone && s.m > 4)
            return std::ceil(wgs / double(cus)) * double(cus) / wgs * bytes / kGemvManyRowsRate + kGemvManyRowsMicros + launch;
        const double t      = std::max(bytes / (kHbmBytesPerMicro * fill), per_cu / kCuBytesPerMicro) + serial_us + launch;
        // The split-k skinny kernel keeps few loads in flight per wave and runs well below the
        // streaming model, more so with more rows of a (measured on MI355X, us, model in brackets:
        // 1x1024x4096 11.9 [8.7], 4x1024x4096 16.5 [8.9], 8x1024x8192 40.1 [12.0], 1x4096x4096 28.4
        // [16.5], 8x4096x4096 68.3 [17.2]); it lost to the one-pass kernel or a DMA split-k tile on
        // every shape measured (1x1024x4096 one-pass 6.7, 8x1024x8192 64x128 DMA split-k 13.4).
        return vi.split == SplitKind::kPartial ? t * (1.5 + double(std::min<uint64_t>(s.m, 8)) / 4.0) : t;
    }
    // Work per workgroup includes the tile padding at the m/n edges.  The
    // dispatcher refills a CU as soon as one of its workgroups retires, so a
    // CU's load is its share of workgroups, ceil(wgs / CUs), each at the
    // CU's sustained rate; below `occupancy` resident workgroups a CU runs
    // correspondingly below that rate.
    const uint64_t chunk   = splits == 1 ? s.k : ceilDiv(ceilDiv(s.k, splits), vi.bk) * vi.bk;
    const uint64_t used    = chunk == 0 ? 1 : ceilDiv(s.k, chunk);
    const uint64_t tiles   = ceilDiv(s.m, vi.bm) * ceilDiv(s.n, vi.bn);
    const uint64_t wgs     = tiles * used;
    const uint64_t per_cu  = ceilDiv(wgs, cus);
    const double depth     = double(std::max<uint64_t>(chunk, vi.bk));
    // SIMT FMAs run at half the matrix rate without packed FP32.
    double cu_rate         = vi.flop_per_clk * kClockPerMicro * residentEfficiency(vi, per_cu) * (vi.simt ? 0.5 : 1.0);
    // The whole-k form of the fp32 64x64 split tile loads twice what the 128x128 tile does per FLOP.  Rows
    // that are not whole 128-byte lines cost it more (us, against 128x128 whole-k or split: 3652x12080x7296
    // 4760 / 4410, 9584x4124x7564 4380 / 4180, 2192x2228x5840 539 / 433, but 11008x2560x1024, whole lines, 401 /
    // 472), and so does one workgroup per CU on operands that no L2 holds (7392x72x2912 73 / 50,
    // 37x13728x1992 53 / 41; 512x1536x768, in L2, 16.5 / 20).
    if (vi.split == SplitKind::kPartial && splits == 1 && vi.vec) {
        if (o.part_lines) cu_rate *= kWholePartLines;
        if (per_cu == 1 && eb * (m * k + k * n) > kL2Bytes) cu_rate *= kWholeStreaming;
    }
    const double rounds    = double(ceilDiv(per_cu, uint64_t(vi.occupancy)));
    // The deep-k kernel runs one workgroup per CU: each round pays the ramp
    // and, when split, its workgroups' partial-tile stores and arrival.
    const double per_round = vi.split != SplitKind::kFused ? kRoundMicros
                             : kFusedRampMicros + (splits > 1 ? kFusedStoreMicros : 0.0);
    // The tail pass: every tile's when whole-k, the last split's tiles when split.
    const double tails     = !dmaTail(vi, s.k) ? 0.0 : used == 1 ? rounds
                                                   : double(ceilDiv(ceilDiv(tiles, cus), uint64_t(vi.occupancy)));
    double mfma = double(per_cu) * 2.0 * vi.bm * vi.bn * depth / cu_rate;
    // The 16-bit 128x128 DMA tiles between one and two workgroups per CU: a second workgroup costs a
    // CU half of what the first does, and only some CUs hold one (bf16, k 4096: 288 tiles 45 us, 384 52,
    // 512 60).
    if (half128Dma(vi) && wgs > uint64_t(cus) && wgs <= 2 * uint64_t(cus)) {
        const double one = mfma / 2.0 * residentEfficiency(vi, 2) / kPairedSoloEfficiency;
        mfma             = one + (mfma - one) * (double(wgs) / double(cus) - 1.0);
    }
    // A second round of 16-bit 256x256 tiles on a fifth of the CUs or fewer has nothing beside its loads
    // and stores (bf16, 256x256 against 128x128 DMA tile, us: 12714x1344x1216 62.7 / 56.8, 1824x9088x640
    // 37.4 / 33.4, 7789x2176x128 27.7 / 19.2; from k 4160 on the 256x256 tile wins: 8960x2048x4160 160 /
    // 165, 12614x1408x5056 199 / 212).  Not where n leaves rows of odd 64-byte pieces, which the smaller
    // tiles touch twice: 2048x9432x64 22.7 / 41.5, 7424x2328x256 32.8 / 37.8, 3584x5112x768 44 / 59.
    if (vi.input != FTRAIN_NUMERIC_TYPE_FP32 && vi.bm == 256 && s.n % 32 == 0 && wgs > uint64_t(cus) &&
        5 * wgs <= 6 * uint64_t(cus))
        mfma += kThinRoundMicros;
    // Whole-k 16-bit tiles other than the 256x256 DMA one, where a split over k would still be one round.
    // Rows of part lines slow a 128x128 tile's loads (bf16, us, whole-k against split 128x128 DMA tile:
    // 141x1176x1128 14.2 / 9.4, 253x2136x1392 16.6 / 13.1, 233x3336x1560 18.5 / 14.8; whole lines 350x1824x1088
    // 10.5 / 11.6), and a 16-bit c, which these tiles load 2 bytes at a time, comes on top (122x2032x1144 with c
    // 21.6 / 11.0, 107x6680x1552 29.0 / 14.3, 659x1384x704 20.7 / 11.9).  The per-element 64x64 tile pays for
    // its c at any number of workgroups (596x2864x568 26.8 against 16.5 on the split tile).
    if (vi.input != FTRAIN_NUMERIC_TYPE_FP32 && vi.split == SplitKind::kNone && !half256Dma(vi)) {
        const bool few = 2 * wgs <= uint64_t(cus);
        if (vi.bm == 128 && o.part_lines && few) mfma *= kHalfPartLines;
        if (has_c && o.cd_half && (vi.bm == 64 || few)) mfma += kHalfCMicros * vi.bm / 128.0;
    }
    const double compute   = mfma + rounds * per_round + tails * tailMicros(vi);
    // A launch with fewer workgroups than CUs streams memory through only that many of them (a CU
    // moves a bounded number of bytes per clock): 64x4096x14336 bf16 on the 64x128 split tile took
    // 36.3 us at 4 splits (128 workgroups) against 23.8 us at 8.  On the 16-bit 64x128 split tile
    // (m of at most 64) 85% of the CUs already stream at the full rate: 32x14336x4096 22.5 us at 2
    // splits (224 workgroups) against 24.1 at 4, and 5-10% the same way at 4 to 64 rows of n 13824
    // and 14336; the 128x128 split tile at such counts lost 4-15%, so it keeps the plain fraction.
    const double fill = std::min(1.0, double(wgs) / (double(cus) * (half64x128(vi) ? 0.85 : 1.0)));
    double memory     = bytes / (kHbmBytesPerMicro * fill);
    // A whole-k launch of at most half as many workgroups as CUs is bound by what each workgroup
    // loads at one CU's rate, not by a fraction of HBM: bf16 128x4096x1024 on the 128x128 DMA
    // tile (32 workgroups of 0.5 MiB) 9.3 us against 13.2 for the split tile the fraction picked,
    // 128x256x512 6.5 against 10.7 for the 64x64 unaligned tile.  At 224 workgroups (4x28672x4096)
    // the fraction still ranks right.
    if ((vi.split == SplitKind::kNone || (vi.split == SplitKind::kPartial && splits == 1)) && !vi.simt &&
        2 * wgs <= uint64_t(cus)) {
        const double wg_bytes = eb * double(vi.bm + vi.bn) * double(s.k) + 4.0 * vi.bm * vi.bn;
        memory = std::max(bytes / kHbmBytesPerMicro, wg_bytes / kCuBytesPerMicro);
    }
    // When memory bounds several variants alike, the one with the least compute overlaps it best
    // (64x14336x4096 bf16 at 4 splits: the 64x128 DMA split tile 25.9 us, the 128x128 one 27.6,
    // the register-staged 128x128 30.2): a thousandth of the compute time breaks such ties.
    return std::max(compute, memory) + serial_us + launch + kTieWeight * compute;
}

}  // namespace

namespace {
std::atomic<uint32_t> g_forced_splits{0};
}

void forceSplits(uint32_t s) { g_forced_splits.store(s, std::memory_order_relaxed); }

uint32_t chooseSplits(Variant v, const GemmShape& s, int cus) {
    const VariantInfo& vi = info(v);
    if (vi.split == SplitKind::kNone) return 1;
    if (const uint32_t forced = g_forced_splits.load(std::memory_order_relaxed); forced > 0 && !vi.gemv) {
        // Clamped to whole reduction steps per split, the workspace cap, and
        // (deep-k) one arrival counter per tile.
        const uint64_t tiles = std::max<uint64_t>(ceilDiv(s.m, vi.bm) * ceilDiv(s.n, vi.bn), 1);
        const uint64_t unit  = vi.split == SplitKind::kPartial ? s.m * s.n * sizeof(float)
                                                               : tiles * vi.bm * vi.bn * sizeof(float);
        const uint64_t most =
            std::min<uint64_t>(s.k / vi.bk, (kMaxPartialBytes - kCounterBytes) / std::max<uint64_t>(unit, 1));
        const uint64_t got = std::min<uint64_t>(forced, most);
        return static_cast<uint32_t>(got >= 2 ? got : vi.split == SplitKind::kPartial ? 0 : 1);
    }
    const uint64_t min_depth = vi.gemv ? kMinGemvDepth : kMinSplitDepth;
    uint64_t most            = std::min<uint64_t>(1024, s.k / min_depth);
    if (vi.split == SplitKind::kPartial && s.m * s.n > 0)
        most = std::min<uint64_t>(most, (kMaxPartialBytes - kCounterBytes) / (s.m * s.n * sizeof(float)));
    if (vi.split == SplitKind::kFused) {
        // One split is a plain whole-k launch; more only while the partial
        // tiles fit the cap.
        const uint64_t tile_bytes = ceilDiv(s.m, vi.bm) * ceilDiv(s.n, vi.bn) * vi.bm * vi.bn * sizeof(float);
        most = std::min<uint64_t>(most, (kMaxPartialBytes - kCounterBytes) / std::max<uint64_t>(tile_bytes, 1));
        uint64_t best = 1;
        double best_t = modelMicros(vi, s, false, cus, 1);
        for (uint64_t sp = 2; sp <= most; sp *= 2) {
            const double t = modelMicros(vi, s, false, cus, sp);
            if (t < best_t * 0.999) {
                best_t = t;
                best   = sp;
            }
        }
        return static_cast<uint32_t>(best);
    }
    if (vi.gemv && most < 2) return 1;  // the skinny kernel also runs unsplit
    if (s.m == 0 || s.n == 0) return 0;
    // Smallest modelled time over 2^i and 3 * 2^i in [2, most] (ties: fewer splits), and 1 for a tile
    // with a whole-k form.
    uint64_t best = 0;
    double best_t = std::numeric_limits<double>::infinity();
    const auto consider = [&](uint64_t sp) {
        const double t = modelMicros(vi, s, false, cus, sp);
        if (t < best_t * 0.999) {
            best_t = t;
            best   = sp;
        }
    };
    if (unsplitForm(v)) consider(1);
    for (uint64_t sp = 2; sp <= most; sp *= 2) {
        consider(sp);
        // Not for the 16-bit 64x128 tile: it streams from memory, and workgroups just past a multiple of
        // the CUs cost it more than the finer choice gives (bf16, column-major b, us at 2 / 3 / 4 splits:
        // 16x11008x5120 28.6 / 33.1 / 29.8, 4x13824x5120 30.6 / 35.2 / 32.6; 2x6016x8992 at 4 / 6 25.0 / 32.0).
        // Nor for the 128x128 DMA tile where that one applies: a finer count would win it the tie on memory
        // that the smaller tile runs faster (bf16, 64x128 / 128x128 tile: 42x13040x13920 87 / 110 at 3 splits,
        // 12x12168x13472 60 / 81, 57x11832x6224 45 / 57).
        if (!vi.gemv && !half64x128(vi) && !(half128Dma(vi) && s.m <= 64) && sp + sp / 2 <= most) consider(sp + sp / 2);
    }
    return static_cast<uint32_t>(best);
}

double estimateMicros(Variant v, const GemmShape& s, bool has_c, int cus, const OperandForm& o) {
    const VariantInfo& vi = info(v);
    if (vi.gemv && s.m > uint64_t(vi.bm)) return std::numeric_limits<double>::infinity();
    const uint32_t splits = vi.split != SplitKind::kNone ? chooseSplits(v, s, cus) : 1;
    if (splits == 0) return std::numeric_limits<double>::infinity();
    return modelMicros(vi, s, has_c, cus, splits, o);
}

// A row-major b needs n, a column-major a m of at least a tile (the kernel moves its last tile inside the
// matrix).  The large tile runs a stage in half the time, but costs more before its first and after its last
// one, most with a 16-bit c, which it loads 2 bytes at a time.  bf16, us, 64x64 / 128x128 tile:
//   16-bit c and d: 1000x1003x700 28 / 36, x1100 40 / 40; 1500x3501x316 36 / 37, x700 60 / 45; 3000x4001x700
//     100 / 80; column-major b 1000x3003x700 31 / 36, x1100 44 / 42, 4000x9001x316 131 / 171, x700 224 / 204;
//   fp32 c and d: 1000x1003x508 20 / 22, x700 26 / 24, x1100 37 / 28; 3000x4001x316 55 / 58, x508 75 / 64;
//     column-major b 3000x4001x508 64 / 63, 4000x9001x508 174 / 174, x1100 330 / 211;
//   no c: 1000x1003x316 12 / 13, x508 18 / 15, x700 24 / 16; 3000x4001x316 46 / 48, x508 66 / 53; column-major b
//     1000x1003x508 16 / 16, x700 21 / 18; 4000x9001x316 111 / 134, x508 158 / 143; 16-bit d 1000x1003x316
//     13 / 18, x700 25 / 21.
bool takes128(const GemmShape& s, bool ta, bool tb, bool has_c, bool cd_half, int cus) {
    if (s.m <= 64 || s.n <= 64 || (ta && s.m < 128) || (!tb && s.n < 128)) return false;
    const uint64_t tiles = ceilDiv(s.m, 64) * ceilDiv(s.n, 64);
    if (has_c && cd_half) return s.k >= (tiles > 4 * uint64_t(cus) ? 640 : 1152);
    if (tiles > 2 * uint64_t(cus)) return s.k >= (tb || has_c ? 512 : 384);
    return s.k >= 640;
}

namespace {
// Terms of a grouped launch on a 16-bit tile, added up, in microseconds: per microsecond of MFMAs at peak rate
// (padding included) of the CU with the most tiles, where it has one (alone) or more, and of all CUs on average
// (mean: tiles of unlike depth even out); fixed; per round with a k tail; and per microsecond that the operands,
// d, and a d whose rows are not whole 64-byte pieces take at HBM rate.  Unlike a plain launch, where the larger
// of compute and memory decides, every group streams operands of its own through few workgroups.
struct GroupedTerms {
    double mfma, alone, mean, fixed, tail, operands, d, d_pieces;
};

// Fitted (least relative squares, MI355X) to every tile on 1197 sampled bf16 and fp16 products: 2 to 128 experts,
// 32 to 32768 ragged tokens, sides of 64 to 14336, forward and weight gradient.  The tile ranked first takes 2%
// longer than the fastest on average, also of those below 20 GFLOP; ranked by the terms of a plain launch it took
// 6% longer in the large forwards, 26% in the large weight gradients and 17% in the small products (bf16, us,
// register-staged / two-group 256x256 tile: weight gradient 5824x5736 over 53 experts and 1121 tokens 3888 /
// 1623, 9584x4416 over 11 and 14374 1559 / 1215; forward, 128x128 DMA / two-group tile: 3805x10000x5776 over 9
// experts 729 / 514, 1689x2136x3264 over 18 61 / 94).
GroupedTerms groupedTerms(const VariantInfo& vi) {
    const bool dma = std::strstr(vi.name, "_Dma") != nullptr;
    if (vi.bm == 256)
        return dma ? GroupedTerms{0.83, 1.17, 0.86, 4.0, 2.7, 0.59, 1.10, 0.20} : GroupedTerms{1.29, 1.41, 0.80, 4.6, 3.8, 0.32, 0.82, 1.25};
    if (vi.bm == 128)
        return dma ? GroupedTerms{2.22, 3.10, 0.28, 1.6, 2.0, 0.67, 0.67, 1.15} : GroupedTerms{2.61, 3.61, 0.29, 2.2, 2.5, 0.52, 0.72, 0.96};
    return GroupedTerms{14.0, 30.6, 0.0, 2.3, 0.1, 0.0, 0.43, 0.41};
}
}  // namespace

double groupedMicros(Variant v, const std::vector<GemmShape>& shapes, bool has_c, bool cd_half, int cus) {
    // The groups' tiles share one grid: a CU's load is its share of all
    // tiles, each costing its own group's depth; bytes add over the groups.
    const VariantInfo& vi = info(v);
    const bool half = vi.input != FTRAIN_NUMERIC_TYPE_FP32;
    const double eb = half ? 2.0 : 4.0, ed = cd_half ? 2.0 : 4.0;
    double flops = 0.0, operands = 0.0, d = 0.0, d_pieces = 0.0;
    uint64_t tiles = 0, tail_tiles = 0;
    for (const GemmShape& s : shapes) {
        const uint64_t t = ceilDiv(s.m, vi.bm) * ceilDiv(s.n, vi.bn);
        tiles += t;
        if (half ? s.k % 64 != 0 : dmaTail(vi, s.k)) tail_tiles += t;
        flops += tileRows(vi, s.m) * double(ceilDiv(s.n, vi.bn)) * 2.0 * vi.bm * vi.bn * double(std::max<uint64_t>(s.k, half ? 64 : vi.bk));
        operands += eb * (double(s.m) * s.k + double(s.k) * s.n);
        const double out = ed * double(s.m) * double(s.n) * (has_c ? 2.0 : 1.0);
        d += out;
        if (s.n % (cd_half ? 32 : 16) != 0) d_pieces += out;
    }
    if (tiles == 0) return kLaunchMicros;
    const uint64_t per_cu = ceilDiv(tiles, cus);
    const double peak     = double(per_cu) * (flops / double(tiles)) / (vi.flop_per_clk * kClockPerMicro);
    const double rounds   = double(ceilDiv(per_cu, uint64_t(vi.occupancy)));
    const double tails    = double(ceilDiv(ceilDiv(tail_tiles, cus), uint64_t(vi.occupancy)));
    if (half) {
        const GroupedTerms g = groupedTerms(vi);
        const double mean    = flops / (double(cus) * vi.flop_per_clk * kClockPerMicro);
        return (per_cu > 1 ? g.mfma : g.alone) * peak + g.mean * mean + g.fixed + g.tail * tails +
               (g.operands * operands + g.d * d + g.d_pieces * d_pieces) / kHbmBytesPerMicro + kLaunchMicros;
    }
    const double compute = peak / residentEfficiency(vi, per_cu) + rounds * kRoundMicros + tails * tailMicros(vi);
    return std::max(compute, (operands + d) / kHbmBytesPerMicro) + kLaunchMicros;
}

}  // namespace gemm

std::vector<std::string> ShapeCostFinder::candidates(const GemmProblem& problem, const Constraints& constraints) {
    // Rank on the shape the kernels run: a column-major d swaps m and n.
    GemmLaunch g;
    const bool runs   = problem.launch(g) == nullptr;
    const GemmShape s = runs ? g.shape : problem.shape();
    const int cus     = gemm::computeUnits(constraints.device());
    const bool has_c  = problem.c().memory() != nullptr;
    gemm::OperandForm o;
    if (runs) {
        const int64_t line = problem.a().numericType() == FTRAIN_NUMERIC_TYPE_FP32 ? 32 : 64;  // elements
        o.tb               = g.tb;
        o.cd_half          = problem.d().numericType() != FTRAIN_NUMERIC_TYPE_FP32;
        o.part_lines       = g.lda % line != 0 || g.ldb % line != 0;
    }
    std::vector<std::pair<double, int>> ranked;
    for (int i = 0; i < static_cast<int>(gemm::Variant::kCount); ++i) {
        // Only variants for a's element type compete.
        if (gemm::info(static_cast<gemm::Variant>(i)).input != problem.a().numericType()) continue;
        const double t = gemm::estimateMicros(static_cast<gemm::Variant>(i), s, has_c, cus, o);
        if (std::isfinite(t)) ranked.emplace_back(t, i);
    }
    std::stable_sort(ranked.begin(), ranked.end(),
                     [](const auto& x, const auto& y) { return x.first < y.first; });
    std::vector<std::string> names;
    names.reserve(ranked.size());
    for (const auto& r : ranked) names.emplace_back(gemm::info(static_cast<gemm::Variant>(r.second)).name);
    return names;
}

}  // namespace ftrain
