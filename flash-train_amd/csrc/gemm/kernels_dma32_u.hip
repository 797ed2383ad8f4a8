// FP32 tiles with LDS staging by DMA for operands without 16-byte alignment, row-major a and either
// b (see gemm/dma32_tile.hpp).
#include "dma32_tile.hpp"

namespace ftrain::gemm {

namespace {
template <bool TB>
const void* unaligned(Variant v) {
    using namespace d32;
    switch (v) {
        case Variant::kMfma16Dma128x128U: return reinterpret_cast<const void*>(&fp32_gemm_dma<128, 128, 2, 2, 2, false, TB, false, true>);
        case Variant::kMfma16Dma128x128US: return reinterpret_cast<const void*>(&fp32_gemm_dma<128, 128, 2, 2, 2, true, TB, false, true>);
        case Variant::kMfma16Dma64x128U: return reinterpret_cast<const void*>(&fp32_gemm_dma<64, 128, 2, 2, 2, false, TB, false, true>);
        case Variant::kMfma16Dma64x128US: return reinterpret_cast<const void*>(&fp32_gemm_dma<64, 128, 2, 2, 2, true, TB, false, true>);
        case Variant::kMfma16Dma128x64US: return reinterpret_cast<const void*>(&fp32_gemm_dma<128, 64, 4, 1, 2, true, TB, false, true>);
        case Variant::kMfma16Dma64x64US: return reinterpret_cast<const void*>(&fp32_gemm_dma<64, 64, 4, 1, 2, true, TB, false, true>);
        default: return nullptr;
    }
}
}  // namespace

const void* dma32KernelU(Variant v, bool tb) { return tb ? unaligned<true>(v) : unaligned<false>(v); }

const void* dma32Kernel64x64U(bool tb) {
    using namespace d32;
    return tb ? reinterpret_cast<const void*>(&fp32_gemm_dma<64, 64, 4, 1, 2, false, true, false, true>)
              : reinterpret_cast<const void*>(&fp32_gemm_dma<64, 64, 4, 1, 2, false, false, false, true>);
}

}  // namespace ftrain::gemm
