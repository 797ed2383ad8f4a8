// BF16 tiles with LDS staging by DMA, every operand orientation: 256x256 (gemm/pingpong_tile.hpp),
// 128x128 and 64x128 (gemm/dma_tile.hpp).
#include "dma_tile.hpp"
#include "pingpong_tile.hpp"

namespace ftrain::gemm {

const void* dmaKernelBf16(bool ta, bool tb) { return ppdev::ppKernel<true>(ta, tb); }

const void* groupedDmaKernelBf16(bool ta, bool tb) { return ppdev::groupedPpKernel<true>(ta, tb); }

const void* groupedDma128KernelBf16(bool ta, bool tb) { return ddev::groupedDmaKernel<true>(ta, tb); }

const void* dma64x128KernelBf16(bool ta, bool tb) { return ddev::dma64x128Kernel<true>(ta, tb); }

const void* dma128KernelBf16(bool ta, bool tb, bool split, bool solo) {
    return ddev::dma128Kernel<true>(ta, tb, split, solo);
}

}  // namespace ftrain::gemm
