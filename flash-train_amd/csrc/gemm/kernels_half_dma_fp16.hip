// FP16 tiles with LDS staging by DMA, every operand orientation: 256x256 (gemm/pingpong_tile.hpp),
// 128x128 and 64x128 (gemm/dma_tile.hpp).
#include "dma_tile.hpp"
#include "pingpong_tile.hpp"

namespace ftrain::gemm {

const void* dmaKernelFp16(bool ta, bool tb) { return ppdev::ppKernel<false>(ta, tb); }

const void* groupedDmaKernelFp16(bool ta, bool tb) { return ppdev::groupedPpKernel<false>(ta, tb); }

const void* groupedDma128KernelFp16(bool ta, bool tb) { return ddev::groupedDmaKernel<false>(ta, tb); }

const void* dma64x128KernelFp16(bool ta, bool tb) { return ddev::dma64x128Kernel<false>(ta, tb); }

const void* dma128KernelFp16(bool ta, bool tb, bool split, bool solo) {
    return ddev::dma128Kernel<false>(ta, tb, split, solo);
}

}  // namespace ftrain::gemm
