// The plain int8 matmul on the direct-to-LDS tiles of matmul_w8a8_tile.h where k ends inside a K step.
#include "matmul_w8a8_tile.h"

namespace ascq {

void run_dma_ragged(const GemmParams& p, const DmaLaunch& l, int b_layout, hipStream_t st)
{
    run_dma<k32Ragged>(p, l, b_layout, st);
}

}  // namespace ascq
