// The plain int8 matmul on the direct-to-LDS tiles of matmul_w8a8_tile.h, half and bfloat16 outputs on v_mfma_i32_16x16x64_i8.
#include "matmul_w8a8_tile.h"

namespace ascq {

void run_dma_long(const GemmParams& p, const DmaLaunch& l, int b_layout, hipStream_t st)
{
    run_dma<k16>(p, l, b_layout, st);
}

}  // namespace ascq
