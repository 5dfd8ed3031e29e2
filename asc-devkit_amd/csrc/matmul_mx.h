// Shared by the kernels of the block-scaled (MX) matmul: matmul_mx.hip (256 x 256 tiles) and matmul_mx_decode.hip (few
// rows).
#pragma once
#include "ascq_common.h"
#include "ascq_device.h"

namespace ascq {

struct MxParams {
    const uint8_t* a;
    const uint8_t* b;
    const uint8_t* sa;
    const uint8_t* sb;
    const float* bias;
    void* c;
    uint32_t m, n, k;       // k in elements
    uint32_t row_bytes;     // bytes of a row of a / b in the tile kernel (both operands have the same width there)
    uint32_t sk;            // bytes of a scale row
    uint32_t tiles_m, tiles_n;
    int32_t a_format, b_format, out_dtype;
};

__device__ __forceinline__ void mx_store(const MxParams& p, size_t idx, float v)
{
    if (p.out_dtype == ASCQ_F32) {
        static_cast<float*>(p.c)[idx] = v;
    } else if (p.out_dtype == ASCQ_BF16) {
        static_cast<uint16_t*>(p.c)[idx] = static_cast<uint16_t>(f32_to_bf16_bits(v));
    } else {
        static_cast<uint16_t*>(p.c)[idx] = static_cast<uint16_t>(f32_to_half_bits_sat(v));
    }
}

// matmul_mx_decode.hip: whole columns per workgroup, wavefronts split k; any m, n.  tile_shape: the tiles could take the call,
// so fp8 operands may have their precision
bool mx_decode_supported(const MxParams& p);
int launch_mx_decode(const MxParams& p, bool tile_shape, hipStream_t st);

// matmul_mx_ring.hip: tiles of 64 x 64 (shape 0), 128 x 64 and 128 x 128 for medium sizes; formats as the matrix instruction's codes (0
// e4m3, 1 e5m2, 4 e2m1, that as b beside an 8-bit a or as both), k a multiple of 128, of 256 with a 4-bit operand
int launch_mx_ring(const MxParams& p, int shape, int code_a, int code_b, hipStream_t st);

// matmul_mx_six.hip: two e1m2 operands, k a multiple of 128, on a workspace of mx_six_bytes (16-byte aligned)
size_t mx_six_bytes(uint32_t m, uint32_t n, uint32_t k);
int launch_mx_six(const MxParams& p, void* workspace, hipStream_t st);

}  // namespace ascq
