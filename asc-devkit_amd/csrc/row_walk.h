// How the row-wise kernels of elementwise.hip share out a matrix: integers only, for the device and for a host compiler alone.
// Every count of 32 bits is in range, also the last ones, where a sum such as n + 7 does not fit.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define ASCQ_HD __host__ __device__ __attribute__((always_inline))
#else
#define ASCQ_HD
#endif

namespace ascq {

ASCQ_HD inline uint32_t ceil_div(uint32_t a, uint32_t b) { return a / b + (a % b != 0u ? 1u : 0u); }

// Lanes of 8 columns for a row of n.
ASCQ_HD inline uint32_t row_lanes(uint32_t n) { return ceil_div(n, 8u); }

// The first of a lane's 8 columns, at a row's end moved back so that they end with the row (n >= 8).
ASCQ_HD inline uint32_t whole_columns(uint32_t j, uint32_t n) { return j < n && n - j < 8u ? n - 8u : j; }

// Launch shape of the row-wise vector kernels: grid_x walks the lanes of a row, grid_y groups of rows.  The
// block size (threads, half or a quarter of them) is the one that leaves the fewest idle lanes in a row's last block: 11008 columns at 8
// per lane are 10.75 blocks of 128 but 5.4 of 256, and that mostly empty sixth block cost 8 % of the kernel's time.
struct RowWalk {
    uint32_t grid_x, grid_y, block;
};
inline RowWalk row_walk(uint32_t lanes, uint32_t rows, uint32_t rows_per_group, uint32_t threads)
{
    uint32_t block = threads;
    for (uint32_t b = threads / 2u; b >= 64u; b /= 2u) {
        if (ceil_div(lanes, b) * b < ceil_div(lanes, block) * block) {
            block = b;
        }
    }
    RowWalk r{ceil_div(lanes, block), ceil_div(rows, rows_per_group), block};
    // enough blocks to fill 256 CUs several times over, but no more row groups than exist
    const uint32_t want = ceil_div(8192u * (threads / block), r.grid_x);
    r.grid_y = r.grid_y < want ? r.grid_y : want;
    r.grid_y = r.grid_y < 65535u ? r.grid_y : 65535u;
    return r;
}

// Whether the rows r0 of every workgroup's walk, r0 += grid_y * rows_per_group up to the first past the end, fit 32 bits.
inline bool walk_fits(uint32_t rows, uint32_t rows_per_group) { return rows <= 0xFFFFFFFFu - 65535u * rows_per_group; }

}  // namespace ascq
