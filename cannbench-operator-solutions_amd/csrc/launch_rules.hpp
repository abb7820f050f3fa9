// launch_rules.hpp - the rules that size and choose launches, plain host arithmetic without HIP types, so
// that a host program can check them at sizes no test allocates (tests/launch_rules).
#pragma once

#include <stdint.h>

namespace cb {

// A dispatch counts its work-items (blocks x threads per dimension) in 32 bits.  The row kernels
// launch one block per row (or per few rows); an operator whose launch would not fit returns
// CB_ERR_SHAPE instead of launching a truncated grid.
inline bool grid_fits(int64_t blocks, int64_t threads) { return blocks * threads < (1LL << 32); }

// Workgroups of the vectorised DequantSwigluQuant kernel, which walks the rows in steps of its grid: two
// rows per workgroup (the second row's loads in flight while the first is reduced), and at least
// enough workgroups to fill every CU twice.  Longer walks drift apart: 131072 x 4096 int32 takes
// 413 us with 2 rows each, 424 with 4, 530 with 16, 468 with 64, and 452 with 1; bf16 211, 231, 239,
// 251 and 226; 16384 rows int32 53.8 against 58.7 with 8.  From 2^33 / threads rows on (2^27 with 64
// threads) the workgroups walk more, as many as a dispatch holds.
inline int64_t dqsq_blocks(int64_t M, int64_t threads)
{
    const int64_t per_cu = 2048 / threads;  // workgroups resident per CU (8 waves per SIMD)
    const int64_t fill = 256 * per_cu * 2, half = (M + 1) / 2;
    const int64_t want = M < fill ? M : (half > fill ? half : fill), most = ((1LL << 32) - 1) / threads;
    return want < most ? want : most;
}

}  // namespace cb
