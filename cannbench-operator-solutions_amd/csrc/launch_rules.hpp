// launch_rules.hpp - the rules that size and choose launches, plain host arithmetic without HIP types, so
// that a host program can check them at sizes no test allocates (tests/launch_rules).
#pragma once

#include <cmath>
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

// Workgroups of the decode-shaped GroupedMatmulSwigluQuant, which draw ntl tiles for each group with rows:
// one per CU (cus), at most ntl for every group, with rows or without.  A grid of only as many
// workgroups as there are tiles was slower: 22 of 256 experts (198 tiles of 5568 x 2176) take 72 to 105 us
// from 256 workgroups, 108 from 198.
inline int64_t gmsq_decode_grid(int64_t groups, int64_t ntl, int64_t cus) { return groups * ntl < cus ? groups * ntl : cus; }

// How groups fill 256-row tiles.
struct TileFill {
    int64_t frags = 0, tiles = 0, max_rows = 0;  // 32-row fragments with valid rows, 256-row tiles
    int64_t used = 0, heavy = 0;                 // groups with rows, with more than 256
};

inline TileFill tile_fill(const int64_t* gl, int64_t E)
{
    TileFill f;
    int64_t prev = 0;
    for (int64_t g = 0; g < E; ++g) {
        const int64_t rows = gl[g] - prev;
        f.frags += (rows + 31) / 32;
        f.tiles += (rows + 255) / 256;
        f.used += rows > 0;
        f.heavy += rows > 256;
        f.max_rows = rows > f.max_rows ? rows : f.max_rows;
        prev = gl[g];
    }
    return f;
}

// Whether the GroupedMatmulSwigluQuant prefill kernel leaves out the publish and requant of 32-row
// fragments without valid rows (its SKIP instance): yes when no 256-row tile is full enough to lose by it,
// or when most groups have one tile and enough fragments are empty.  Measured gain of SKIP, by valid
// share of the fragments:
//   256 x 7168 x 4096:  47 rows per expert (0.25) 1.035, 128 rows (0.5) 1.037, 192 (0.75) 1.016,
//                       256 (1.0) 0.99, Zipf 128 on average (0.43) 1.025, Zipf 512 (0.81) 1.004
//   128 x 2048 x 2048:  47 rows 1.18, 128 rows 1.08, 300 rows (0.62) 0.93, 288 rows (0.56) 0.93
//   64 x 2048 x 1536:   47 rows 1.22, 300 rows 0.95; 64 x 1024 x 2048, 600 rows uneven (0.80) 1.06
//   80 calls with Zipf routing (0.45 to 0.86, 70 to 5600 tiles): 0.99 to 1.09
// Experts of just over 256 rows (a full tile and a nearly empty one, valid share 9/16 at least) lose
// most: a workgroup meets the same kind of tile in every round, and the early ones run out of step.
inline bool gmsq_skips_empty(const int64_t* gl, int64_t E)
{
    const TileFill f = tile_fill(gl, E);
    return f.max_rows <= 192 || (2 * f.heavy < f.used && 20 * f.frags < 17 * 8 * f.tiles);  // 0.85
}

// The same question for the epilogue of the ring dequant GEMM (its SKIP instance): yes unless at least
// half of the groups have more than one tile and 9 of 16 fragments are valid.  Time with SKIP over
// without, 130 calls of 800 to 70000 rows:
//   groups of at most 256 rows:                                     0.90 to 1.01
//   under half of the groups past 256 rows (skewed routing):        0.87 to 1.01
//   half of the groups or more past 256 rows, valid share under 0.56: 0.92 to 1.0
//   the same, valid share 0.56 to 0.9:                              0.97 to 1.09: 64 experts of 2944 x 6464
//     with 336 rows on average 606 us without, 659 with; 256 experts of 1088 x 4672 with 273 rows 857 against
//     902; 64 experts of 3328 x 6400 with 571 rows 956 against 924
// (a group's full and nearly empty tile again: with SKIP the light tiles' workgroups run ahead and
// the row tiles of a group no longer meet at their weight slab).
inline bool ring_skips_empty(const int64_t* gl, int64_t E)
{
    const TileFill f = tile_fill(gl, E);
    return 2 * f.heavy < f.used || 16 * f.frags < 9 * 8 * f.tiles;
}

// Time model of a tiled GEMM for the rules that choose a tile: a tile alone on its CU takes p us per
// K unit and o us for its prologue and epilogue; with a tile on each of the cus CUs a round takes r us
// per K unit and o us (r above p: the CUs share L2 and fabric bandwidth; below: several workgroups
// per CU hide each other's latency).
inline double tile_rounds_us(int64_t tiles, double units, double p, double r, double o, int64_t cus)
{
    const double alone = units * p + o, full = units * r + o;
    if (tiles < cus && full > alone) return alone + (full - alone) * (double)tiles / (double)cus;
    const double t = (double)((tiles + cus - 1) / cus) * full;
    return t > alone ? t : alone;
}

// ---- the dequant GEMM's choice of kernel (QuantMatmul, the grouped down-projection) -------------
// Estimated time in us of a BM x BN tile kernel over the call (tile_rounds_us: p us per 128 of K for a
// tile alone on its CU, r in a full round of 256, o per tile); the bytes the call must move pass at
// bw TB/s, partly hidden by the multiplications (the two times combine as the root of their
// squares: powers of 3 and 4 fit worse); f us per call.  The skinny kernel (at most 32 rows per group, in
// one or two blocks of 16), the 256 x 256 ring core (more than 32 rows, batch 1, K of at least 256) and the
// 8-wave 256 x 256 kernel (more than 32 rows, other batches and K) are candidates like the others.  The
// constants are fits (bw and f need not be physical) to 1900 calls, 1 to 65536 rows, K 64 to 10240, N 64 to
// 16384, 1 to 256 groups, evenly and unevenly filled, 1 to 32 batches, on which every candidate was timed:
// the choice is 0.9% off the fastest on average.  Against taking no tile at all one call in a hundred loses
// more than 2% (32 x (79 x 1728 x 832), 28 us against 24; 256 groups of 768 x 6656 with 1 row, at most 30,
// 129 against 118); with the ring at 1.55 us per 128 of K and its constants for the 8-wave kernel too it was
// one in sixteen, up to 40% (1614 x 3648 x 12288, 111 against 95; 11288 x 208 x 1088, 19 against 14).
// Measured:
//   us, by rows (dense 7168 x 4096)          us, by rows per expert (256 x 2048 x 7168, drawn unevenly)
//                  24    300   1024  2048  4096       8     24    47    96    256
//   32 x 64       19.2   39     96   189   379       803    -     -     -      -
//   64 x 128      23.5   25     47    90   182       677   777   822  1054  2076
//   64 x 256      36     36     47    82   164       656   723   794   984  1766
//   128 x 128     26     28     37    74   152       910   954   993  1080  2120
//   128 x 256     42     43     49    65   131       787   830   894   988  1749
//   ring           -     67    101   104   105        -    752   817   917  1403
//   skinny        52      -      -     -     -       615
// With 2048 x 1024 weights 24 rows take 6.0 us (32 x 64) against 16.3 (skinny), 1024 rows 11.3
// (64 x 128) against 28 (ring); 64 x 768 x 2048 with 96 / 200 rows per expert 34 / 44 (ring) against
// 41 / 63 (64 x 256).  8-wave kernel: 11288 x 208 x 1088 13.7 against 19.2 (64 x 256), 32 x (94 x 832 x
// 1280) 14.3 against 18.9 (64 x 128).
inline constexpr int kSkinnyMaxRows = 32;  // groups up to this many rows can take the skinny core

struct DeqCand {
    int bm, bn, threads;  // threads 0: the launch does not grow with the number of tiles
    double p, r, o, bw, f;
    double e;  // share of p and r that a tile takes whatever its valid rows; the rest goes with its valid 32-row fragments
};
enum { DEQ_RING = 5, DEQ_SKINNY = 6, DEQ_LDS = 7, DEQ_SKINNY2 = 8 };  // 6, 8: one and two blocks of 16 rows
inline constexpr DeqCand kDeqCand[] = {
    {32, 64, 256, 0.30, 0.152, 1.5, 5.2, 2.0, 1.0},   {64, 128, 256, 0.30, 0.31, 2.7, 7.0, 2.9, 1.0},
    {64, 256, 256, 0.66, 0.57, 4.2, 6.7, 1.2, 1.0},   {128, 128, 512, 0.34, 0.486, 6.8, 6.5, 2.0, 1.0},
    {128, 256, 512, 0.31, 0.78, 8.9, 5.8, 1.62, 1.0}, {256, 256, 0, 1.07, 1.07, 12.9, 5.6, 3.7, 0.39},
    {32, 256, 0, 0.85, 0.30, 1.0, 6.3, 3.0, 1.0},     {256, 256, 0, 0.92, 0.92, 5.7, 5.9, 5.3, 0.73},
    {32, 256, 0, 0.70, 0.30, 6.0, 6.3, 3.0, 1.0},
};

// The index of the cheapest candidate, -1 where none fits a dispatch.
inline int pick_deq(const int64_t* gl, int64_t E, int64_t M, int64_t K, int64_t N, int64_t batch, bool ring_ok, int64_t cus)
{
    const double units = (double)((K + 127) / 128);
    int64_t mt[4] = {0, 0, 0, 0}, used = 0, prev = 0, max_rows = 0;  // row tiles of 32, 64, 128 and 256 rows
    for (int64_t g = 0; g < E; ++g) {
        const int64_t rows = gl[g] - prev;
        max_rows = rows > max_rows ? rows : max_rows;
        for (int j = 0; j < 4; ++j) mt[j] += (rows + (32 << j) - 1) >> (5 + j);
        used += rows > 0;
        prev = gl[g];
    }
    const double bytes = (double)batch * ((double)used * K * N + (double)M * (K + 2 * N));
    const double valid = (double)mt[0] / (8.0 * (double)mt[3]);  // of the 256-row tiles' fragments
    // the kernel that the call takes without a tile
    const int untiled = max_rows <= 16               ? DEQ_SKINNY
                        : max_rows <= kSkinnyMaxRows ? DEQ_SKINNY2
                        : ring_ok && batch == 1      ? DEQ_RING
                                                     : DEQ_LDS;
    double best_t = 0;
    int best = -1;
    for (int i = 0; i < (int)(sizeof(kDeqCand) / sizeof(kDeqCand[0])); ++i) {
        const DeqCand& c = kDeqCand[i];
        if (i >= DEQ_RING && i != untiled) continue;
        int64_t tiles = mt[c.bm == 32 ? 0 : c.bm == 64 ? 1 : c.bm == 128 ? 2 : 3] * ((N + c.bn - 1) / c.bn);
        if (!grid_fits(tiles, c.threads)) continue;
        tiles *= batch;
        const double k = c.bm == 256 ? c.e + (1.0 - c.e) * valid : 1.0, o = c.bm == 256 ? c.o * (0.2 + 0.8 * valid) : c.o;
        const double run = tile_rounds_us(tiles, units, c.p * k, c.r * k, o, cus);
        const double mem = bytes / (c.bw * 1e6);
        const double t = c.f + std::sqrt(run * run + mem * mem);
        if (best < 0 || t < best_t) {
            best = i;
            best_t = t;
        }
    }
    return best;
}

// ---- the 16-bit GroupedMatmul's choice of tile --------------------------------------------------
// Estimated time of each tile over the call, in the terms of the int8 rule (tile_rounds_us, units of 128
// bytes of K), combined with the bytes at bw TB/s as the root of the sum of fourth powers (squares put calls
// near the weight stream's time a tile too low); the least is taken.  The choice does not look at the
// weight layout, so that [K][N] and [N][K] storage of the same weights are summed in the same order and
// agree bit for bit.  The constants are fitted to 500 calls (8 to 16384 rows, K and N 256 to 5120, 1 to 64
// groups, both layouts) on which every tile was timed: the choice is 0.8% off the fastest on average.
// Measured us, 64 experts of 4096 x 4096 bf16, [K][N] / [N][K] weights, groups drawn unevenly (first: the
// 256 x 256 double-buffered kernel for every call):
//   rows per expert     8          24         64         128        256         512
//   (256 x 256 only) 457 / 493  470 / 498  475 / 517  513 / 537  854 / 793  1332 / 1312
//   32 x 64          363 / 349  384 / 365  576 / 584  881 / 877    -           -
//   64 x 128         360 / 349  376 / 361  461 / 451  606 / 592  921 / 927  1651 / 1714
//   64 x 256         334 / 362  342 / 375  429 / 498  556 / 633  858 / 994  1513 / 1872
//   128 x 128        392 / 367  403 / 377  429 / 400  566 / 547  837 / 819  1430 / 1429
//   128 x 256        354 / 359  360 / 366  373 / 383  524 / 487  752 / 724  1246 / 1240
//   256 x 256        418 / 493  425 / 498  443 / 517  480 / 537  807 / 793  1177 / 1312
// With 64 rows in every group 64 x 256 takes 361 / 398 and 128 x 256 376 / 384; with 128 rows 491 / 544 and
// 397 / 410; with 256 rows 128 x 256 takes 645 / 632 and 256 x 256 562 / 603.
// 8 experts of 2048 x 1536, 8 rows each: 53 -> 13.6 (32 x 64); 1024 rows each: 69 -> 62 (256 x 256).
struct GmmCand {
    int bm, bn, threads;
    double p, r, o, bw;
};
inline constexpr GmmCand kGmmCand[] = {
    {32, 64, 256, 0.15, 0.15, 1.8, 6.1},   {64, 128, 256, 0.36, 0.30, 4.7, 6.0},  {64, 256, 256, 0.79, 0.79, 4.8, 6.3},
    {128, 128, 512, 0.24, 0.46, 7.9, 5.9}, {128, 256, 512, 0.36, 0.82, 10.1, 6.3}, {256, 256, 512, 0.66, 1.55, 10.2, 11.7},
};

// The index of the cheapest tile, -1 where none fits a dispatch.
inline int pick_gmm(const int64_t* gl, int64_t E, int64_t M, int64_t K, int64_t N, int64_t cus)
{
    const double units = (double)((K + 63) / 64);
    int64_t mt[4] = {0, 0, 0, 0}, used = 0, prev = 0;  // row tiles of 32, 64, 128 and 256 rows
    for (int64_t g = 0; g < E; ++g) {
        const int64_t rows = gl[g] - prev;
        for (int j = 0; j < 4; ++j) mt[j] += (rows + (32 << j) - 1) >> (5 + j);
        used += rows > 0;
        prev = gl[g];
    }
    const double bytes = 2.0 * ((double)used * K * N + (double)M * (K + N));
    double best_t = 0;
    int best = -1;
    for (int i = 0; i < (int)(sizeof(kGmmCand) / sizeof(kGmmCand[0])); ++i) {
        const GmmCand& c = kGmmCand[i];
        const int64_t tiles = mt[c.bm == 32 ? 0 : c.bm == 64 ? 1 : c.bm == 128 ? 2 : 3] * ((N + c.bn - 1) / c.bn);
        if (!grid_fits(tiles, c.threads)) continue;
        const double run = tile_rounds_us(tiles, units, c.p, c.r, c.o, cus);
        const double mem = bytes / (c.bw * 1e6);
        const double t = run * run * run * run + mem * mem * mem * mem;
        if (best < 0 || t < best_t) {
            best = i;
            best_t = t;
        }
    }
    return best;
}

}  // namespace cb
