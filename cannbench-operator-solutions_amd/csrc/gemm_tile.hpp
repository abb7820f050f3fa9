// gemm_tile.hpp - GEMM tiles for the shapes between the skinny (decode) cores and the 256 x 256
// cores: int8 (QuantMatmul, the grouped down-projection) and fp16 / bf16 (GroupedMatmul).
//
// One workgroup of 4 or 8 waves computes one BM x BN tile.  The waves split the tile's rows (WM), its
// columns (WN) and each stage's K (WK): with WK = 4 every wave multiplies the whole tile over a
// quarter of each stage, so a wave reads FM + FN fragments for FM x FN MFMAs (the LDS traffic per
// MFMA of a large tile) although the tile is small, and a product with few rows can use many
// small tiles: the chip is filled by the number of tiles, not by their size.  The WK partial
// products meet in LDS after the K loop (int32: exact; floats: summed in wave order).
//
// K runs in stages of BKB bytes per row through a ring of STAGES LDS slots filled by
// buffer_load_dwordx4 ... lds (the ring of gemm_lds.hpp with its swizzles).  The fragments of
// stage kt + 1 are read while those of stage kt are multiplied, and stage kt + STAGES goes into
// the slot that stage kt has left, so STAGES - 1 stages are in flight.  Rows past the tile's valid
// rows, columns past N and K past its end lie outside the buffer resources: they read zeros and
// fetch nothing.
#pragma once

#include "gemm_lds.hpp"
#include "quad16.hpp"

namespace cb {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short v4i16 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ u32 pack_f16x2(const float a, const float b)
{
    return (u32)f32_to_f16(a) | ((u32)f32_to_f16(b) << 16);
}

// Rows of two accumulator slices (a: rows r .. r + 3, b: rows r + 8 .. r + 11 of the lane's column,
// already narrowed to 16 bits) to one 16-byte vector of 8 consecutive columns of one row: a quad
// transpose of each slice, then one exchange with lane c ^ 4 (ds_swizzle bit mode, xor mask 4,
// executed by every lane).  The lane keeps row r + qi when bit 2 of c is clear, row r + 8 + qi
// otherwise, and columns (c & ~7) .. + 7.
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4u slices_to_row8(const u32 a01, const u32 a23, const u32 b01, const u32 b23,
                                              const Quad16Sel& qs, const bool hi4)
{
    u32 x0, x1, z0, z1;
    quad_transpose16(a01, a23, qs, x0, x1);
    quad_transpose16(b01, b23, qs, z0, z1);
    const u32 s0 = hi4 ? x0 : z0, s1 = hi4 ? x1 : z1;
    const u32 r0 = (u32)__builtin_amdgcn_ds_swizzle((int)s0, 0x101F);
    const u32 r1 = (u32)__builtin_amdgcn_ds_swizzle((int)s1, 0x101F);
    return hi4 ? v4u{r0, r1, z0, z1} : v4u{x0, x1, r0, r1};
}

// ---- operand types ---------------------------------------------------------------------------
// Every type multiplies 32 bytes of K per MFMA step: v_mfma_i32_32x32x32_i8 or
// v_mfma_f32_32x32x16_{f16,bf16}, whose lane holds 16 consecutive K bytes of one row / column.
struct TileI8 {
    using Acc = v16i;
    static constexpr int ESZ = 1;
    __device__ static __forceinline__ Acc mma(const v4i a, const v4i b, const Acc c)
    {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
};
struct TileBF16 {
    using Acc = f32x16;
    static constexpr int ESZ = 2;
    __device__ static __forceinline__ Acc mma(const v4i a, const v4i b, const Acc c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
struct TileF16 {
    using Acc = f32x16;
    static constexpr int ESZ = 2;
    __device__ static __forceinline__ Acc mma(const v4i a, const v4i b, const Acc c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
};

// OP: operand type; BT: the weight is [N][K] (K contiguous).  FM x FN fragments per wave, WM x WN x
// WK waves, SK steps (32 bytes of K) per wave and stage, WGS workgroups resident per CU.
template <class OP_, bool BT_, int FM_, int FN_, int WM_, int WN_, int WK_, int SK_, int STAGES_, int WGS_>
struct TileCfg {
    using OP = OP_;
    static constexpr bool BT = BT_;
    static constexpr int FM = FM_, FN = FN_, WM = WM_, WN = WN_, WK = WK_, SK = SK_, STAGES = STAGES_, WGS = WGS_;
    static constexpr int NW = WM * WN * WK, NT = 64 * NW;
    static constexpr int BM = 32 * FM * WM, BN = 32 * FN * WN;
    static constexpr int BKB = 32 * WK * SK;         // bytes of K per row and stage
    static constexpr int BKE = BKB / OP::ESZ;        // elements of K per stage
    static constexpr int ACH = BKB / 16;             // 16-byte chunks per K-contiguous row
    static constexpr int BCH = BN * OP::ESZ / 16;    // 16-byte chunks per row of a [K][N] weight stage
    static constexpr int A_BYTES = BM * BKB, B_BYTES = BN * BKB, STAGE = A_BYTES + B_BYTES;
    static constexpr int A_ISSUE = A_BYTES / 16 / NT, B_ISSUE = B_BYTES / 16 / NT, ISSUE = A_ISSUE + B_ISSUE;
    static constexpr int RING = STAGES * STAGE;
    // partial products in LDS after the K loop: units of 8 accumulator registers (half a fragment,
    // 2 KB per wave), PU units of every fragment position per pass over the ring's memory
    static constexpr int UNITS = FM * FN * 2;
    static constexpr int UNIT_BYTES = 2048;
    static constexpr int PASS_MAX = RING / (NW * UNIT_BYTES);
    static constexpr int pass_units(int u) { return u <= PASS_MAX ? u : pass_units(u / 2); }
    static constexpr int PU = WK == 1 ? UNITS : pass_units(UNITS);
    static constexpr int SC = RING;                  // row scales [BM], then 3 column values [BN]
    static constexpr int LDS = RING + (BM + 3 * BN) * 4;
    static_assert(NW == 4 || NW == 8, "one or two waves per SIMD");
    static_assert(A_BYTES % (16 * NT) == 0 && B_BYTES % (16 * NT) == 0, "whole DMA chunks");
    static_assert(BKB == 64 || BKB == 128, "stage depth");
    static_assert(STAGES >= 3 && STAGES * ISSUE <= 63, "vmcnt counts at most 63");
    static_assert(WK == 1 || UNITS % PU == 0, "whole passes");
    static_assert(LDS <= 160 * 1024 / WGS, "LDS");
    static_assert(BM <= 256 && BN <= 256, "one thread per tile row and column loads the scales");
};

// Swizzle key of row k of a [K][N] weight stage (xor-ed into the 16-byte chunk position, even, so
// that chunk pairs stay together): int8, the 8 rows of a transposing read on distinct bank groups;
// 16-bit, its 4 rows.  Rows shorter than 256 bytes (BCH < 16) already differ in their bank half or
// quarter.
template <class C>
__device__ __forceinline__ int tile_bkey(const int k)
{
    if constexpr (C::OP::ESZ == 1) {
        return C::BCH >= 16 ? (k & 7) << 1 : (C::BCH == 8 ? ((k >> 1) & 3) << 1 : (C::BCH == 4 ? ((k >> 2) & 1) << 1 : 0));
    } else {
        return C::BCH >= 16 ? (k & 3) << 1 : (C::BCH == 8 ? ((k >> 1) & 1) << 1 : 0);
    }
}

// Tile number t: groups in order; within a group bands of 8 row tiles, column tile by column tile
// with the row tiles fastest, so consecutive tiles share a weight slab (few rows: neighbouring
// columns of the same weight rows).
struct TileAt {
    int g, m0, vrows, nt;
};

__device__ __forceinline__ TileAt tile_at(const GroupTable& gt, const int ntiles, const int bm, const int t)
{
    int lo = 0, hi = gt.n_groups - 1;
    while (lo < hi) {  // last g whose first tile is <= t (empty groups share it with the next)
        const int mid = (lo + hi + 1) >> 1;
        if (gt.tile_start[mid] * ntiles <= t) lo = mid;
        else hi = mid - 1;
    }
    TileAt r;
    r.g = lo;
    const int tm = gt.tile_start[lo + 1] - gt.tile_start[lo];
    const int local = t - gt.tile_start[lo] * ntiles;
    const int band = local / (8 * ntiles), rem = local - band * 8 * ntiles;
    const int rows = tm - band * 8 < 8 ? tm - band * 8 : 8;
    r.nt = rem / rows;
    const int mt = band * 8 + rem - r.nt * rows;
    const int r0 = lo ? gt.row_end[lo - 1] : 0;
    r.m0 = r0 + mt * bm;
    r.vrows = gt.row_end[lo] - r.m0;
    return r;
}

// Workgroup b (on XCD b % 8) takes a contiguous run of tiles per XCD: tiles sharing a weight slab,
// or the 128-byte lines of narrow column tiles, meet in one L2.
__device__ __forceinline__ int tile_xcd_order(const int b, const int total)
{
    const int x = b & 7, q = total >> 3, r = total & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// One BM x BN tile.  EPI: the epilogue (its Args, its prefetched values and its narrowing); see
// TileDeqEpi and GmmTileEpi.
template <class C, class EPI>
__global__ __launch_bounds__(C::NT, C::WGS * C::NW / 4) void tile_gemm_kernel(const typename EPI::Args a)
{
    using OP = typename C::OP;
    using Acc = typename OP::Acc;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % C::WK, wn = (wave / C::WK) % C::WN, wm = wave / (C::WK * C::WN);
    const TileAt t = tile_at(a.gt, a.ntiles, C::BM, tile_xcd_order((int)blockIdx.x, (int)gridDim.x));
    const int b = blockIdx.y;
    const int64_t K = a.K, N = a.N;
    const int n0 = t.nt * C::BN;
    const uint32_t kbytes = (uint32_t)(K * OP::ESZ), nbytes = (uint32_t)(N * OP::ESZ);
    const int vr = t.vrows < C::BM ? t.vrows : C::BM;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(CB_LDS uint8_t*)smem;

    const typename EPI::Pre pre = EPI::load(a, t, b, n0, vr, tid);  // used after the K loop

    // ---- DMA plan ------------------------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t ares =
        make_rsrc(EPI::x_base(a, b) + (int64_t)t.m0 * kbytes, (uint32_t)((int64_t)vr * kbytes));
    const uint8_t* wbase = EPI::w_base(a, t.g, b);
    const uint32_t wbytes = (uint32_t)(K * N * OP::ESZ);
    const __amdgpu_buffer_rsrc_t bres = make_rsrc(wbase, wbytes);
    uint32_t a_off[C::A_ISSUE], a_k[C::A_ISSUE], b_off[C::B_ISSUE], b_k[C::B_ISSUE];
#pragma unroll
    for (int i = 0; i < C::A_ISSUE; ++i) {
        const int cid = (i * C::NW + wave) * 64 + lane;
        const int row = cid / C::ACH, q = (cid % C::ACH) ^ a_swizzle<C::ACH>(row);
        a_k[i] = (uint32_t)(q * 16);
        a_off[i] = row < vr ? (uint32_t)row * kbytes + (uint32_t)(q * 16) : kOffNone;
    }
#pragma unroll
    for (int i = 0; i < C::B_ISSUE; ++i) {
        const int cid = (i * C::NW + wave) * 64 + lane;
        if constexpr (C::BT) {
            const int row = cid / C::ACH, q = (cid % C::ACH) ^ a_swizzle<C::ACH>(row);
            b_k[i] = (uint32_t)(q * 16);
            b_off[i] = n0 + row < N ? (uint32_t)(n0 + row) * kbytes + (uint32_t)(q * 16) : kOffNone;
        } else {
            const int row = cid / C::BCH, c = (cid % C::BCH) ^ tile_bkey<C>(row);
            const uint32_t col = (uint32_t)(n0 * OP::ESZ + c * 16);
            b_k[i] = (uint32_t)row * OP::ESZ;
            b_off[i] = col < nbytes ? (uint32_t)row * nbytes + col : kOffNone;
        }
    }
    const int nk = __builtin_amdgcn_readfirstlane((int)((K + C::BKE - 1) / C::BKE));
    // DMA chunk i of stage kt (activation chunks first)
    auto issue_one = [&](const int i, const int kt, const int slot) {
        const uint32_t sa = lds_base + (uint32_t)(slot * C::STAGE);
        const uint32_t kb = (uint32_t)(kt * C::BKB);
        if (i < C::A_ISSUE) {
            dma16(ares, kb + a_k[i] < kbytes ? a_off[i] + kb : kOffNone,
                  __builtin_amdgcn_readfirstlane(sa + (uint32_t)((i * C::NW + wave) * 1024)));
        } else {
            const int j = i - C::A_ISSUE;
            const uint32_t step = C::BT ? kb : (uint32_t)(kt * C::BKE) * nbytes;
            dma16(bres, kb + b_k[j] < kbytes ? b_off[j] + step : kOffNone,
                  __builtin_amdgcn_readfirstlane(sa + C::A_BYTES + (uint32_t)((j * C::NW + wave) * 1024)));
        }
    };
    auto issue = [&](const int kt, const int slot) {
#pragma unroll
        for (int i = 0; i < C::ISSUE; ++i) issue_one(i, kt, slot);
    };

    // ---- fragment reads ------------------------------------------------------------------------
    // K-contiguous rows: lane l takes row l % 32, 16-byte chunk 2 step + l / 32.  [K][N] weights: the
    // transposing reads (gemm_lds.hpp; 16-bit: in each 16-lane group, lane s addresses row s / 4,
    // columns 4 (s % 4) .. + 3, and lane j receives 4 consecutive K of column j).
    const int grp = lane >> 4, s = lane & 15;
    auto rd_row = [&](const CB_LDS uint8_t* base, const int row, const int step) -> v4i {
        const int q = 2 * step + (lane >> 5);
        return *(const CB_LDS v4i*)(base + row * C::BKB + ((q ^ a_swizzle<C::ACH>(row)) << 4));
    };
    auto rd = [&](const int slot, v4i (&af)[C::SK][C::FM], v4i (&bf)[C::SK][C::FN]) {
        const CB_LDS uint8_t* sa = (const CB_LDS uint8_t*)smem + slot * C::STAGE;
        const CB_LDS uint8_t* sb = sa + C::A_BYTES;
#pragma unroll
        for (int ks = 0; ks < C::SK; ++ks) {
            const int step = wk * C::SK + ks;
#pragma unroll
            for (int fn = 0; fn < C::FN; ++fn) {
                const int col0 = (wn * C::FN + fn) * 32;
                if constexpr (C::BT) {
                    bf[ks][fn] = rd_row(sb, col0 + (lane & 31), step);
                } else if constexpr (OP::ESZ == 1) {
                    const int k = step * 32 + (grp >> 1) * 16 + (s >> 1);
                    const int pos = ((col0 >> 4) + (grp & 1)) ^ tile_bkey<C>(k);  // the key of k + 8 too
                    const CB_LDS uint8_t* p = sb + k * C::BN + pos * 16 + (s & 1) * 8;
                    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((CB_LDS v2i*)p);
                    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((CB_LDS v2i*)(p + 8 * C::BN));
                    bf[ks][fn] = v4i{lo[0], lo[1], hi[0], hi[1]};
                } else {
                    const int k = step * 16 + 8 * (grp >> 1) + (s >> 2);
                    const int col = col0 + 16 * (grp & 1) + 4 * (s & 3);
                    const int pos = (col >> 3) ^ tile_bkey<C>(k);  // the key of k + 4 too
                    const CB_LDS uint8_t* p = sb + k * (C::BN * 2) + pos * 16 + (col & 7) * 2;
                    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((CB_LDS v4i16*)p);
                    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((CB_LDS v4i16*)(p + 4 * (C::BN * 2)));
                    const v2i l2 = __builtin_bit_cast(v2i, lo), h2 = __builtin_bit_cast(v2i, hi);
                    bf[ks][fn] = v4i{l2[0], l2[1], h2[0], h2[1]};
                }
            }
#pragma unroll
            for (int fm = 0; fm < C::FM; ++fm) af[ks][fm] = rd_row(sa, (wm * C::FM + fm) * 32 + (lane & 31), step);
        }
    };
    Acc acc[C::FM][C::FN];
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn) acc[fm][fn] = Acc{};
    // ---- K loop --------------------------------------------------------------------------------
#pragma unroll
    for (int st = 0; st < C::STAGES; ++st) issue(st, st);
    v4i a0[C::SK][C::FM], b0[C::SK][C::FN], a1[C::SK][C::FM], b1[C::SK][C::FN];
    wait_vmcnt_barrier<(C::STAGES - 1) * C::ISSUE>();
    rd(0, a0, b0);
    int slot = 0;  // of stage kt
    // multiplies stage kt (fragments in fa, fb) while stage kt + 1 is read and stage kt + STAGES issued
    auto body = [&](const int kt, v4i (&fa)[C::SK][C::FM], v4i (&fb)[C::SK][C::FN], v4i (&na)[C::SK][C::FM],
                    v4i (&nb)[C::SK][C::FN]) {
        wait_vmcnt_barrier<(C::STAGES - 2) * C::ISSUE>();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0) in the compiler's own accounting
        const int free_slot = slot;
        slot = slot + 1 == C::STAGES ? 0 : slot + 1;
        // two waves per SIMD: the other wave's MFMAs cover the DMA issue, so the reads go first
        // (128 x 256: 62 -> 60 us at 2048 x 7168 x 4096); one wave: the DMAs first (128 x 128: 38
        // against 39 us at 1024 rows)
        if constexpr (C::NW == 8) rd(slot, na, nb);
        issue(kt + C::STAGES, free_slot);
        if constexpr (C::NW == 4) rd(slot, na, nb);
#pragma unroll
        for (int ks = 0; ks < C::SK; ++ks)
#pragma unroll
            for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
                for (int fn = 0; fn < C::FN; ++fn) acc[fm][fn] = OP::mma(fa[ks][fm], fb[ks][fn], acc[fm][fn]);
    };
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        body(kt, a0, b0, a1, b1);
        body(kt + 1, a1, b1, a0, b0);
    }
    if (kt < nk) body(kt, a0, b0, a1, b1);

    // ---- epilogue ------------------------------------------------------------------------------
    epi_barrier();  // the ring is free, every DMA has landed
    CB_LDS float* sc = (CB_LDS float*)((CB_LDS uint8_t*)smem + C::SC);
    EPI::put(pre, sc, C::BM, C::BN, tid);
    const __amdgpu_buffer_rsrc_t ores = make_rsrc(EPI::out_base(a, b) + (int64_t)t.m0 * N, (uint32_t)((int64_t)vr * N * 2));
    const int h = lane >> 5, c = lane & 31, qi = c & 3;
    const bool hi4 = (c >> 2) & 1;
    const Quad16Sel qs = quad16_sel(qi);
    // half fragment u = (fm, fn, qp) of wave column / row (wm, wn): v[0..3] rows row0 + i, v[4..7]
    // rows row0 + 8 + i of column c (32x32 C layout: register r is row 8 (r / 4) + 4 h + r % 4)
    auto store_unit = [&](const int fr, const int fc, const int qp, const auto (&v)[8]) {
        const int row0 = fr * 32 + 16 * qp + 4 * h;
        u32 p[4];
        EPI::narrow(a, sc, C::BM, C::BN, row0, fc * 32 + c, v, p);
        const v4u w = slices_to_row8(p[0], p[1], p[2], p[3], qs, hi4);
        const int64_t c8 = (int64_t)n0 + fc * 32 + (c & ~7);
        const uint32_t roff = (uint32_t)(row0 + (hi4 ? 8 : 0) + qi) * (uint32_t)N * 2u;
        __builtin_amdgcn_raw_buffer_store_b128(w, ores, c8 < N ? roff + (uint32_t)c8 * 2u : kOffNone, 0, 0);
    };
    if constexpr (C::WK == 1) {
        __syncthreads();  // the scales
#pragma unroll
        for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < C::FN; ++fn)
#pragma unroll
                for (int qp = 0; qp < 2; ++qp) {
                    decltype(acc[0][0][0] + 0) v[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = acc[fm][fn][8 * qp + i];
                    store_unit(wm * C::FM + fm, wn * C::FN + fn, qp, v);
                }
    } else {
        // every wave writes its partial units (unit u: fragment u / 2, half u % 2), then each sums
        // and stores the units u = wk, wk + WK, ... of its (wm, wn) position
        CB_LDS uint8_t* part = (CB_LDS uint8_t*)smem;
#pragma unroll
        for (int p0 = 0; p0 < C::UNITS; p0 += C::PU) {
            if (p0) __syncthreads();  // the previous pass has been read
#pragma unroll
            for (int u = p0; u < p0 + C::PU; ++u) {
                CB_LDS uint8_t* d = part + (wave * C::PU + (u - p0)) * C::UNIT_BYTES + lane * 16;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    v4i w;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const auto x = acc[(u >> 1) / C::FN][(u >> 1) % C::FN][8 * (u & 1) + 4 * j + i];
                        w[i] = __builtin_bit_cast(int, x);
                    }
                    *(CB_LDS v4i*)(d + j * 1024) = w;
                }
            }
            __syncthreads();
            const int wbase = (wm * C::WN + wn) * C::WK;  // first wave of this position
            for (int u = p0 + wk; u < p0 + C::PU; u += C::WK) {
                decltype(acc[0][0][0] + 0) v[8] = {};
#pragma unroll
                for (int w = 0; w < C::WK; ++w) {
                    const CB_LDS uint8_t* d = part + ((wbase + w) * C::PU + (u - p0)) * C::UNIT_BYTES + lane * 16;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const v4i r = *(const CB_LDS v4i*)(d + j * 1024);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const auto x = __builtin_bit_cast(decltype(acc[0][0][0] + 0), (int)r[i]);
                            v[4 * j + i] = w == 0 ? x : v[4 * j + i] + x;
                        }
                    }
                }
                const int f = u >> 1;
                store_unit(wm * C::FM + f / C::FN, wn * C::FN + f % C::FN, u & 1, v);
            }
        }
    }
}

// ---- epilogues -------------------------------------------------------------------------------
// The QuantMatmul dequant chain (apply_deq of gemm_i8.hpp) to bf16 / fp16.  SIMPLE: column scale,
// optional per-token scale, bf16 out, without the selects of the other variants.
template <bool SIMPLE>
struct TileDeqEpi {
    using Args = GemmArgs;
    struct Pre {
        float xs;
        ColDeq cd;
    };
    __device__ static __forceinline__ const uint8_t* x_base(const Args& a, const int b)
    {
        return (const uint8_t*)a.x + (int64_t)b * a.x_bstride;
    }
    __device__ static __forceinline__ const uint8_t* w_base(const Args& a, const int g, const int b)
    {
        return (const uint8_t*)a.w + (int64_t)b * a.w_bstride + (int64_t)g * a.w_gstride;
    }
    __device__ static __forceinline__ uint16_t* out_base(const Args& a, const int b)
    {
        return (uint16_t*)a.epi.out + (int64_t)b * a.epi.out_bstride;
    }
    // thread tid: the scale of tile row tid and the dequant values of tile column tid (rows and
    // columns past the tile's valid ones repeat its last)
    __device__ static __forceinline__ Pre load(const Args& a, const TileAt& t, const int b, const int n0, const int vr,
                                               const int tid)
    {
        Pre p;
        const EpiArgs& e = a.epi;
        p.xs = e.has_pt ? e.pertoken[t.m0 + (tid < vr ? tid : vr - 1)] : 1.0f;
        const int64_t col = (int64_t)n0 + tid < a.N ? (int64_t)n0 + tid : a.N - 1;
        if constexpr (SIMPLE) {
            const int64_t si = (int64_t)t.g * e.scale_gstride + (e.scale_perchan ? col : 0);
            p.cd = ColDeq{e.scale_bf16 ? bf16_to_f32(((const uint16_t*)e.scale)[si]) : ((const float*)e.scale)[si], 0.0f, 0.0f};
        } else {
            p.cd = col_deq(e, t.g, b, col);
        }
        return p;
    }
    __device__ static __forceinline__ void put(const Pre& p, CB_LDS float* sc, const int bm, const int bn, const int tid)
    {
        if (tid < bm) sc[tid] = p.xs;
        if (tid < bn) {
            sc[bm + tid] = p.cd.scale;
            if constexpr (!SIMPLE) {
                sc[bm + bn + tid] = p.cd.offset;
                sc[bm + 2 * bn + tid] = p.cd.bias;
            }
        }
    }
    __device__ static __forceinline__ void narrow(const Args& a, const CB_LDS float* sc, const int bm, const int bn,
                                                  const int row0, const int col, const int (&v)[8], u32 (&p)[4])
    {
        const EpiArgs& e = a.epi;
        ColDeq cd{sc[bm + col], 0.0f, 0.0f};
        if constexpr (!SIMPLE) {
            cd.offset = sc[bm + bn + col];
            cd.bias = sc[bm + 2 * bn + col];
        }
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float pt = sc[row0 + (i & 3) + 2 * (i & 4)];
            if constexpr (SIMPLE) f[i] = ((float)v[i] * cd.scale) * pt;
            else f[i] = apply_deq(e, cd, v[i], pt);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            p[i] = SIMPLE || e.out_bf16 ? pack_bf16x2(f[2 * i], f[2 * i + 1]) : pack_f16x2(f[2 * i], f[2 * i + 1]);
    }
};

}  // namespace cb
