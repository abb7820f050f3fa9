// gmm_float.hip - GroupedMatmul, the reference's float grouped GEMM (C ABI cb_grouped_matmul):
//   y[rows_g] = x[rows_g] @ weight[g] (+ bias[g]),  rows_g = [group_list[g-1], group_list[g])
// in the dtype of x (fp16, bf16 or fp32), weight [E, K, N] or, with transpose_weight, [E, N, K]
// (operators/groupedmatmul/csrc/ops/grouped_matmul/op_plugin/grouped_matmul_plugin.cpp:14-17,
// 116-183; op_kernel/grouped_matmul_kernel.cpp:15-17, 111-150).
//
// 16-bit inputs run on v_mfma_f32_32x32x16_{f16,bf16} through the tiles of gemm_tile.hpp (32 x 64 to
// 256 x 256, chosen by pick_gmm), fp32 accumulation, the bias added in fp32, one
// round-to-nearest-even narrowing.  Rows or outputs past 32-bit offsets and outputs off 16-byte
// alignment take a 128 x 128 register-staged kernel.  fp32 inputs and shapes off the vector path
// (K or N not a multiple of 8, misaligned operands, 32-bit offsets exceeded) take a plain fp32 loop.
#include <cstdlib>
#include <cstring>

#include "gemm_tile.hpp"

namespace cb {

constexpr int kGmmMaxExperts = 64;  // GMM_MAX_E (grouped_matmul_launch.h)
constexpr int GF_BK = 32;
// elements per LDS row (BK + 8: 80 B at BK 32): a 16-lane b128 read phase hits 16 distinct bank groups
constexpr int GF_PITCH = GF_BK + 8;
constexpr int GF_KCH = GF_BK / 8;  // 16-byte chunks per row and stage

struct GmmFArgs {
    const void* x;
    const void* w;
    const void* bias;
    void* y;
    int64_t M, K, N;
    int32_t x_dt, bias_dt;  // cb_dtype codes; bias_dt 0 = no bias
    int32_t trans, ntiles;
    GroupTable gt;
};

__device__ __forceinline__ float gf_load(const void* p, int dt, int64_t i)
{
    if (dt == CB_DT_FLOAT32) return ((const float*)p)[i];
    if (dt == CB_DT_BFLOAT16) return bf16_to_f32(((const uint16_t*)p)[i]);
    return f16_to_f32(((const uint16_t*)p)[i]);
}

__device__ __forceinline__ void gf_store(void* p, int dt, int64_t i, float v)
{
    if (dt == CB_DT_FLOAT32) ((float*)p)[i] = v;
    else if (dt == CB_DT_BFLOAT16) ((uint16_t*)p)[i] = f32_to_bf16_hw(v);
    else ((uint16_t*)p)[i] = f32_to_f16(v);
}

// One BM x BN tile per workgroup of WM x WN waves (wave tiles (BM / WM) x (BN / WN)): pid -> (row
// tile, column tile) with 4 row tiles per column sweep.  Launched as 128 x 128 with 2 x 2 waves.
template <bool BF16, bool TRANS, int GF_BM, int GF_BN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 64 * WM * WN > 256 ? 1 : 2) void gmm_mfma_kernel(const GmmFArgs a)
{
    constexpr int NT = 64 * WM * WN;
    constexpr int TM = GF_BM / WM, TN = GF_BN / WN, FM = TM / 32, FN = TN / 32;
    constexpr int GF_CA = GF_BM * GF_KCH / NT;             // A chunks per thread
    constexpr int GF_CB = GF_BN * GF_KCH / NT;             // [N][K] weight chunks per thread
    constexpr int GF_CP = (GF_BK / 2) * (GF_BN / 8) / NT;  // [K][N] weight: (k, k + 1) chunk pairs per thread
    constexpr int NCH = GF_BN / 8;                         // 8-column chunks per weight row
    static_assert(GF_CA >= 1 && GF_CB >= 1 && GF_CP >= 1, "tile too small for the workgroup");
    __shared__ __attribute__((aligned(16))) uint16_t As[2][GF_BM * GF_PITCH];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][GF_BN * GF_PITCH];  // [n][k]

    constexpr int GROUP_M = 4;
    const int pid = blockIdx.x;
    const int T_m = a.gt.total_mtiles, T_n = a.ntiles;
    const int per_group = GROUP_M * T_n;
    const int first_m = (pid / per_group) * GROUP_M;
    const int gsz = (T_m - first_m) < GROUP_M ? (T_m - first_m) : GROUP_M;
    const int mt = first_m + (pid % per_group) % gsz;
    const int nt = (pid % per_group) / gsz;

    const int g = group_of_tile(a.gt, mt);
    const int rs = g ? a.gt.row_end[g - 1] : 0;
    const int r1 = a.gt.row_end[g];
    const int m0 = rs + (mt - a.gt.tile_start[g]) * GF_BM;
    const int vrows = r1 - m0;
    const int n0 = nt * GF_BN;
    const int64_t K = a.K, N = a.N;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;

    // Operand streams through buffer resources (offsets outside a resource read zeros).
    // A: rows [m0, r1) of x; thread chunks c = tid + 256 i: row c / KCH, k chunk c % KCH (8 elements).
    const __amdgpu_buffer_rsrc_t ares = make_rsrc((const uint16_t*)a.x + (int64_t)m0 * K,
                                                     (uint32_t)((vrows < GF_BM ? vrows : GF_BM) * K * 2));
    const __amdgpu_buffer_rsrc_t bres = make_rsrc((const uint16_t*)a.w + (int64_t)g * K * N, (uint32_t)(K * N * 2));
    uint32_t aoff[GF_CA], boff[GF_CB];
    int arow[GF_CA], akc[GF_CA], brow[GF_CB], bkc[GF_CB];
#pragma unroll
    for (int i = 0; i < GF_CA; ++i) {
        const int c = tid + NT * i;
        arow[i] = c / GF_KCH;
        akc[i] = c % GF_KCH;
        aoff[i] = arow[i] < vrows ? (uint32_t)((arow[i] * K + akc[i] * 8) * 2) : 0x80000000u;
    }
#pragma unroll
    for (int i = 0; i < GF_CB; ++i) {
        // weight [N][K]: like A, rows are output columns
        const int c = tid + NT * i;
        brow[i] = c / GF_KCH;
        bkc[i] = c % GF_KCH;
        const int n = n0 + brow[i];
        boff[i] = n < N ? (uint32_t)((n * K + bkc[i] * 8) * 2) : 0x80000000u;
    }
    // weight [K][N]: pair p = tid + NT i takes k rows 2 (p / NCH) and + 1 of n chunk p % NCH
    int bkp[GF_CP], bnc[GF_CP];
    bool bn_ok[GF_CP];
#pragma unroll
    for (int i = 0; i < GF_CP; ++i) {
        const int p2 = tid + NT * i;
        bkp[i] = p2 / NCH;
        bnc[i] = p2 % NCH;
        bn_ok[i] = n0 + bnc[i] * 8 < N;
    }
    const int nk = (int)((K + GF_BK - 1) / GF_BK);

    uint4 ra[GF_CA], rb[TRANS ? GF_CB : 2 * GF_CP];
    auto ld16 = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
        const v4i v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
        return make_uint4((u32)v[0], (u32)v[1], (u32)v[2], (u32)v[3]);
    };
    auto load_stage = [&](int kt) {
        const int k0 = kt * GF_BK;
#pragma unroll
        for (int i = 0; i < GF_CA; ++i)
            ra[i] = ld16(ares, k0 + akc[i] * 8 < K ? aoff[i] + (uint32_t)(k0 * 2) : 0x80000000u);
        if constexpr (TRANS) {
#pragma unroll
            for (int i = 0; i < GF_CB; ++i)
                rb[i] = ld16(bres, k0 + bkc[i] * 8 < K ? boff[i] + (uint32_t)(k0 * 2) : 0x80000000u);
        } else {
#pragma unroll
            for (int i = 0; i < GF_CP; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int k = k0 + 2 * bkp[i] + h;
                    rb[2 * i + h] = ld16(bres, k < K && bn_ok[i] ? (uint32_t)((k * N + n0 + bnc[i] * 8) * 2) : 0x80000000u);
                }
        }
    };
    auto store_stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < GF_CA; ++i)
            *reinterpret_cast<uint4*>(&As[buf][arow[i] * GF_PITCH + akc[i] * 8]) = ra[i];
        if constexpr (TRANS) {
#pragma unroll
            for (int i = 0; i < GF_CB; ++i)
                *reinterpret_cast<uint4*>(&Bs[buf][brow[i] * GF_PITCH + bkc[i] * 8]) = rb[i];
        } else {
            // 8 columns x 2 consecutive k: one 32-bit (k, k + 1) pair per column
#pragma unroll
            for (int i = 0; i < GF_CP; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const u32 lo = comp(rb[2 * i], j >> 1), hi = comp(rb[2 * i + 1], j >> 1);
                    const u32 pair = (j & 1) ? ((lo >> 16) | (hi & 0xffff0000u)) : ((lo & 0xffffu) | (hi << 16));
                    *reinterpret_cast<u32*>(&Bs[buf][(bnc[i] * 8 + j) * GF_PITCH + 2 * bkp[i]]) = pair;
                }
        }
    };

    f32x16 acc[FM][FN];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[fm][fn][r] = 0.0f;

    load_stage(0);
    store_stage(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) load_stage(kt + 1);  // in flight during this stage's MFMAs
#pragma unroll
        for (int kk = 0; kk < GF_BK / 16; ++kk) {
            // 32x32x16 operands: lane l holds row / column l % 32, k 8 (l / 32) .. + 7
            uint4 af[FM], bf[FN];
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
                af[fm] = *reinterpret_cast<const uint4*>(
                    &As[buf][(wm * TM + fm * 32 + (lane & 31)) * GF_PITCH + kk * 16 + (lane >> 5) * 8]);
#pragma unroll
            for (int fn = 0; fn < FN; ++fn)
                bf[fn] = *reinterpret_cast<const uint4*>(
                    &Bs[buf][(wn * TN + fn * 32 + (lane & 31)) * GF_PITCH + kk * 16 + (lane >> 5) * 8]);
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) {
                    if constexpr (BF16)
                        acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, af[fm]), __builtin_bit_cast(bf16x8, bf[fn]), acc[fm][fn], 0, 0, 0);
                    else
                        acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(f16x8, af[fm]), __builtin_bit_cast(f16x8, bf[fn]), acc[fm][fn], 0, 0, 0);
                }
        }
        if (kt + 1 < nk) store_stage(buf ^ 1);  // the other buffer was last read one stage ago
        __syncthreads();
    }

    // Epilogue.  32x32 C layout: lane l holds column l % 32, rows 8 (r / 4) + 4 (l / 32) + r % 4.
    uint16_t* y = (uint16_t*)a.y;
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
        const int64_t col = n0 + wn * TN + fn * 32 + (lane & 31);
        if (col >= N) continue;
        const float bv = a.bias_dt ? gf_load(a.bias, a.bias_dt, (int64_t)g * N + col) : 0.0f;
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int lrow = wm * TM + fm * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (lrow < vrows) {
                    const float v = acc[fm][fn][r] + bv;
                    y[(int64_t)(m0 + lrow) * N + col] = BF16 ? f32_to_bf16_hw(v) : f32_to_f16(v);
                }
            }
    }
}

// Epilogue of the tiled GEMM (gemm_tile.hpp): the bias added in fp32, one narrowing.
template <bool BF16>
struct GmmTileEpi {
    using Args = GmmFArgs;
    struct Pre {
        float bias;
    };
    __device__ static __forceinline__ const uint8_t* x_base(const Args& a, const int) { return (const uint8_t*)a.x; }
    __device__ static __forceinline__ const uint8_t* w_base(const Args& a, const int g, const int)
    {
        return (const uint8_t*)a.w + (int64_t)g * a.K * a.N * 2;
    }
    __device__ static __forceinline__ uint16_t* out_base(const Args& a, const int) { return (uint16_t*)a.y; }
    // thread tid: the bias of tile column tid (columns past N repeat the last)
    __device__ static __forceinline__ Pre load(const Args& a, const TileAt& t, const int, const int n0, const int, const int tid)
    {
        const int64_t col = (int64_t)n0 + tid < a.N ? (int64_t)n0 + tid : a.N - 1;
        return Pre{a.bias_dt ? gf_load(a.bias, a.bias_dt, (int64_t)t.g * a.N + col) : 0.0f};
    }
    __device__ static __forceinline__ void put(const Pre& p, CB_LDS float* sc, const int bm, const int bn, const int tid)
    {
        if (tid < bn) sc[bm + tid] = p.bias;
    }
    __device__ static __forceinline__ void narrow(const Args&, const CB_LDS float* sc, const int bm, const int, const int,
                                                  const int col, const float (&v)[8], u32 (&p)[4])
    {
        const float b = sc[bm + col];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            p[i] = BF16 ? pack_bf16x2(v[2 * i] + b, v[2 * i + 1] + b) : pack_f16x2(v[2 * i] + b, v[2 * i + 1] + b);
    }
};

// Any dtype and layout: one output element per thread iteration (grid-stride), fp32 accumulation
// in k order, the bias added in fp32, one narrowing to the output dtype.
__global__ __launch_bounds__(256) void gmm_generic_kernel(const GmmFArgs a)
{
    const int64_t total = a.M * a.N;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int row = (int)(i / a.N);
        const int64_t col = i % a.N;
        const int g = group_of_row(a.gt, row);
        const int64_t wb = (int64_t)g * a.K * a.N;
        float acc = 0.0f;
        for (int64_t k = 0; k < a.K; ++k) {
            const float xv = gf_load(a.x, a.x_dt, (int64_t)row * a.K + k);
            const float wv = gf_load(a.w, a.x_dt, wb + (a.trans ? col * a.K + k : k * a.N + col));
            acc = acc + xv * wv;
        }
        if (a.bias_dt) acc = acc + gf_load(a.bias, a.bias_dt, (int64_t)g * a.N + col);
        gf_store(a.y, a.x_dt, i, acc);
    }
}

template <template <class, bool> class Cfg>
static void launch_gmm_tile(GmmFArgs& a, const int64_t* gl, int64_t E, hipStream_t st)
{
    using C0 = Cfg<TileBF16, false>;
    build_group_table(a.gt, gl, E, C0::BM);
    a.ntiles = (int)((a.N + C0::BN - 1) / C0::BN);
    const dim3 grid((unsigned)(a.gt.total_mtiles * a.ntiles));
    auto go = [&](auto cfg, auto epi) {
        using C = decltype(cfg);
        auto kern = tile_gemm_kernel<C, decltype(epi)>;
        set_dynamic_lds_once((const void*)kern, C::LDS);
        hipLaunchKernelGGL(kern, grid, dim3(C::NT), C::LDS, st, a);
    };
    const bool bf = a.x_dt == CB_DT_BFLOAT16;
    if (bf && a.trans) go(Cfg<TileBF16, true>{}, GmmTileEpi<true>{});
    else if (bf) go(Cfg<TileBF16, false>{}, GmmTileEpi<true>{});
    else if (a.trans) go(Cfg<TileF16, true>{}, GmmTileEpi<false>{});
    else go(Cfg<TileF16, false>{}, GmmTileEpi<false>{});
}

template <class OP, bool BT> using GmmT0 = TileCfg<OP, BT, 1, 2, 1, 1, 4, 1, 6, 2>;  // 32 x 64
template <class OP, bool BT> using GmmT1 = TileCfg<OP, BT, 2, 4, 1, 1, 4, 1, 3, 2>;  // 64 x 128
template <class OP, bool BT> using GmmT2 = TileCfg<OP, BT, 2, 4, 1, 2, 2, 1, 3, 2>;  // 64 x 256
template <class OP, bool BT> using GmmT3 = TileCfg<OP, BT, 2, 4, 2, 1, 4, 1, 4, 1>;  // 128 x 128, 8 waves
template <class OP, bool BT> using GmmT4 = TileCfg<OP, BT, 2, 4, 2, 2, 2, 2, 3, 1>;  // 128 x 256, 8 waves
template <class OP, bool BT> using GmmT5 = TileCfg<OP, BT, 2, 4, 4, 2, 1, 2, 4, 1>;  // 256 x 256, 8 waves

}  // namespace cb

using namespace cb;

// The reference's launch_gmm (grouped_matmul_launch.h:66-70) with the plugin's checks
// (grouped_matmul_plugin.cpp:127-157, in order) moved behind a status return.  K = 0 writes the
// bias (or zeros).
extern "C" int cb_grouped_matmul(const void* x, const void* weight, const void* bias, int x_dtype, int bias_dtype,
                                 const int64_t* group_list, int64_t group_len, int64_t M, int64_t K, int64_t N,
                                 int64_t E, int transpose_weight, void* y, void* stream)
{
    if (M < 0 || K < 0 || N < 0 || E < 0) return CB_ERR_SHAPE;
    if (E < 1 || E > kGmmMaxExperts) return CB_ERR_GROUP_COUNT;  // plugin :138-139
    if (x_dtype != CB_DT_FLOAT16 && x_dtype != CB_DT_BFLOAT16 && x_dtype != CB_DT_FLOAT32) return CB_ERR_DTYPE;
    if (bias && bias_dtype != CB_DT_FLOAT16 && bias_dtype != CB_DT_BFLOAT16 && bias_dtype != CB_DT_FLOAT32)
        return CB_ERR_DTYPE;
    const int vs = validate_group_list(group_list, group_len, E, M);
    if (vs != CB_OK) return vs;
    if (M == 0 || N == 0) return CB_OK;
    if (!x && K > 0) return CB_ERR_NULL_POINTER;
    if ((!weight && K > 0) || !y) return CB_ERR_NULL_POINTER;
    if (M > 0x7fffffffLL) return CB_ERR_SHAPE;

    GmmFArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = x;
    a.w = weight;
    a.bias = bias;
    a.y = y;
    a.M = M;
    a.K = K;
    a.N = N;
    a.x_dt = x_dtype;
    a.bias_dt = bias ? bias_dtype : 0;
    a.trans = transpose_weight ? 1 : 0;
    hipStream_t st = (hipStream_t)stream;
    TimedLaunch timed(st);

    const bool mfma = x_dtype != CB_DT_FLOAT32 && K > 0 && K % 8 == 0 && N % 8 == 0 && aligned(x, 16) &&
                      aligned(weight, 16) && K * N * 2 < (1LL << 31) && 128 * K * 2 < (1LL << 31);
    if (mfma) {
        // a test override of 128 selects the 128 x 128 register-staged kernel for every shape (it is
        // otherwise taken only where a 256-row block of x or y passes 2 GiB or y is not 16-byte
        // aligned: it stores single values)
        const int tile = g_overrides.gmm_tile;
        int pick = -1;
        if (tile != 128 && 256 * K * 2 < (1LL << 31) && 256 * N * 2 < (1LL << 31) && aligned(y, 16))  // 16-byte stores
            pick = tile >= 1 && tile <= 6 ? tile - 1 : pick_gmm(group_list, E, M, K, N, rule_cus());
        switch (pick) {
            case 0: launch_gmm_tile<GmmT0>(a, group_list, E, st); return check_launch();
            case 1: launch_gmm_tile<GmmT1>(a, group_list, E, st); return check_launch();
            case 2: launch_gmm_tile<GmmT2>(a, group_list, E, st); return check_launch();
            case 3: launch_gmm_tile<GmmT3>(a, group_list, E, st); return check_launch();
            case 4: launch_gmm_tile<GmmT4>(a, group_list, E, st); return check_launch();
            case 5: launch_gmm_tile<GmmT5>(a, group_list, E, st); return check_launch();
            default: break;
        }
        build_group_table(a.gt, group_list, E, 128);
        a.ntiles = (int)((N + 127) / 128);
        const int64_t blocks = (int64_t)a.gt.total_mtiles * a.ntiles;
        if (blocks <= 0) return CB_OK;
        const dim3 grid((unsigned)blocks);
        const bool bf = x_dtype == CB_DT_BFLOAT16;
        if (bf && a.trans) hipLaunchKernelGGL((gmm_mfma_kernel<true, true, 128, 128, 2, 2>), grid, dim3(256), 0, st, a);
        else if (bf) hipLaunchKernelGGL((gmm_mfma_kernel<true, false, 128, 128, 2, 2>), grid, dim3(256), 0, st, a);
        else if (a.trans) hipLaunchKernelGGL((gmm_mfma_kernel<false, true, 128, 128, 2, 2>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((gmm_mfma_kernel<false, false, 128, 128, 2, 2>), grid, dim3(256), 0, st, a);
        return check_launch();
    }
    build_group_table(a.gt, group_list, E, 1);
    const int64_t total = M * N;
    const int64_t blocks = (total + 255) / 256;
    hipLaunchKernelGGL(gmm_generic_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0, st, a);
    return check_launch();
}
