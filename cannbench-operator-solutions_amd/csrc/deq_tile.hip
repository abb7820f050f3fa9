// deq_tile.hip - the tiles of gemm_tile.hpp with the int8 dequant epilogue (QuantMatmul and the grouped
// down-projection); moe_ops.hip chooses among them.  A translation unit of its own: compiled next to
// the ring core's kernels, these changed the register allocation of gpf_dequant_kernel's epilogue
// (1.6 us of 103 at 4096 x 7168 x 4096).
#include "gemm_tile.hpp"

namespace cb {

// Tiles of gemm_tile.hpp.
using DeqT0 = TileCfg<TileI8, false, 1, 2, 1, 1, 4, 1, 6, 2>;  // 32 x 64
using DeqT1 = TileCfg<TileI8, false, 2, 4, 1, 1, 4, 1, 3, 2>;  // 64 x 128
using DeqT2 = TileCfg<TileI8, false, 2, 4, 1, 2, 2, 1, 3, 2>;  // 64 x 256
using DeqT3 = TileCfg<TileI8, false, 2, 4, 2, 1, 4, 1, 4, 1>;  // 128 x 128, 8 waves
using DeqT4 = TileCfg<TileI8, false, 2, 4, 2, 2, 2, 1, 6, 1>;  // 128 x 256, 8 waves

template <class C>
static void launch_tile(GemmArgs& a, const int64_t* gl, int64_t E, int64_t batch, hipStream_t st)
{
    build_group_table(a.gt, gl, E, C::BM);
    a.ntiles = (int)((a.N + C::BN - 1) / C::BN);
    const EpiArgs& e = a.epi;
    const bool simple = !e.has_offset && e.bias_kind == BIAS_NONE && e.out_bf16;
    const dim3 grid((unsigned)(a.gt.total_mtiles * a.ntiles), (unsigned)batch);
    auto go = [&](auto kern) {
        set_dynamic_lds_once((const void*)kern, C::LDS);
        hipLaunchKernelGGL(kern, grid, dim3(C::NT), C::LDS, st, a);
    };
    if (simple) go(tile_gemm_kernel<C, TileDeqEpi<true>>);
    else go(tile_gemm_kernel<C, TileDeqEpi<false>>);
}

bool launch_deq_tile(int tile, GemmArgs& a, const int64_t* gl, int64_t E, int64_t batch, hipStream_t st)
{
    switch (tile) {
        case 0: launch_tile<DeqT0>(a, gl, E, batch, st); return true;
        case 1: launch_tile<DeqT1>(a, gl, E, batch, st); return true;
        case 2: launch_tile<DeqT2>(a, gl, E, batch, st); return true;
        case 3: launch_tile<DeqT3>(a, gl, E, batch, st); return true;
        case 4: launch_tile<DeqT4>(a, gl, E, batch, st); return true;
        default: return false;
    }
}

}  // namespace cb
