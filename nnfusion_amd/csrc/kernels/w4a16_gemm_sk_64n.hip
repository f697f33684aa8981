// fp16 x int4 tile GEMM, tiles of 64 x 128 (one column tile per wavefront; four wavefronts or eight): the instantiations of w4a16_gemm_sk.h.
#include "w4a16_gemm_sk_launch.h"

namespace nnf
{
    hipError_t launch_gemm_sk_64_narrow(hipStream_t stream, const SkGemmParams& p, int grid, bool eight)
    {
        return eight ? gemm_sk::launch_tile_height_plain<gemm_sk::TileOf<64, 128, true>>(stream, p, grid)
                     : gemm_sk::launch_tile_height_plain<gemm_sk::TileOf<64, 128>>(stream, p, grid);
    }
} // namespace nnf
