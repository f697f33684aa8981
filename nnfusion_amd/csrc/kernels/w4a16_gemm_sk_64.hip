// fp16 x int4 tile GEMM, tiles of 64 x 256: the instantiations of w4a16_gemm_sk.h for this tile height.
#include "w4a16_gemm_sk_launch.h"

namespace nnf
{
    hipError_t launch_gemm_sk_64(hipStream_t stream, const SkGemmParams& p, int grid, bool gate, bool eight)
    {
        return eight ? gemm_sk::launch_tile_height<gemm_sk::TileOf<64, 256, true>>(stream, p, grid, gate)
                     : gemm_sk::launch_tile_height<gemm_sk::TileOf<64, 256>>(stream, p, grid, gate);
    }
} // namespace nnf
