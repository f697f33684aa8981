// fp16 x int4 tile GEMM, tiles of 128 x 192 (whole tiles, even multiples of 128 along K): the instantiations of w4a16_gemm_sk.h.
#include "w4a16_gemm_sk_launch.h"

namespace nnf
{
    hipError_t launch_gemm_sk_192(hipStream_t stream, const SkGemmParams& p, int grid, bool gate)
    {
        return gemm_sk::launch_tile_height<gemm_sk::TileOf<128, 192>>(stream, p, grid, gate);
    }
} // namespace nnf
