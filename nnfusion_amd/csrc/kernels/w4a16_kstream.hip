// The K-streaming kernel for groups of 128 with a scalar zero point (w4a16_kstream.h).
#include "w4a16_kstream.h"

namespace nnf
{
    hipError_t launch_w4a16_kstream(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* Wq, const void* S,
                                    void* Y, int M, int N, int K, int zp, const GemvFusion& fusion, float* partial, uint32_t* sync)
    {
        return launch_w4a16_kstream_g<0>(stream, plan, A, Wq, S, Y, M, N, K, zp, fusion, partial, sync, nullptr);
    }
} // namespace nnf
