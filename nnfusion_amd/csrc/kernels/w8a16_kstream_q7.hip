// The K-streaming kernel for 8-bit weights in groups of 128, a scalar zero point or one per (row, group) (w4a16_kstream.h).
#include "w4a16_kstream.h"

namespace nnf
{
    hipError_t launch_w8a16_kstream_q7(hipStream_t stream, const workspace::KstreamPlan& plan, const void* A, const void* Wq, const void* S,
                                       void* Y, int M, int N, int K, int zp, const void* zero_points, const GemvFusion& fusion)
    {
        return launch_w4a16_kstream_g<7, 8>(stream, plan, A, Wq, S, Y, M, N, K, zp, fusion, nullptr, nullptr, zero_points);
    }
} // namespace nnf
