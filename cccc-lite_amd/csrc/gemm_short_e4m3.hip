#include "gemm_short.h"

namespace ccq
{

void launch_gemm_short_e4m3(const LinearArgs& a, bool half, bool tiled, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    launch_short_type<DT_E4M3>(a, half, tiled, pair, p, partial, e);
}

}    // namespace ccq
