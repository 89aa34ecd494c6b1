#include "gemm_short.h"

namespace ccq
{

void launch_gemm_short_e5m2(const LinearArgs& a, bool half, bool tiled, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    launch_short_type<DT_E5M2>(a, half, tiled, pair, p, partial, e);
}

void launch_gemm_short(const LinearArgs& a, int w_type, bool half, bool tiled, bool pair, const GemmPlan& plan, float* partial, const AddNormArgs* e)
{
    (w_type == DT_E5M2 ? launch_gemm_short_e5m2 : launch_gemm_short_e4m3)(a, half, tiled, pair, plan, partial, e);
}

}    // namespace ccq
