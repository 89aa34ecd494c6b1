#include "gemm_staged.h"

namespace ccq
{

void launch_gemm_staged_e5m2(const LinearArgs& a, bool half, bool tiled, bool scaled, const GemmPlan& p, int n_tiles, float* partial)
{
    launch_staged_type<DT_E5M2>(a, half, tiled, scaled, p, n_tiles, partial);
}

}    // namespace ccq
