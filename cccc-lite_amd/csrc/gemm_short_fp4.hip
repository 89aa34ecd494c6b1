// The small tiles of plan_gemm (gemm_plan.h) on the register-fed FP4 GEMM.
#include "gemm_kernels.h"
#include "prefill_kernels.h"

namespace ccq
{

namespace
{

template <int BLOCK, int MB, int NB, bool PAIR, bool SEG>
void launch_tile(const LinearArgs& a, const uint8_t* scales, int n_tiles, int splits, float* partial)
{
    const dim3 grid(((n_tiles + 7) & ~7) * ((a.tokens + MB * 16 - 1) / (MB * 16)), splits);
    if (splits > 1) { gemm4_mfma_direct_kernel<BLOCK, MB, true, NB, SEG, PAIR><<<grid, 256, 0, stream()>>>(a, scales, n_tiles, partial); }
    else { gemm4_mfma_direct_kernel<BLOCK, MB, false, NB, SEG, PAIR><<<grid, 256, 0, stream()>>>(a, scales, n_tiles, nullptr); }
}

template <int BLOCK, bool PAIR, bool SEG>
void launch_shape(LinearArgs a, const uint8_t* scales, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    const int width = 64 * (PAIR ? p.nb / 2 : p.nb);
    if (e && p.splits <= 1)
    {
        a.Y = (uint16_t*)partial;
        a.y_stride_tok = a.n_out;
    }
    int n_tiles = (a.n_out + width - 1) / width;
    long long features = a.n_out;
    if constexpr (SEG)
    {
        n_tiles = 0;
        features = 0;
        for (int s = 0; s < 3; s++)
        {
            a.seg_tile0[s] = n_tiles;
            if (s < a.n_segments)
            {
                n_tiles += (a.seg_n_out[s] + width - 1) / width;
                features += a.seg_n_out[s];
            }
        }
        a.seg_tile0[3] = n_tiles;
    }
    if constexpr (!PAIR)
    {
        if (p.mb == 2 && p.nb == 1) { launch_tile<BLOCK, 2, 1, PAIR, SEG>(a, scales, n_tiles, p.splits, partial); }
        if (p.mb == 4 && p.nb == 1) { launch_tile<BLOCK, 4, 1, PAIR, SEG>(a, scales, n_tiles, p.splits, partial); }
    }
    if (p.mb == 2 && p.nb == 2) { launch_tile<BLOCK, 2, 2, PAIR, SEG>(a, scales, n_tiles, p.splits, partial); }
    if (p.mb == 4 && p.nb == 2) { launch_tile<BLOCK, 4, 2, PAIR, SEG>(a, scales, n_tiles, p.splits, partial); }
    if (p.mb == 8) { launch_tile<BLOCK, 8, 2, PAIR, SEG>(a, scales, n_tiles, p.splits, partial); }
    if (p.splits <= 1)
    {
        if (e) { add_rms_norm_rows_kernel<<<(a.tokens + 3) / 4, 256, 0, stream()>>>(e->res, a.Y, e->sum, e->norm_w, e->y, a.tokens, a.n_out, e->eps); }
        return;
    }
    if (!PAIR && !SEG)
    {
        launch_splitk_combine<DT_BF16>(partial, p.splits, a, e);
        return;
    }
    const long long blocks = ((long long)a.tokens * (features / 4) + 255) / 256, cap = (long long)cu_count() * 16;
    gemm_splitk_combine_kernel<DT_BF16, SEG, PAIR><<<(unsigned)(blocks < cap ? blocks : cap), 256, 0, stream()>>>(partial, p.splits, a);
}

template <int BLOCK>
void launch_block(const LinearArgs& a, const uint8_t* scales, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    if (pair) { launch_shape<BLOCK, true, false>(a, scales, p, partial, e); }
    else if (a.n_segments > 0) { launch_shape<BLOCK, false, true>(a, scales, p, partial, e); }
    else { launch_shape<BLOCK, false, false>(a, scales, p, partial, e); }
}

}    // namespace

void launch_gemm4_short(const LinearArgs& a, const uint8_t* tiled_scales, int block, bool pair, const GemmPlan& plan, float* partial, const AddNormArgs* e)
{
    block == 16 ? launch_block<16>(a, tiled_scales, pair, plan, partial, e) : launch_block<32>(a, tiled_scales, pair, plan, partial, e);
}

}    // namespace ccq
