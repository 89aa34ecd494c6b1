// The small tiles of plan_gemm (gemm_plan.h) on the register-fed FP8 GEMM, every one with weights requested three k-tiles ahead,
// and the k-split launches of the larger ones: one translation unit per weight type (gemm_short_e5m2.hip, gemm_short_e4m3.hip) instantiates them.
// The plans of staged_plan run gemm_staged_kernel instead (gemm_staged_e5m2.hip, gemm_staged_e4m3.hip).
#pragma once
#include "gemm_kernels.h"
#include "prefill_kernels.h"

namespace ccq
{

void launch_gemm_staged_e5m2(const LinearArgs& a, bool half, bool tiled, bool scaled, const GemmPlan& p, int n_tiles, float* partial);
void launch_gemm_staged_e4m3(const LinearArgs& a, bool half, bool tiled, bool scaled, const GemmPlan& p, int n_tiles, float* partial);

template <int WT, bool SCALED, bool TILED, int AT, int MB, int NB, bool PAIR, bool SEG, int PD = 3, bool SPLIT_ONLY = false>
void launch_short_tile(const LinearArgs& a, int n_tiles, int splits, float* partial)
{
    const dim3 grid(((n_tiles + 7) & ~7) * ((a.tokens + MB * 16 - 1) / (MB * 16)), splits);
    if (splits > 1) { gemm_mfma_direct_kernel<WT, SCALED, MB, true, TILED, AT, NB, PAIR, SEG, PD><<<grid, 256, 0, stream()>>>(a, n_tiles, partial); }
    else if constexpr (!SPLIT_ONLY) { gemm_mfma_direct_kernel<WT, SCALED, MB, false, TILED, AT, NB, PAIR, SEG, PD><<<grid, 256, 0, stream()>>>(a, n_tiles, nullptr); }
}

template <int WT, bool SCALED, bool TILED, int AT, bool PAIR, bool SEG>
void launch_short_shape(LinearArgs a, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    const int width = (PAIR ? 32 : 64) * p.nb;
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
        for (int s = a.n_segments; s < 4; s++) { a.seg_tile0[s] = n_tiles; }       // empty segments start past the last tile
        a.seg_tile0[3] = n_tiles;
    }
    if (p.staged) { (WT == DT_E5M2 ? launch_gemm_staged_e5m2 : launch_gemm_staged_e4m3)(a, AT == DT_HALF, TILED, SCALED, p, n_tiles, partial); }
    else if (p.mb == 2)
    {
        if constexpr (!PAIR)
        {
            if (p.nb == 1) { launch_short_tile<WT, SCALED, TILED, AT, 2, 1, PAIR, SEG>(a, n_tiles, p.splits, partial); }
        }
        if (p.nb == 2) { launch_short_tile<WT, SCALED, TILED, AT, 2, 2, PAIR, SEG>(a, n_tiles, p.splits, partial); }
        if (p.nb == 4) { launch_short_tile<WT, SCALED, TILED, AT, 2, 4, PAIR, SEG, 3, true>(a, n_tiles, p.splits, partial); }
    }
    else if (p.mb == 4)
    {
        if constexpr (!PAIR)
        {
            if (p.nb == 1) { launch_short_tile<WT, SCALED, TILED, AT, 4, 1, PAIR, SEG>(a, n_tiles, p.splits, partial); }
        }
        if (p.nb == 2) { launch_short_tile<WT, SCALED, TILED, AT, 4, 2, PAIR, SEG>(a, n_tiles, p.splits, partial); }
        if (p.nb == 4) { launch_short_tile<WT, SCALED, TILED, AT, 4, 4, PAIR, SEG>(a, n_tiles, p.splits, partial); }
    }
    else if (p.nb == 4) { launch_short_tile<WT, SCALED, TILED, AT, 8, 4, PAIR, SEG, 1, true>(a, n_tiles, p.splits, partial); }
    else if constexpr (!TILED && !SCALED) { launch_short_tile<WT, SCALED, TILED, AT, 8, 2, PAIR, SEG>(a, n_tiles, p.splits, partial); }
    if (p.splits <= 1)
    {
        if (e) { add_rms_norm_rows_kernel<<<(a.tokens + 3) / 4, 256, 0, stream()>>>(e->res, a.Y, e->sum, e->norm_w, e->y, a.tokens, a.n_out, e->eps); }
        return;
    }
    if (!PAIR && !SEG)
    {
        launch_splitk_combine<AT>(partial, p.splits, a, e);
        return;
    }
    const long long blocks = ((long long)a.tokens * (features / 4) + 255) / 256, cap = (long long)cu_count() * 16;
    gemm_splitk_combine_kernel<AT, SEG, PAIR><<<(unsigned)(blocks < cap ? blocks : cap), 256, 0, stream()>>>(partial, p.splits, a);
}

template <int WT, bool SCALED, bool TILED>
void launch_short_layout(const LinearArgs& a, bool half, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    if (pair) { launch_short_shape<WT, SCALED, TILED, DT_BF16, true, false>(a, p, partial, e); }
    else if (a.n_segments > 0) { launch_short_shape<WT, SCALED, TILED, DT_BF16, false, true>(a, p, partial, e); }
    else if (half) { launch_short_shape<WT, SCALED, TILED, DT_HALF, false, false>(a, p, partial, e); }
    else { launch_short_shape<WT, SCALED, TILED, DT_BF16, false, false>(a, p, partial, e); }
}

template <int WT>
void launch_short_type(const LinearArgs& a, bool half, bool tiled, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e)
{
    bool scaled = a.n_segments == 0 && (a.w_scale != 1.0f || (pair && a.w_scale_pair != 1.0f));
    for (int s = 0; s < a.n_segments; s++) { scaled = scaled || a.seg_w_scale[s] != 1.0f; }
    if (scaled) { tiled ? launch_short_layout<WT, true, true>(a, half, pair, p, partial, e) : launch_short_layout<WT, true, false>(a, half, pair, p, partial, e); }
    else { tiled ? launch_short_layout<WT, false, true>(a, half, pair, p, partial, e) : launch_short_layout<WT, false, false>(a, half, pair, p, partial, e); }
}

void launch_gemm_short_e5m2(const LinearArgs& a, bool half, bool tiled, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e);
void launch_gemm_short_e4m3(const LinearArgs& a, bool half, bool tiled, bool pair, const GemmPlan& p, float* partial, const AddNormArgs* e);

}    // namespace ccq
