// Prompt GEMM whose operands reach LDS by direct loads, several k-stages ahead, issued by waves that do nothing else.
#pragma once
#include "gemm_kernels.h"

namespace ccq
{

// all but the newest N loads of this wave have arrived, then the workgroup's barrier
template <int N>
__device__ __forceinline__ void wait_loads_barrier()
{
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N) : "memory");
}

// FP8 weights, K % 64 == 0.  A workgroup owns 16 MB tokens x 64 WF features (a pair: 32 WF of gate and of up) and walks K in stages of
// 128.  Four loading waves keep S stages of activations and S + 1 of weights (the codes as they are) on their way into LDS; 4 WF
// computing waves take 16 features and all the tokens each and convert their codes in registers, a k-tile of 64 ahead of their use.
//   Why: a prompt of 17 to some 500 tokens is bound by neither the matrix cores nor HBM but by what a CU waits for.  In
// gemm_mfma_direct_kernel each wave issues its own loads between its matrix-core instructions and reads a row of the file layout
// 64 bytes at a time (half a line).  Here loads never hold up a computing wave (with the loads spread over the computing waves 38
// against 34 us on the pair below), a line is read whole, and what is in flight (60 to 120 KiB a CU) does not cost registers.
//   E5M2, file layout, MI355X, gemm_mfma_direct_kernel -> this one, us: gate / up pair 4096 x 12288 at 100 tokens 43.7 -> 33.2, at 20 tokens
// 29.7 -> 24.2; 12288 x 4096 at 160 tokens 37.7 -> 31.3; 4096 x 4096 at 512 tokens 31.4 -> 23.0, at 100 tokens 15.6 -> 13.8.
//   An element's products are added in the order of every other prompt GEMM, v_mfma_f32_16x16x32 by v_mfma_f32_16x16x32 in ascending k, so a
// launch has the same bits whichever kernel its plan takes.  (With each of four waves on a quarter of every stage and their sums
// added at the end an activation is read from LDS once per 64 features and not once per 16, yet that was 2 % slower over the shapes
// measured, 5 % on tiles of 32 tokens, and faster, by up to 7 %, only where a CU has several workgroups of 64 tokens or more.)
//
// LDS: X stages (rows of 256 bytes, 16-byte chunk c of row r at c ^ (r % 16)), then W stages (file layout: rows of 128 bytes, chunk c at
// c ^ (r / 2 % 8); tiled copy: its KiB blocks, two per 16 rows).  In a k-tile lane group g holds elements 16 g .. + 7 of the first
// instruction and 16 g + 8 .. + 15 of the second, as in the tiled copy.
// Pair: a.W_pair is set; segments: a.n_segments > 0; k split: `partial` is set and blockIdx.y the range (all as in
// gemm_mfma_direct_kernel, whose combine launches finish the sums).
template <int WT, bool SCALED, bool TILED, int AT, int MB, int WF, int S>
__global__ __launch_bounds__(256 + 256 * WF, WF == 2 ? 3 : 4) void gemm_staged_kernel(const LinearArgs a_in, const int n_tiles, float* __restrict__ partial)
{
    constexpr int COMPUTE = 4 * WF, LOADERS = 4;                            // waves
    constexpr int BTOK = 16 * MB, BF = 64 * WF, BK = 128;
    constexpr int X_STAGE = BTOK * BK * 2, W_STAGE = BF * BK, W_AT = S * X_STAGE;
    constexpr int XI = MB, WI = BF / 8 / LOADERS, LOADS = XI + WI;          // a loading wave's instructions (a KiB each) per stage
    constexpr int RS = BF + 4;                                              // floats per token row of the sums in LDS
    constexpr int SUM_BYTES = BTOK * RS * 4, STAGE_BYTES = W_AT + (S + 1) * W_STAGE;
    constexpr int LDS_BYTES = STAGE_BYTES > SUM_BYTES ? STAGE_BYTES : SUM_BYTES;
    static_assert(S >= 3 && S <= 5 && LDS_BYTES * (3 - WF) <= 160 * 1024, "64-feature tiles: two workgroups on a CU");
    __shared__ __align__(1024) uint8_t lds[LDS_BYTES];
    typedef typename std::conditional<AT == DT_HALF, f16x8, bf16x8>::type frag_t;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_pad = (n_tiles + 7) & ~7;                                   // feature tile n on XCD n % 8, as in gemm_mfma_direct_kernel
    int n_tile = blockIdx.x % n_pad;
    const int m_tile = blockIdx.x / n_pad;
    if (n_tile >= n_tiles) { return; }                                      // padding
    LinearArgs a = a_in;
    const bool pair = a_in.W_pair != nullptr;
    if (a_in.n_segments > 0)
    {
        const int s = n_tile >= a_in.seg_tile0[2] ? 2 : (n_tile >= a_in.seg_tile0[1] ? 1 : 0);
        a.W = a_in.seg_W[s];
        a.Y = a_in.seg_Y[s];
        a.n_out = a_in.seg_n_out[s];
        a.w_scale = a_in.seg_w_scale[s];
        a.y_stride_tok = a_in.seg_y_stride_tok[s];
        n_tile -= a_in.seg_tile0[s];
        // the partial sums of a segment follow those of the segments before it
        if (partial) { partial += (long long)gridDim.y * a_in.tokens * ((s > 0 ? a_in.seg_n_out[0] : 0) + (s > 1 ? a_in.seg_n_out[1] : 0)); }
    }
    const int width = pair ? BF / 2 : BF;                                   // output features of the tile; pair: rows `width` and up are the up weight's
    const int out_base = n_tile * width;
    const int tok_base = m_tile * BTOK;
    const int n_st_total = (a.K + BK - 1) / BK;
    const int st_begin = (int)((long long)n_st_total * blockIdx.y / gridDim.y);
    const int n_st = (int)((long long)n_st_total * (blockIdx.y + 1) / gridDim.y) - st_begin;

    if (wave >= COMPUTE)
    {
        // ---- loading waves: wave lw takes X instructions lw, lw + 4, ... (four token rows each) and W instructions lw, lw + 4, ... (eight
        // rows of the file layout, or one block of the tiled copy).  Addresses are a uniform base plus a 32-bit lane offset (the
        // launcher checks that both operands are smaller than 4 GiB); rows past the last one re-read it.
        __builtin_amdgcn_s_setprio(3);                                      // 2-6 % on launches with few workgroups: their loads go out first
        const int lw = wave - COMPUTE;
        const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)lds;
        const int n_blk = a.K / 64;
        const uint32_t x_last = (uint32_t)a.K * 2u - 16u, w_last = (uint32_t)a.K - 16u;      // K % 128 == 64: the last stage's second half re-reads the row's end
        uint32_t x_row[XI], x_chunk[XI], w_row[WI], w_chunk[WI];
        const uint8_t* w_base[WI];
#pragma unroll
        for (int i = 0; i < XI; i++)
        {
            const int row = 4 * (lw + LOADERS * i) + (lane >> 4);
            x_row[i] = (uint32_t)((long long)min(tok_base + row, a.tokens - 1) * a.ldx * 2);
            x_chunk[i] = (uint32_t)swizzled_chunk_n<16>(row, lane & 15) * 16u;
        }
#pragma unroll
        for (int i = 0; i < WI; i++)
        {
            const int q = lw + LOADERS * i;
            const int row_q = TILED ? (q >> 1) * 16 : q * 8;
            const bool up = row_q >= width;
            const int row0 = out_base + row_q - (up ? width : 0);
            w_base[i] = up ? a.W_pair : a.W;
            if constexpr (TILED)
            {
                w_base[i] += (long long)min(row0 / 16, (a.n_out + 15) / 16 - 1) * n_blk * 1024;
                w_row[i] = lane * 16;
                w_chunk[i] = 0;
            }
            else
            {
                w_row[i] = (uint32_t)((long long)min(row0 + (lane >> 3), a.n_out - 1) * a.ldw);
                w_chunk[i] = (uint32_t)swizzled_chunk_n<8>(q * 8 + (lane >> 3), lane & 7) * 16u;
            }
        }
        const bool stream = (int)gridDim.x == n_pad;                        // one token tile: each weight is read once (12 % on the pair at 32 tokens)
        auto load_w = [&](int st, int buf) {
            const uint32_t k0 = (uint32_t)(st_begin + st) * BK;
#pragma unroll
            for (int i = 0; i < WI; i++)
            {
                const int q = lw + LOADERS * i;
                const uint32_t dst = lds0 + W_AT + buf * W_STAGE + q * 1024;
                const uint8_t* const base = TILED ? w_base[i] + (long long)min((int)(k0 / 64) + (q & 1), n_blk - 1) * 1024 : w_base[i];
                const uint32_t off = TILED ? w_row[i] : w_row[i] + min(k0 + w_chunk[i], w_last);
                if (stream) { load_to_lds<true>(dst, base, off); }
                else { load_to_lds<false>(dst, base, off); }
            }
        };
        // step j: the weights of stage j + 1 and the activations of stage j (past the last stage: none)
        auto step = [&](int j, int xbuf, int wbuf) {
            if (j + 1 < n_st) { load_w(j + 1, wbuf); }
            if (j >= n_st) { return; }
            const uint32_t k0 = (uint32_t)(st_begin + j) * BK * 2;
#pragma unroll
            for (int i = 0; i < XI; i++) { load_to_lds<false>(lds0 + xbuf * X_STAGE + (lw + LOADERS * i) * 1024, (const uint8_t*)a.X, x_row[i] + min(k0 + x_chunk[i], x_last)); }
        };
        load_w(0, 0);
#pragma unroll
        for (int j = 0; j < S - 1; j++) { step(j, j, j + 1); }
        int xbuf = S - 1, wbuf = S;
        for (int st = 0; st < n_st; st++)
        {
            // step st has arrived; the steps behind it stay in flight: `newer` of them, the last without weights once they have run out.
            // Past the barrier every computing wave is done with stage st - 1, whose buffers step st + S - 1 refills.
            const int newer = min(n_st - 1 - st, S - 2);
            if (newer == 0) { wait_loads_barrier<0>(); }
            else if (st + S - 1 >= n_st)
            {
                if (newer == 1) { wait_loads_barrier<XI>(); }
                else if (newer == 2) { wait_loads_barrier<LOADS + XI>(); }
                else { wait_loads_barrier<2 * LOADS + XI>(); }
            }
            else if (S == 3) { wait_loads_barrier<LOADS>(); }
            else if (S == 4) { wait_loads_barrier<2 * LOADS>(); }
            else { wait_loads_barrier<3 * LOADS>(); }
            step(st + S - 1, xbuf, wbuf);
            xbuf = xbuf == S - 1 ? 0 : xbuf + 1;
            wbuf = wbuf == S ? 0 : wbuf + 1;
        }
        return;                                                             // a wave that has ended no longer counts in the barriers below
    }

    // ---- computing waves: features 16 wave .. + 15 of the tile
    const int i16 = lane & 15, g = lane >> 4;
    const float scale = wave * 16 >= width ? a.w_scale_pair : a.w_scale;
    f32x4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) { acc[mb] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }; }
    int x_lane[4], w_lane[2];                                               // per instruction / k-tile of a stage
#pragma unroll
    for (int s = 0; s < 4; s++) { x_lane[s] = i16 * 256 + swizzled_chunk_n<16>(i16, 8 * (s >> 1) + 2 * g + (s & 1)) * 16; }
#pragma unroll
    for (int h = 0; h < 2; h++) { w_lane[h] = W_AT + wave * 2048 + (TILED ? h * 1024 + lane * 16 : i16 * 128 + swizzled_chunk_n<8>(i16, 4 * h + g) * 16); }
    u32x4 raw, wfr[4];                                                      // codes of a k-tile; weight operands of a stage
    auto read_codes = [&](int buf, int h) { raw = *(const u32x4*)(lds + buf * W_STAGE + w_lane[h]); };
    auto convert = [&](int h) { dequant16_fp8<WT, SCALED, AT>(raw, scale, wfr[2 * h], wfr[2 * h + 1]); };
    int xbuf = 0, wbuf = 0;
    for (int st = 0; st < n_st; st++)
    {
        asm volatile("s_barrier" : : : "memory");                           // activations of stage st, codes of stage st + 1
        // Fragment f: token block f % MB of instruction f / MB.  Reads run ahead of the matrix-core instructions that use them (by 3 or 4: level;
        // 6: 1 to 2 % slower, 12: 2 to 5 %).
        constexpr int FRAGS = 4 * MB, AHEAD = 4;
        const uint8_t* const xp = lds + xbuf * X_STAGE;
        auto read_frag = [&](int f) { return *(const u32x4*)(xp + x_lane[f / MB] + f % MB * 4096); };
        u32x4 ring[AHEAD + 1];
#pragma unroll
        for (int f = 0; f < AHEAD; f++) { ring[f] = read_frag(f); }
        if (st == 0)
        {
            read_codes(0, 0);
            convert(0);
        }
        read_codes(wbuf, 1);
        wbuf = wbuf == S ? 0 : wbuf + 1;
        auto products = [&](int f0, int f1) {
#pragma unroll
            for (int f = f0; f < f1; f++)
            {
                __builtin_amdgcn_sched_barrier(0);
                if (f + AHEAD < FRAGS) { ring[(f + AHEAD) % (AHEAD + 1)] = read_frag(f + AHEAD); }
                const frag_t xf = __builtin_bit_cast(frag_t, ring[f % (AHEAD + 1)]), w = __builtin_bit_cast(frag_t, wfr[f / MB]);
                if constexpr (AT == DT_HALF) { acc[f % MB] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, xf, acc[f % MB], 0, 0, 0); }
                else { acc[f % MB] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, xf, acc[f % MB], 0, 0, 0); }
                // behind the first instruction of a k-tile: the codes of the k-tile after it
                if (f == MB - 1)
                {
                    convert(1);
                    read_codes(wbuf, 0);                                    // (behind the last stage: what is left in LDS, and not used)
                }
                if (f == 3 * MB - 1) { convert(0); }
            }
        };
        products(0, 2 * MB);
        // K % 128 == 64: the last stage has one k-tile.  (A product of the activations read in the other's place with zeros would
        // make NaN of an infinity among them.)
        if ((st_begin + st) * BK + 64 >= a.K) { break; }
        products(2 * MB, FRAGS);
        __builtin_amdgcn_sched_barrier(0);
        xbuf = xbuf == S - 1 ? 0 : xbuf + 1;
    }

    // ---- through LDS to rows: a thread owns 8 consecutive features of a token (a pair: 4 outputs)
    float* const sums = (float*)lds;
    const int s_tok = tid / (BF / 8), s_f = tid % (BF / 8);
    const int f0 = pair ? s_f * 4 : s_f * 8, f1 = pair ? f0 + width : f0 + 4;
    const int out = out_base + f0;
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < MB; mb++) { *(f32x4*)(sums + (mb * 16 + i16) * RS + wave * 16 + 4 * g) = acc[mb]; }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < (MB + 1) / 2; c++)
    {
        const int tok = tok_base + c * 32 + s_tok;
        if (tok >= a.tokens || c * 32 + s_tok >= BTOK || out >= a.n_out) { continue; }
        const f32x4 r0 = *(const f32x4*)(sums + (c * 32 + s_tok) * RS + f0), r1 = *(const f32x4*)(sums + (c * 32 + s_tok) * RS + f1);
        if (partial)
        {
            // n_out is a multiple of 4 on this path; pair: the up weight's sums are a second set behind all of the gate weight's
            float* p = partial + ((long long)blockIdx.y * a.tokens + tok) * a.n_out + out;
            *(f32x4*)p = r0;
            if (pair) { *(f32x4*)(p + (long long)gridDim.y * a.tokens * a.n_out) = r1; }
            else if (out + 4 < a.n_out) { *(f32x4*)(p + 4) = r1; }
            continue;
        }
        uint16_t* y = a.Y + (long long)tok * a.y_stride_tok + (long long)out * a.y_stride_out;
        if (pair)
        {
            uint16_t o[4];
#pragma unroll
            for (int v = 0; v < 4; v++)
            {
                const float gate = bf16_bits_to_f32(f32_to_bf16_bits(r0[v])), up = bf16_bits_to_f32(f32_to_bf16_bits(r1[v]));
                const float sig = bf16_bits_to_f32(f32_to_bf16_bits(1.0f / (1.0f + expf(-gate))));
                o[v] = (uint16_t)f32_to_bf16_bits(bf16_bits_to_f32(f32_to_bf16_bits(gate * sig)) * up);
            }
            if (a.y_stride_out == 1 && a.y_stride_tok % 4 == 0 && ((uintptr_t)a.Y & 7u) == 0 && out + 3 < a.n_out)
            {
                *(uint2*)y = uint2{ (uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16) };
            }
            else
            {
#pragma unroll
                for (int v = 0; v < 4; v++)
                {
                    if (out + v < a.n_out) { y[v * a.y_stride_out] = o[v]; }
                }
            }
        }
        else if (a.y_stride_out == 1 && a.y_stride_tok % 8 == 0 && ((uintptr_t)a.Y & 15u) == 0 && out + 7 < a.n_out)
        {
            u32x4 old = { 0u, 0u, 0u, 0u }, packed;
            if (a.beta != 0.0f) { old = *(const u32x4*)y; }
#pragma unroll
            for (int d = 0; d < 4; d++)
            {
                const uint16_t old_lo = (uint16_t)(old[d] & 0xFFFFu), old_hi = (uint16_t)(old[d] >> 16);
                const uint32_t lo = finish_output_act<AT>(d < 2 ? r0[2 * d] : r1[2 * d - 4], a.alpha, a.beta, &old_lo);
                const uint32_t hi = finish_output_act<AT>(d < 2 ? r0[2 * d + 1] : r1[2 * d - 3], a.alpha, a.beta, &old_hi);
                packed[d] = lo | (hi << 16);
            }
            *(u32x4*)y = packed;
        }
        else
        {
#pragma unroll
            for (int v = 0; v < 8; v++)
            {
                if (out + v < a.n_out) { y[v * a.y_stride_out] = finish_output_act<AT>(v < 4 ? r0[v & 3] : r1[v & 3], a.alpha, a.beta, y + v * a.y_stride_out); }
            }
        }
    }
}

template <int WT, bool SCALED, bool TILED, int AT, int MB, int WF, int S>
void launch_staged_tile(const LinearArgs& a, int n_tiles, int splits, float* partial)
{
    const dim3 grid(((n_tiles + 7) & ~7) * ((a.tokens + MB * 16 - 1) / (MB * 16)), splits);
    gemm_staged_kernel<WT, SCALED, TILED, AT, MB, WF, S><<<grid, 256 + 256 * WF, 0, stream()>>>(a, n_tiles, splits > 1 ? partial : nullptr);
}

// the tiles of kStagedTiles (gemm_plan.h), each with as many stages as LDS holds
template <int WT, bool SCALED, bool TILED, int AT>
void launch_staged_tiles(const LinearArgs& a, const GemmPlan& p, int n_tiles, float* partial)
{
    if (p.mb == 2 && p.nb == 1) { launch_staged_tile<WT, SCALED, TILED, AT, 2, 1, 4>(a, n_tiles, p.splits, partial); }
    else if (p.mb == 2) { launch_staged_tile<WT, SCALED, TILED, AT, 2, 2, 5>(a, n_tiles, p.splits, partial); }
    else if (p.mb == 3) { launch_staged_tile<WT, SCALED, TILED, AT, 3, 2, 5>(a, n_tiles, p.splits, partial); }
    else if (p.mb == 4 && p.nb == 1) { launch_staged_tile<WT, SCALED, TILED, AT, 4, 1, 3>(a, n_tiles, p.splits, partial); }
    else if (p.mb == 4) { launch_staged_tile<WT, SCALED, TILED, AT, 4, 2, 4>(a, n_tiles, p.splits, partial); }
    else if (p.mb == 5) { launch_staged_tile<WT, SCALED, TILED, AT, 5, 2, 4>(a, n_tiles, p.splits, partial); }
    else { launch_staged_tile<WT, SCALED, TILED, AT, 7, 2, 3>(a, n_tiles, p.splits, partial); }
}

template <int WT>
void launch_staged_type(const LinearArgs& a, bool half, bool tiled, bool scaled, const GemmPlan& p, int n_tiles, float* partial)
{
    if (half)
    {
        if (scaled) { tiled ? launch_staged_tiles<WT, true, true, DT_HALF>(a, p, n_tiles, partial) : launch_staged_tiles<WT, true, false, DT_HALF>(a, p, n_tiles, partial); }
        else { tiled ? launch_staged_tiles<WT, false, true, DT_HALF>(a, p, n_tiles, partial) : launch_staged_tiles<WT, false, false, DT_HALF>(a, p, n_tiles, partial); }
    }
    else if (scaled) { tiled ? launch_staged_tiles<WT, true, true, DT_BF16>(a, p, n_tiles, partial) : launch_staged_tiles<WT, true, false, DT_BF16>(a, p, n_tiles, partial); }
    else { tiled ? launch_staged_tiles<WT, false, true, DT_BF16>(a, p, n_tiles, partial) : launch_staged_tiles<WT, false, false, DT_BF16>(a, p, n_tiles, partial); }
}

}    // namespace ccq
