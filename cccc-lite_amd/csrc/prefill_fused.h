// Causal attention of a prompt on direct loads to LDS and transposing LDS reads: with the reference's rounding points in two passes over the keys,
// or in one pass (the split-softmax form of attn_fused_kernel for T tokens).
#pragma once
#include "prefill_kernels.h"

namespace ccq
{

// Causal GQA attention of T query tokens over cache rows 0 .. pos0 + t, head_dim 128, scores rounded to BF16 and masked.
//   PF_WHOLE_ROW: probabilities of the whole row, rounded to BF16 behind the division by their sum: a pass over the keys for (max, sum) of every
// row, then one for the products.  The sums of attn_prefill_kernel in the same order: the same bits.
//   PF_ONE_PASS: softmax against a running maximum, probabilities rounded to BF16 before the division by their FP32 sum.
// PF_ONE_PASS_RANGE: the same over the keys of one range, FP32 sums and statistics left to attn_prefill_fused_combine_kernel.
//   A workgroup of four waves owns 64 rows of one kv head -- 16 tokens of four query heads, 32 of two, 64 of one -- and a wave two groups
// of 16 rows (a head's 16 tokens) and one half, 32 keys, of every block of 64.  Keys and values go from memory to LDS by direct loads, a
// block ahead, rows of 256 bytes as they are; the products of the next block are issued before the softmax of this one.  The first pass of
// PF_WHOLE_ROW has the values' half of the LDS to itself and loads three blocks ahead.
//   scores: v_mfma_f32_16x16x32_bf16, key rows as row operand, rotated queries as columns: D lane (row j = lane % 16, g = lane / 16) holds
//           keys 4 g .. + 3 of 16.
//   V p:    the eight probabilities of a lane (keys 4 g .. + 3 and 16 + 4 g .. + 3) are its column operand as they are; the row operand (dim,
//           the same keys) comes from ds_read_b64_tr_b16, which hands lane i of 16 element i % 4 of the 8 bytes that lanes i / 4, 4 + i / 4, 8 + i / 4,
//           12 + i / 4 point at.  D lane (row j, g) holds dims 4 g .. + 3: a row's scale is a lane's.
// The running maximum of a row moves only when a score exceeds it by more than PF_LAG: until then the weights are at most e^PF_LAG (403), which
// FP32 sums and BF16's exponent do not notice, and the sums are left alone.
//   Bound: by what a wave issues between its matrix-core instructions (one pass: 0.87 us per block with one workgroup per CU, 1.35 for two side by
// side; matrix cores 40 % busy with two).  MI355X, us, attn_prefill_kernel / two passes here / one pass: 32 / 8 heads, 2048 tokens from 0
// 111 / 78 / 53, 512 behind 3000 103 / 84 / 52, 1024 behind 3000 165 / 120 / 78; 8 / 8 heads, 2048 from 0 103 / 51 / 33.  There each row group
// read the keys twice, key and value rows went through registers with 32 lines per load instruction, and values were transposed by the VALU.
// LDS: chunk c (16 bytes) of key row r lies at c ^ (r % 16), of value row r at c ^ (2 (r % 8)): the operand reads hit all banks.
// A block's rows past the last written one repeat that row; their weight is 0 and their values are cleared in front of the products.
constexpr float PF_LAG = 6.0f;

typedef short tr_b16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint2 read_transposed(const uint8_t* p)
{
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_b16x4*)p));
}

// What a launch of the kernel below does with its keys.
constexpr int PF_ONE_PASS = 0, PF_ONE_PASS_RANGE = 1, PF_WHOLE_ROW = 2;

template <int G, int FORM>
__global__ __launch_bounds__(256, 2) void attn_prefill_tile_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ v_cache,
                                                                    uint16_t* __restrict__ y, int n_q, int t_kv, int n_tokens, int pos0, float scale, const PrefillRanges ranges)
{
    static_assert(G == 1 || G == 2 || G == 4, "query heads per kv head");
    constexpr bool RANGE = FORM == PF_ONE_PASS_RANGE, WHOLE_ROW = FORM == PF_WHOLE_ROW;
    constexpr int TOKENS = 16 * (4 / G);        // of a workgroup
    constexpr int BLOCK = PF_KEYS * 256;        // bytes of a staged block
    constexpr int RS = 132;                     // floats per row of the sums: the lanes of a store hit different banks
    __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * BLOCK];         // two blocks of keys, two of values; then the sums
    __shared__ float2 stat[4][2][16];                                         // (max, sum) per wave, group and row
    static_assert(64 * RS * 4 <= 4 * BLOCK, "sums");
    const int n_kv = n_q / G;
    const int kvh = blockIdx.x % n_kv;          // an XCD's workgroups share few heads, whose rows stay in its L2
    const int t0 = ((int)gridDim.x / n_kv - 1 - (int)blockIdx.x / n_kv) * TOKENS;      // the workgroups that see the most keys go first
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int n_written = pos0 + n_tokens;
    const int n_blocks = (pos0 + min(t0 + TOKENS, n_tokens) + PF_KEYS - 1) / PF_KEYS;
    const int b_begin = RANGE ? (int)blockIdx.y * ranges.per : 0;             // even: block b always goes to buffer b & 1
    const int b_end = RANGE ? min(n_blocks, b_begin + ranges.per) : n_blocks;
    if (RANGE && b_begin >= n_blocks) { return; }           // a range past this tile's last key: nobody reads it
    const int kh = wave & 1;
    const uint8_t* const kbase = (const uint8_t*)(k_cache + (size_t)kvh * t_kv * 128);
    const uint8_t* const vbase = (const uint8_t*)(v_cache + (size_t)kvh * t_kv * 128);

    // the wave's row groups: token and head
    int tok[2], head[2], my_pos[2], group_blocks[2];
    u32x4 qf[2][4];
#pragma unroll
    for (int h = 0; h < 2; h++)
    {
        const int group = (wave >> 1) * 2 + h;
        head[h] = kvh * G + group % G;
        tok[h] = t0 + 16 * (group / G) + j;
        const int t = min(tok[h], n_tokens - 1);
        my_pos[h] = pos0 + t;
        group_blocks[h] = (pos0 + min(t0 + 16 * (group / G) + 16, n_tokens) + PF_KEYS - 1) / PF_KEYS;
        const uint16_t* const row = q + ((size_t)t * n_q + head[h]) * 128 + g * 8;
#pragma unroll
        for (int c = 0; c < 4; c++) { qf[h][c] = *(const u32x4*)(row + c * 32); }
    }

    // staging: an instruction moves four rows, lane l chunk l % 16 of row l / 16
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + (uint32_t)wave * 4096u;
    auto stage = [&](const uint8_t* base, uint32_t to, int b, bool values) {
#pragma unroll
        for (int i = 0; i < 4; i++)
        {
            const int r = 4 * i + g;            // of the wave's 16
            const uint32_t row = (uint32_t)min(b * PF_KEYS + wave * 16 + r, n_written - 1);
            load_to_lds<false>(lds0 + to + i * 1024u, base, row * 256u + (uint32_t)((values ? j ^ (2 * (r & 7)) : j ^ r) * 16));
        }
    };
    auto stage_keys = [&](int b, int buffers = 2) { stage(kbase, (b & (buffers - 1)) * BLOCK, b, false); };
    auto stage_values = [&](int b) { stage(vbase, (2 + (b & 1)) * BLOCK, b, true); };

    int k_at[4];                                // of chunk 4 c + g of key row 32 kh + j
#pragma unroll
    for (int c = 0; c < 4; c++) { k_at[c] = (32 * kh + j) * 256 + (((4 * c + g) ^ j) << 4); }
    // raw scores of the wave's two key tiles (keys 32 kh + 16 kt + 4 g + v) of a staged block
    auto score_products = [&](int buffer, f32x4 (&acc)[2][2]) {
        const uint8_t* const kb = lds + buffer * BLOCK;
        u32x4 kf[2][4];
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int c = 0; c < 4; c++) { kf[kt][c] = *(const u32x4*)(kb + k_at[c] + kt * 16 * 256); }
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int kt = 0; kt < 2; kt++) { acc[h][kt] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }; }
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                {
                    acc[h][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf[kt][c]), __builtin_bit_cast(bf16x8, qf[h][c]), acc[h][kt], 0, 0, 0);
                }
    };

    // scaled, rounded to BF16 and masked
    auto score_round = [&](const f32x4 (&raw)[2][2], int b, auto masked_c, float (&s)[2][2][4]) {
        constexpr bool masked = decltype(masked_c)::value;
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
            {
                const f32x4 a = raw[h][kt];
                const uint32_t w01 = pf_pack_bf16(scale * a[0], scale * a[1]), w23 = pf_pack_bf16(scale * a[2], scale * a[3]);
                s[h][kt][0] = __builtin_bit_cast(float, w01 << 16);
                s[h][kt][1] = __builtin_bit_cast(float, w01 & 0xFFFF0000u);
                s[h][kt][2] = __builtin_bit_cast(float, w23 << 16);
                s[h][kt][3] = __builtin_bit_cast(float, w23 & 0xFFFF0000u);
#pragma unroll
                for (int v = 0; v < 4; v++)
                {
                    if (masked && b * PF_KEYS + kh * 32 + kt * 16 + 4 * g + v > my_pos[h]) { s[h][kt][v] = -INFINITY; }
                }
            }
    };

    float m[2] = { -INFINITY, -INFINITY }, l[2] = { 0.0f, 0.0f }, poff[2];
    f32x4 out[2][8];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int d = 0; d < 8; d++) { out[h][d] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }; }
    // dims 16 d + 4 (lane % 4) .. + 3 of value row 32 kh + 4 g + lane % 16 / 4 (and of the one 16 further)
    const int v_row = 4 * g + (j >> 2);
    const int v_at = (32 * kh + v_row) * 256 + (((j & 3) >> 1) << 4) + ((j & 1) << 3), v_swz = (2 * (v_row & 7)) << 4;

    auto weigh = [&](const f32x4 (&raw)[2][2], int b, auto masked_c) {
        constexpr bool masked = decltype(masked_c)::value;
        const uint8_t* const vb = lds + (2 + (b & 1)) * BLOCK + v_at;
        u32x4 vf[8];
#pragma unroll
        for (int d = 0; d < 8; d++)
        {
            const uint8_t* const p = vb + ((32 * d) ^ v_swz);
            const uint2 lo = read_transposed(p), hi = read_transposed(p + 16 * 256);
            vf[d] = u32x4{ lo.x, lo.y, hi.x, hi.y };
        }
        if (masked && (b + 1) * PF_KEYS > n_written)
        {
            // rows past the last written one weigh 0, but 0 times a repeated infinity is NaN
            const int key = b * PF_KEYS + 32 * kh + 4 * g;
            u32x4 keep;
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                const int k0 = key + (i >> 1) * 16 + (i & 1) * 2;
                keep[i] = (k0 < n_written ? 0x0000FFFFu : 0u) | (k0 + 1 < n_written ? 0xFFFF0000u : 0u);
            }
#pragma unroll
            for (int d = 0; d < 8; d++) { vf[d] &= keep; }
        }
        float s[2][2][4];
        score_round(raw, b, masked_c, s);
        if constexpr (WHOLE_ROW)
        {
#pragma unroll
            for (int h = 0; h < 2; h++)
            {
                if (masked && b >= group_blocks[h]) { continue; }       // none of the group's tokens sees the block
                bf16x8 pb;
#pragma unroll
                for (int e = 0; e < 8; e++) { pb[e] = (__bf16)pf_exp2(fmaf(s[h][e >> 2][e & 3], PF_LOG2E, poff[h])); }
#pragma unroll
                for (int d = 0; d < 8; d++) { out[h][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vf[d]), pb, out[h][d], 0, 0, 0); }
            }
            return;
        }
        float top[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            top[h] = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; e++) { top[h] = fmaxf(top[h], s[h][e >> 2][e & 3]); }
        }
        if (__any(top[0] > m[0] + PF_LAG || top[1] > m[1] + PF_LAG))
        {
#pragma unroll
            for (int h = 0; h < 2; h++)
            {
                float nm = fmaxf(top[h], __shfl_xor(top[h], 16));
                nm = fmaxf(m[h], fmaxf(nm, __shfl_xor(nm, 32)));
                const float shrink = nm > -INFINITY ? pf_exp2((m[h] - nm) * PF_LOG2E) : 1.0f;
                m[h] = nm;
                l[h] *= shrink;
#pragma unroll
                for (int d = 0; d < 8; d++) { out[h][d] *= shrink; }
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            if (masked && b >= group_blocks[h]) { continue; }           // none of the group's tokens sees the block
            const float off = m[h] > -INFINITY ? -m[h] * PF_LOG2E : 0.0f;      // -inf: the row has seen no key yet, every weight is 2^-inf = 0
            float p[8];
#pragma unroll
            for (int e = 0; e < 8; e++)
            {
                p[e] = pf_exp2(fmaf(s[h][e >> 2][e & 3], PF_LOG2E, off));
            }
            l[h] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            const bf16x8 pb = { (__bf16)p[0], (__bf16)p[1], (__bf16)p[2], (__bf16)p[3], (__bf16)p[4], (__bf16)p[5], (__bf16)p[6], (__bf16)p[7] };
#pragma unroll
            for (int d = 0; d < 8; d++) { out[h][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vf[d]), pb, out[h][d], 0, 0, 0); }
        }
    };
    // loads of this wave into LDS have arrived and its reads of LDS are done, then the workgroup's barrier
    auto staged_barrier = []() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    f32x4 cur[2][2], next[2][2];
    auto take_next = [&]() {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int kt = 0; kt < 2; kt++) { cur[h][kt] = next[h][kt]; }
    };
    // blocks before n_plain end at or before the first token's position and need no mask test
    const int n_plain = max(b_begin, min((pos0 + t0 + 1) / PF_KEYS, b_end));
    if constexpr (WHOLE_ROW)
    {
        // pass 1: row maximum and sum of exp(s - max), per lane over its keys; keys in all four buffers, up to three blocks ahead
        auto statistics = [&](const f32x4 (&raw)[2][2], int b, auto masked_c) {
            float s[2][2][4];
            score_round(raw, b, masked_c, s);
#pragma unroll
            for (int h = 0; h < 2; h++)
            {
                float bm = -INFINITY;
#pragma unroll
                for (int e = 0; e < 8; e++) { bm = fmaxf(bm, s[h][e >> 2][e & 3]); }
                const float nm = fmaxf(m[h], bm);
                // nm = -inf: nothing visible to this lane yet, every term below is 2^(-inf) = 0 with the offset at 0
                const float off = nm > -INFINITY ? -nm * PF_LOG2E : 0.0f;
                l[h] = nm == m[h] ? l[h] : l[h] * pf_exp2(fmaf(m[h], PF_LOG2E, off));
                m[h] = nm;
                float sum = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) { sum += pf_exp2(fmaf(s[h][e >> 2][e & 3], PF_LOG2E, off)); }
                l[h] += sum;
            }
        };
        stage_keys(0, 4);
        if (1 < b_end) { stage_keys(1, 4); }
        if (2 < b_end)
        {
            stage_keys(2, 4);
            asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        else { staged_barrier(); }
        score_products(0, cur);
        // iteration b: keys of b + 1 are in LDS, those of b + 2 on their way, `cur` holds the raw scores of b
        auto block = [&](int b, auto masked_c) {
            if (b + 3 < b_end) { stage_keys(b + 3, 4); }            // the buffer of b - 1, read before the last barrier
            if (b + 1 < b_end) { score_products((b + 1) & 3, next); }
            statistics(cur, b, masked_c);
            if (b + 3 < b_end) { asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
            else { staged_barrier(); }
            take_next();
        };
        for (int b = 0; b < n_plain; b++) { block(b, std::false_type{}); }
        for (int b = n_plain; b < b_end; b++) { block(b, std::true_type{}); }
    }
    // (no block past the last one is loaded: of a short prompt that would be most of the launch)
    stage_keys(b_begin);
    stage_values(b_begin);
    if (b_begin + 1 < b_end) { stage_keys(b_begin + 1); }
    if constexpr (WHOLE_ROW)
    {
        // the four lane groups of a row, then the two halves of its keys
        auto merge = [&](float& ma, float& la, float mb, float lb) {
            const float nm = fmaxf(ma, mb);
            if (nm > -INFINITY) { la = la * pf_exp2((ma - nm) * PF_LOG2E) + lb * pf_exp2((mb - nm) * PF_LOG2E); }
            ma = nm;
        };
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
#pragma unroll
            for (int off = 16; off < 64; off <<= 1) { merge(m[h], l[h], __shfl_xor(m[h], off), __shfl_xor(l[h], off)); }
            if (g == 0) { stat[wave][h][j] = make_float2(m[h], l[h]); }
        }
        lds_barrier();
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const float2 other = stat[wave ^ 1][h][j];
            merge(m[h], l[h], other.x, other.y);
            // p = 2^(s log2 e - (m log2 e + log2 l)): the division by the sum rides in the exponent
            poff[h] = l[h] > 0.0f ? -(m[h] * PF_LOG2E + __builtin_amdgcn_logf(l[h])) : -INFINITY;
        }
    }
    if (b_begin + 1 < b_end) { asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
    else { asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
    score_products(b_begin & 1, cur);
    staged_barrier();
    // iteration b: keys of b + 1 and values of b are in LDS, `cur` holds the raw scores of b
    auto block = [&](int b, auto masked_c) {
        if (b + 2 < b_end) { stage_keys(b + 2); }
        if (b + 1 < b_end)
        {
            stage_values(b + 1);
            score_products((b + 1) & 1, next);
        }
        weigh(cur, b, masked_c);
        staged_barrier();
        take_next();
    };
    for (int b = b_begin; b < n_plain; b++) { block(b, std::false_type{}); }
    for (int b = n_plain; b < b_end; b++) { block(b, std::true_type{}); }

    // the two halves of a row's keys meet: statistics first, then one half's sums through LDS
    if constexpr (!WHOLE_ROW)
    {
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            l[h] += __shfl_xor(l[h], 16);
            l[h] += __shfl_xor(l[h], 32);
            if (g == 0) { stat[wave][h][j] = make_float2(m[h], l[h]); }
        }
        lds_barrier();
    }
    float* const sums = (float*)lds + ((wave >> 1) * 32 + j) * RS + 4 * g;
#pragma unroll
    for (int h = 0; h < 2; h++)
    {
        if constexpr (!WHOLE_ROW)
        {
            const float2 other = stat[wave ^ 1][h][j];
            const float top = fmaxf(m[h], other.x), base = top > -INFINITY ? top : 0.0f;
            const float mine = pf_exp2((m[h] - base) * PF_LOG2E);                   // 2^-inf = 0 for a half without a key
            const float sum = l[h] * mine + other.y * pf_exp2((other.x - base) * PF_LOG2E);
            if (RANGE && kh == 0 && g == 0 && tok[h] < n_tokens) { ranges.stats[((size_t)blockIdx.y * n_q + head[h]) * n_tokens + tok[h]] = make_float2(top, sum); }
            const float by = RANGE ? mine : sum > 0.0f ? mine / sum : 0.0f;         // a row of scores of -inf gives 0, as in attn_prefill_kernel
#pragma unroll
            for (int d = 0; d < 8; d++) { out[h][d] *= by; }
        }
        if (kh == 1)
        {
#pragma unroll
            for (int d = 0; d < 8; d++) { *(f32x4*)(sums + h * 16 * RS + 16 * d) = out[h][d]; }
        }
    }
    lds_barrier();
    if (kh == 0)
    {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int d = 0; d < 8; d++)
            {
                f32x4* const at = (f32x4*)(sums + h * 16 * RS + 16 * d);
                *at += out[h][d];
            }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        const int c = (int)threadIdx.x + i * 256, row = c >> 4, at = (c & 15) * 8;
        const int t = t0 + 16 * ((row >> 4) / G) + (row & 15);
        if (t >= n_tokens) { continue; }
        const size_t dst_at = ((size_t)t * n_q + kvh * G + (row >> 4) % G) * 128 + at;
        const f32x4 lo = *(const f32x4*)((const float*)lds + row * RS + at), hi = *(const f32x4*)((const float*)lds + row * RS + at + 4);
        if constexpr (RANGE)
        {
            float* const dst = ranges.partial + (size_t)blockIdx.y * n_tokens * n_q * 128 + dst_at;
            *(f32x4*)dst = lo;
            *(f32x4*)(dst + 4) = hi;
        }
        else { store_bf16x8(y + dst_at, lo, hi); }
    }
}

// Sums of the key ranges of one token, four dims of a head per thread: rescaled to the largest maximum, added in the order of the ranges,
// divided by the sum of the weights, one rounding.  A token has the ranges of its tile.
static __global__ __launch_bounds__(256) void attn_prefill_fused_combine_kernel(const PrefillRanges ranges, uint16_t* __restrict__ y, int n_q, int n_tokens, int pos0, int tile)
{
    const long long slice = (long long)n_tokens * n_q * 128;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < slice / 4; i += (long long)gridDim.x * 256)
    {
        const int t = (int)(i / (n_q * 32)), head = (int)(i / 32 % n_q);
        const int n_blocks = (pos0 + min(t / tile * tile + tile, n_tokens) + PF_KEYS - 1) / PF_KEYS;
        const int n_ranges = (n_blocks + ranges.per - 1) / ranges.per;
        f32x4 sum = { 0.0f, 0.0f, 0.0f, 0.0f };
        float m = -INFINITY, l = 0.0f;
        for (int r0 = 0; r0 < n_ranges; r0 += 8)
        {
            f32x4 part[8];                                      // eight ranges requested at once
            float2 stat[8];
#pragma unroll
            for (int r = 0; r < 8; r++)
            {
                const long long from = min(r0 + r, n_ranges - 1);
                stat[r] = ranges.stats[(from * n_q + head) * n_tokens + t];
                part[r] = *(const f32x4*)(ranges.partial + from * slice + i * 4);
            }
            float top = m;
#pragma unroll
            for (int r = 0; r < 8; r++) { top = fmaxf(top, stat[r].x); }
            const float base = top > -INFINITY ? top : 0.0f;
            const float shrink = pf_exp2((m - base) * PF_LOG2E);
            m = top;
            l *= shrink;
            sum *= shrink;
#pragma unroll
            for (int r = 0; r < 8; r++)
            {
                const float w = r0 + r < n_ranges ? pf_exp2((stat[r].x - base) * PF_LOG2E) : 0.0f;
                if (r0 + r < n_ranges)
                {
                    l += w * stat[r].y;
                    sum += w * part[r];
                }
            }
        }
        const float by = l > 0.0f ? 1.0f / l : 0.0f;
        sum *= by;
        *(u32x2_any*)(y + i * 4) = u32x2{ f32_to_bf16_bits(sum[0]) | (f32_to_bf16_bits(sum[1]) << 16), f32_to_bf16_bits(sum[2]) | (f32_to_bf16_bits(sum[3]) << 16) };      // y may lie on any element
    }
}

}    // namespace ccq
