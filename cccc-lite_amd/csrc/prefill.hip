// C-ABI entry points of the prompt-phase neighbours (kernels in prefill_kernels.h).
#include "../../include/cccc_hip_quant.h"
#include "prefill_fused.h"
#include "runtime.h"
#include <algorithm>
#include <cmath>

using namespace ccq;

namespace
{
inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Sixteen lanes per head from this many heads x tokens on, a wave per head below.  Measured with 12, 32 and 48 heads a token: level at 4600,
// 3600 and 6100 where every access is aligned, and at 9000, 14500 and 14000 where none is.
inline bool rope_rows_wide(long long heads, bool aligned) { return heads >= (aligned ? 5120 : 14336); }

// Key ranges of a prompt's attention.  In one piece a workgroup takes 5 us and 1.75 per block of 64 keys; in n ranges the three launches
// take 16 us, 1.75 per block of one range, and 0.25 per MB of FP32 sums written and read.  At most one workgroup per CU (two take as long
// as one after the other: 64 tokens of 32 / 8 heads behind 4000: 34.5 us with 8 ranges, 43.9 with 12; 300 tokens behind 1000, 152 workgroups:
// 45.6 in one piece, 50.4 in two ranges), and 10 % to gain at least.  One piece without scratch memory, as under graph capture.
// Measured on MI355X, one piece -> ranges: those 64 tokens 121 -> 34.5 us, 64 tokens of 4 / 1 heads behind 14000 424 -> 34, 200 tokens of
// 32 / 8 behind 2000 70 -> 51, 2 tokens of one head behind 16000 353 -> 23.
struct AttentionRanges
{
    int n, per;
};

AttentionRanges attention_ranges(long long tiles, int n_keys, size_t outputs)
{
    const int blocks = (n_keys + PF_KEYS - 1) / PF_KEYS;
    const int want = (int)std::min({ cu_count() / tiles, (long long)PF_RANGES, (long long)blocks / 2 });
    if (want < 2) { return { 1, blocks }; }
    const int per = ((blocks + want - 1) / want + 1) & ~1;
    const int n = (blocks + per - 1) / per;
    const double whole = 5.0 + 1.75 * blocks, split = 16.0 + 1.75 * per + 0.25e-6 * 8.0 * 128.0 * (double)outputs * n;
    return split < 0.9 * whole ? AttentionRanges{ n, per } : AttentionRanges{ 1, blocks };
}

// The same in one pass: 4.5 us and 0.87 per block where a CU has one workgroup, 1.35 for two side by side; ranges add 6 us for the combine launch
// and 0.35 per MB of FP32 sums written and read.  One or two workgroups per CU, whichever the estimate has ahead by 5 %.
// Measured, 1 / 2 / 4 / 8 ranges: 512 tokens of 32 / 8 heads behind 3000 53 / 53 / 57 / 67 us, 256 tokens 47.6 / 35.4 / 36.5 / 38.8, 128 tokens
// 46 / 31.6 / 25.1 / 27.7, 2048 tokens of 4 / 1 behind 4000 83 / 52 / 45 / 52, 700 of 2 / 1 behind 5000 80 / 48 / 30 / 22, 512 of 32 / 8 from 0 12.7
// / 23.9 / 28.2.
AttentionRanges fused_attention_ranges(long long tiles, int n_keys, size_t outputs)
{
    const int blocks = (n_keys + PF_KEYS - 1) / PF_KEYS;
    AttentionRanges best = { 1, blocks };
    double least = 4.5 + blocks * std::max(0.87, 1.35 * (double)tiles / (2.0 * cu_count()));
    for (int side = 1; side <= 2; side++)
    {
        const int want = (int)std::min({ side * cu_count() / tiles, (long long)PF_RANGES, (long long)blocks / 2 });
        if (want < 2) { continue; }
        const int per = ((blocks + want - 1) / want + 1) & ~1;
        const int n = (blocks + per - 1) / per;
        const double time = 10.5 + per * (side == 1 ? 0.87 : 1.35) + 0.35e-6 * 8.0 * 128.0 * (double)outputs * n;
        if (n > 1 && time < 0.95 * least) { least = time; best = { n, per }; }
    }
    return best;
}

// FP32 sums and statistics of the ranges: tiles of 64 rows, `side` workgroups per CU at most (two in one pass, one with whole rows).
char* range_scratch(int side)
{
    constexpr size_t ROW = 128 * sizeof(float) + sizeof(float2);
    return (char*)fixed_scratch((size_t)cu_count() * side * 64 * ROW);
}

bool prefill_args_ok(const void* q, const void* k_cache, const void* v_cache, const void* y, int n_q_heads, int n_kv_heads, int head_dim, int t_kv, int n_tokens, int pos0)
{
    if (head_dim != 128 || n_kv_heads <= 0 || n_q_heads <= 0 || n_q_heads % n_kv_heads != 0 || t_kv <= 0 || n_tokens <= 0) { return false; }
    if (pos0 < 0 || (long long)pos0 + n_tokens > t_kv || n_kv_heads > 65535) { return false; }
    if (!q || !k_cache || !v_cache || !y || !aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache)) { return false; }
    if ((long long)((n_tokens + 15) / 16) * n_kv_heads > 0x7FFFFFFFLL) { return false; }
    // the kernels address cache rows with 32-bit byte offsets inside a KV head (row * 256)
    if ((long long)pos0 + n_tokens > (1LL << 24)) { return false; }
    const int group = n_q_heads / n_kv_heads;
    return group == 1 || group == 2 || group == 4;
}

// attn_prefill_tile_kernel: 64 rows of a kv head per workgroup
template <int FORM>
void launch_tiles(const void* q, const void* k_cache, const void* v_cache, void* y, int n_q_heads, int n_kv_heads, int t_kv, int n_tokens, int pos0, int n_ranges, const PrefillRanges& ranges)
{
    const int group = n_q_heads / n_kv_heads, tile = 64 / group;
    const dim3 grid((unsigned)((long long)((n_tokens + tile - 1) / tile) * n_kv_heads), n_ranges);
    const auto kernel = group == 4 ? attn_prefill_tile_kernel<4, FORM> : group == 2 ? attn_prefill_tile_kernel<2, FORM> : attn_prefill_tile_kernel<1, FORM>;
    kernel<<<grid, 256, 0, stream()>>>((const uint16_t*)q, (const uint16_t*)k_cache, (const uint16_t*)v_cache, (uint16_t*)y, n_q_heads, t_kv, n_tokens, pos0, 1.0f / sqrtf(128.0f), ranges);
}
}    // namespace

int hip_qk_norm_rope_kv_rows_bf16(const void* q, const void* k, const void* v, const void* q_norm_w, const void* k_norm_w,
                                  const void* cos_tab, const void* sin_tab, void* q_out, void* k_cache, void* v_cache,
                                  int n_q_heads, int n_kv_heads, int head_dim, int t_kv, int n_tokens, int pos0, float epsilon)
{
    if (head_dim != 128 || n_q_heads <= 0 || n_kv_heads <= 0 || t_kv <= 0 || n_tokens <= 0 || n_tokens > 65535) { return -1; }
    if (pos0 < 0 || (long long)pos0 + n_tokens > t_kv) { return -1; }
    if (!q || !k || !v || !cos_tab || !sin_tab || !q_out || !k_cache || !v_cache) { return -1; }
    if ((q_norm_w == nullptr) != (k_norm_w == nullptr)) { return -1; }
    const int heads = n_q_heads + 2 * n_kv_heads;
    const bool aligned = (((uintptr_t)q | (uintptr_t)k | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w | (uintptr_t)cos_tab | (uintptr_t)sin_tab | (uintptr_t)q_out | (uintptr_t)k_cache) & 7u) == 0
                         && aligned16(v) && aligned16(v_cache);
    const bool wide = rope_rows_wide((long long)heads * n_tokens, aligned);
    auto* const kernel = wide ? qk_norm_rope_kv_rows_kernel : qk_norm_rope_kv_few_rows_kernel;
    kernel<<<dim3((heads + (wide ? 15 : 3)) / (wide ? 16 : 4), n_tokens), 256, 0, stream()>>>((const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (const uint16_t*)q_norm_w,
                                                                                             (const uint16_t*)k_norm_w, (const uint16_t*)cos_tab, (const uint16_t*)sin_tab,
                                                                                             (uint16_t*)q_out, (uint16_t*)k_cache, (uint16_t*)v_cache, n_q_heads, n_kv_heads, t_kv, pos0, epsilon);
    return finish("qk_norm_rope_kv_rows");
}

int hip_attention_prefill_bf16(const void* q, const void* k_cache, const void* v_cache, void* y,
                               int n_q_heads, int n_kv_heads, int head_dim, int t_kv, int n_tokens, int pos0)
{
    if (!prefill_args_ok(q, k_cache, v_cache, y, n_q_heads, n_kv_heads, head_dim, t_kv, n_tokens, pos0)) { return -1; }
    const long long tiles = (long long)((n_tokens + 15) / 16) * n_kv_heads;
    const int group = n_q_heads / n_kv_heads;
    const float scale = 1.0f / sqrtf(128.0f);
    const size_t outputs = (size_t)n_tokens * n_q_heads;
    const AttentionRanges split = attention_ranges(tiles, pos0 + n_tokens, outputs);
    char* const scratch = split.n > 1 ? range_scratch(1) : nullptr;
    const PrefillRanges ranges = { split.per, (float2*)(scratch + (size_t)split.n * outputs * 128 * sizeof(float)), (float*)scratch };
    const dim3 grid((unsigned)tiles, scratch ? split.n : 1);
#define CCQ_ATTN_PREFILL(G, PASS)                                                                                                                  \
    attn_prefill_kernel<G, PASS><<<grid, 256, 0, stream()>>>((const uint16_t*)q, (const uint16_t*)k_cache, (const uint16_t*)v_cache, (uint16_t*)y, \
                                                             n_q_heads, t_kv, n_tokens, pos0, scale, ranges)
#define CCQ_ATTN_PREFILL_GROUPS(PASS)                                                                                                              \
    group == 4 ? CCQ_ATTN_PREFILL(4, PASS) : group == 2 ? CCQ_ATTN_PREFILL(2, PASS) : CCQ_ATTN_PREFILL(1, PASS)
    // Whole rows in one piece go by tiles of 64 rows, except where one query head per kv head leaves tiles of 16 tokens a CU each: those have two
    // waves on half the rows.  The same bits either way.  4 / 4 heads, 16 tokens -> 64 rows: 1024 tokens (256 tiles of 16) behind 3000 90.1 / 93.6 us,
    // from 0 26.3 / 28.2; 1100 tokens (276) behind 3000 154.7 / 95.2, from 0 33.1 / 30.0.  Two heads 1 to 15 % ahead on 64 rows at any size, four 15 to 30.
    if (pos0 + n_tokens <= PF_SHORT * PF_KEYS) { CCQ_ATTN_PREFILL_GROUPS(3); }
    else if (!scratch && group == 1 && tiles <= cu_count()) { CCQ_ATTN_PREFILL(1, 0); }
    else if (!scratch) { launch_tiles<PF_WHOLE_ROW>(q, k_cache, v_cache, y, n_q_heads, n_kv_heads, t_kv, n_tokens, pos0, 1, ranges); }
    else
    {
        CCQ_ATTN_PREFILL_GROUPS(1);
        CCQ_ATTN_PREFILL_GROUPS(2);
        const long long blocks = ((long long)outputs * 32 + 255) / 256, cap = (long long)cu_count() * 16;
        attn_prefill_combine_kernel<<<(unsigned)(blocks < cap ? blocks : cap), 256, 0, stream()>>>(ranges.partial, (uint16_t*)y, n_q_heads * 128, n_tokens, pos0, split.per);
    }
#undef CCQ_ATTN_PREFILL_GROUPS
#undef CCQ_ATTN_PREFILL
    return finish("attention_prefill");
}

int hip_attention_prefill_fused_bf16(const void* q, const void* k_cache, const void* v_cache, void* y,
                                     int n_q_heads, int n_kv_heads, int head_dim, int t_kv, int n_tokens, int pos0)
{
    if (!prefill_args_ok(q, k_cache, v_cache, y, n_q_heads, n_kv_heads, head_dim, t_kv, n_tokens, pos0)) { return -1; }
    const int tile = 64 * n_kv_heads / n_q_heads;
    const long long tiles = (long long)((n_tokens + tile - 1) / tile) * n_kv_heads;
    const size_t outputs = (size_t)n_tokens * n_q_heads;
    const AttentionRanges split = fused_attention_ranges(tiles, pos0 + n_tokens, outputs);
    char* const scratch = split.n > 1 ? range_scratch(2) : nullptr;
    const PrefillRanges ranges = { split.per, (float2*)(scratch + (size_t)split.n * outputs * 128 * sizeof(float)), (float*)scratch };
    if (!scratch) { launch_tiles<PF_ONE_PASS>(q, k_cache, v_cache, y, n_q_heads, n_kv_heads, t_kv, n_tokens, pos0, 1, ranges); }
    else
    {
        launch_tiles<PF_ONE_PASS_RANGE>(q, k_cache, v_cache, y, n_q_heads, n_kv_heads, t_kv, n_tokens, pos0, split.n, ranges);
        const long long blk = ((long long)outputs * 32 + 255) / 256, cap = (long long)cu_count() * 16;
        attn_prefill_fused_combine_kernel<<<(unsigned)(blk < cap ? blk : cap), 256, 0, stream()>>>(ranges, (uint16_t*)y, n_q_heads, n_tokens, pos0, tile);
    }
    return finish("attention_prefill_fused");
}

int hip_add_bf16(const void* a, const void* b, void* y, unsigned long long n)
{
    if (!a || !b || !y || n == 0 || n % 8 != 0 || !aligned16(a) || !aligned16(b) || !aligned16(y)) { return -1; }
    const long long chunks = (long long)(n / 8);
    const long long blocks = (chunks + 255) / 256, cap = (long long)cu_count() * 16;
    add_rows_kernel<<<(unsigned)(blocks < cap ? blocks : cap), 256, 0, stream()>>>((const u32x4*)a, (const u32x4*)b, (u32x4*)y, chunks);
    return finish("add_bf16");
}

int hip_add_rms_norm_bf16(const void* a, const void* b, void* sum, const void* norm_w, void* y, unsigned int rows, unsigned int inner, float epsilon)
{
    if (!a || !b || !sum || !norm_w || !y || rows == 0 || inner == 0 || inner % 8 != 0 || inner > 64u * 8u * RMS_CHUNKS) { return -1; }
    if (!aligned16(a) || !aligned16(b) || !aligned16(sum) || !aligned16(norm_w) || !aligned16(y)) { return -1; }
    add_rms_norm_rows_kernel<<<(rows + 3) / 4, 256, 0, stream()>>>((const uint16_t*)a, (const uint16_t*)b, (uint16_t*)sum, (const uint16_t*)norm_w,
                                                                   (uint16_t*)y, rows, inner, epsilon);
    return finish("add_rms_norm_bf16");
}

int hip_swiglu_bf16(const void* gate, const void* up, void* y, unsigned long long n)
{
    if (!gate || !up || !y || n == 0 || n % 8 != 0 || !aligned16(gate) || !aligned16(up) || !aligned16(y)) { return -1; }
    const long long chunks = (long long)(n / 8);
    const long long blocks = (chunks + 255) / 256, cap = (long long)cu_count() * 16;
    swiglu_rows_kernel<<<(unsigned)(blocks < cap ? blocks : cap), 256, 0, stream()>>>((const u32x4*)gate, (const u32x4*)up, (u32x4*)y, chunks);
    return finish("swiglu_bf16");
}
