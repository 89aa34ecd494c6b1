// C-ABI entry points of the prompt-phase neighbours (kernels in prefill_kernels.h).
#include "../../include/cccc_hip_quant.h"
#include "prefill_kernels.h"
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
    if (head_dim != 128 || n_kv_heads <= 0 || n_q_heads <= 0 || n_q_heads % n_kv_heads != 0 || t_kv <= 0 || n_tokens <= 0) { return -1; }
    if (pos0 < 0 || (long long)pos0 + n_tokens > t_kv || n_kv_heads > 65535) { return -1; }
    if (!q || !k_cache || !v_cache || !y || !aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache)) { return -1; }
    if ((long long)((n_tokens + 15) / 16) * n_kv_heads > 0x7FFFFFFFLL) { return -1; }
    // the kernel addresses cache rows with 32-bit byte offsets inside a KV head (row * 256)
    if ((long long)pos0 + n_tokens > (1LL << 24)) { return -1; }
    const long long tiles = (long long)((n_tokens + 15) / 16) * n_kv_heads;
    const int group = n_q_heads / n_kv_heads;
    if (group != 1 && group != 2 && group != 4) { return -1; }
    const float scale = 1.0f / sqrtf(128.0f);
    const size_t outputs = (size_t)n_tokens * n_q_heads;
    const AttentionRanges split = attention_ranges(tiles, pos0 + n_tokens, outputs);
    // ranges x tiles is at most the number of CUs, and a tile is 16 tokens of at most four heads
    constexpr size_t ROW = 128 * sizeof(float) + sizeof(float2);
    char* const scratch = split.n > 1 ? (char*)fixed_scratch((size_t)cu_count() * 16 * 4 * ROW) : nullptr;
    const PrefillRanges ranges = { split.per, (float2*)(scratch + (size_t)split.n * outputs * 128 * sizeof(float)), (float*)scratch };
    const dim3 grid((unsigned)tiles, scratch ? split.n : 1);
#define CCQ_ATTN_PREFILL(G, PASS)                                                                                                                  \
    attn_prefill_kernel<G, PASS><<<grid, 256, 0, stream()>>>((const uint16_t*)q, (const uint16_t*)k_cache, (const uint16_t*)v_cache, (uint16_t*)y, \
                                                             n_q_heads, t_kv, n_tokens, pos0, scale, ranges)
#define CCQ_ATTN_PREFILL_GROUPS(PASS)                                                                                                              \
    group == 4 ? CCQ_ATTN_PREFILL(4, PASS) : group == 2 ? CCQ_ATTN_PREFILL(2, PASS) : CCQ_ATTN_PREFILL(1, PASS)
    if (pos0 + n_tokens <= PF_SHORT * PF_KEYS) { CCQ_ATTN_PREFILL_GROUPS(3); }
    else if (!scratch) { CCQ_ATTN_PREFILL_GROUPS(0); }
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
