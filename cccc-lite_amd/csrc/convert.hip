// hip_convert / hip_fp4_blockscale_to_bf16 / hip_float_to_fp4_blockscale for gfx950.
//
// Every pair is an HBM-bound stream.  A lane handles as many elements as fill 16 bytes on the wider side of the pair, so
// that both the loads and the stores of a wave are contiguous spans (a lane that stores two or four 16-byte pieces side by
// side touches every line twice or four times), four such pieces are requested before the first is used, and the grid is a
// fixed multiple of the CU count walking the buffer with a grid stride.  Scalar kernels take what is left: the last few
// elements, misaligned pointers, odd block lengths.  Measured on a 4096 x 12288 weight, BF16 -> float -> FP4 with block scales
// -> BF16 (659 MB moved): 113 us, 5.8 TB/s (a large copy reaches 5.4; part of what one pass writes the next reads from the
// memory-side cache); through absmax and float -> FP8 and back 154.
// Numerics follow the reference kernels element for element (decode, one FP32 multiply by the
// scale, integer round-to-nearest-even to BF16): cccc-cuda/cuda_functions.cu:2566-2596 (E4M3),
// :2735-2785 (E5M2), :2834-2884 (FP4), :2896-2960 (FP4 block scale), :3066-3090 (dispatch).
#include "../../include/cccc_hip_quant.h"
#include "quant_device.h"
#include "runtime.h"
#include <algorithm>
#include <hip/hip_fp16.h>

using namespace ccq;

namespace
{

constexpr int kThreads = 256;

inline unsigned grid_for(size_t work_items)
{
    const size_t want = (work_items + kThreads - 1) / kThreads;
    const size_t cap = (size_t)cu_count() * 16;
    return (unsigned)(want < 1 ? 1 : (want > cap ? cap : want));
}

template <int SRC>
__device__ __forceinline__ float decode8(uint32_t b)
{
    return SRC == DT_E5M2 ? e5m2_to_f32(b) : e4m3_to_f32(b);
}

template <int DST>
__device__ __forceinline__ void store_one(void* dst, size_t i, float v)
{
    if (DST == DT_FLOAT) { ((float*)dst)[i] = v; }
    else if (DST == DT_HALF) { ((uint16_t*)dst)[i] = (uint16_t)f32_to_half_bits(v); }
    else { ((uint16_t*)dst)[i] = (uint16_t)f32_to_bf16_bits(v); }
}

// A 16-byte piece of results, PIECE elements from element i0 on (dst 16-byte aligned, i0 a multiple of PIECE)
template <int DST>
constexpr int kPiece = DST == DT_FLOAT ? 4 : 8;

template <int DST>
__device__ __forceinline__ void store_piece(void* dst, size_t i0, const float (&v)[kPiece<DST>])
{
    u32x4 p;
#pragma unroll
    for (int j = 0; j < 4; j++)
    {
        if constexpr (DST == DT_FLOAT) { p[j] = f32_to_bits(v[j]); }
        else
        {
            const uint32_t lo = DST == DT_HALF ? f32_to_half_bits(v[2 * j]) : f32_to_bf16_bits(v[2 * j]);
            const uint32_t hi = DST == DT_HALF ? f32_to_half_bits(v[2 * j + 1]) : f32_to_bf16_bits(v[2 * j + 1]);
            p[j] = lo | (hi << 16);
        }
    }
    *(u32x4*)((char*)dst + i0 * (DST == DT_FLOAT ? 4 : 2)) = p;
}

constexpr int kInFlight = 4;            // pieces a lane requests before it uses the first

// Walks n_pieces pieces with every lane of the grid: load(piece) -> value for up to kInFlight pieces, then use(piece, value).
template <typename Load, typename Use>
__device__ __forceinline__ void stream_pieces(size_t n_pieces, Load load, Use use)
{
    const size_t stride = (size_t)gridDim.x * kThreads;
    size_t v = (size_t)blockIdx.x * kThreads + threadIdx.x;
    for (; v + (kInFlight - 1) * stride < n_pieces; v += kInFlight * stride)
    {
        decltype(load(v)) x[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; u++) { x[u] = load(v + u * stride); }
#pragma unroll
        for (int u = 0; u < kInFlight; u++) { use(v + u * stride, x[u]); }
    }
    for (; v < n_pieces; v += stride) { use(v, load(v)); }
}

// ---- FP8 (1 byte / element) -> FP32 / FP16 / BF16

template <int SRC, int DST>
__global__ __launch_bounds__(kThreads) void dequant8_vec_kernel(const uint8_t* __restrict__ src, void* __restrict__ dst, size_t n_pieces, float scale)
{
    constexpr int P = kPiece<DST>, D = P / 4;
    stream_pieces(n_pieces,
        [&](size_t v) {
            if constexpr (D == 2) { return __builtin_nontemporal_load((const u32x2*)src + v); }
            else { return __builtin_nontemporal_load((const uint32_t*)src + v); }
        },
        [&](size_t v, auto w) {
            float out[P];
#pragma unroll
            for (int i = 0; i < P; i++)
            {
                uint32_t d;
                if constexpr (D == 2) { d = w[i / 4]; } else { d = w; }
                out[i] = decode8<SRC>((d >> (8 * (i & 3))) & 0xFFu) * scale;
            }
            store_piece<DST>(dst, v * P, out);
        });
}

template <int SRC, int DST>
__global__ __launch_bounds__(kThreads) void dequant8_scalar_kernel(const uint8_t* __restrict__ src, void* __restrict__ dst, size_t begin, size_t n, float scale)
{
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t i = begin + (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
    {
        store_one<DST>(dst, i, decode8<SRC>(src[i]) * scale);
    }
}

template <int SRC, int DST>
int launch_dequant8(const void* src, void* dst, unsigned n, float scale, const char* what)
{
    if (n == 0) { return 0; }
    const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15u) == 0;
    const size_t n_pieces = aligned ? (size_t)n / kPiece<DST> : 0;
    if (n_pieces) { dequant8_vec_kernel<SRC, DST><<<grid_for(n_pieces), kThreads, 0, stream()>>>((const uint8_t*)src, dst, n_pieces, scale); }
    const size_t done = n_pieces * kPiece<DST>;
    if (done < n) { dequant8_scalar_kernel<SRC, DST><<<grid_for(n - done), kThreads, 0, stream()>>>((const uint8_t*)src, dst, done, n, scale); }
    return finish(what);
}

// ---- FP4 (two elements / byte) -> FP32 / BF16, per-tensor scale or per-block E4M3 scale

// A piece shares one scale byte when block_size is a multiple of its length (checked by the launcher, which falls back to the
// scalar kernel otherwise); its block is the piece index over the pieces of a block, a 32-bit division (an index is below
// 2^30) that the loads hide: 50 M elements 24 us with blocks of 16, 48 or 1040 alike, 75 us one element per lane.
// The nibbles are decoded by the hardware conversion, two at a time, after code 8 (+0.0 in the reference's table, not -0.0)
// has been cleared: 50 M elements of a 4096 x 12288 weight with the software decoder took 35.5 us, 3.6 TB/s.
template <int DST, bool BLOCKSCALE>
__global__ __launch_bounds__(kThreads) void dequant4_vec_kernel(const uint8_t* __restrict__ src, const uint8_t* __restrict__ scales,
                                                               void* __restrict__ dst, size_t n_pieces, unsigned block_pieces, float scale)
{
    constexpr int P = kPiece<DST>;
    struct Piece { uint32_t w, s; };
    stream_pieces(n_pieces,
        [&](size_t v) {
            Piece p;
            p.w = P == 8 ? __builtin_nontemporal_load((const uint32_t*)src + v) : (uint32_t)__builtin_nontemporal_load((const uint16_t*)src + v);
            p.s = BLOCKSCALE ? scales[(uint32_t)v / block_pieces] : 0u;
            return p;
        },
        [&](size_t v, const Piece& p) {
            const float s = BLOCKSCALE ? e4m3_to_f32(p.s) : scale;
            const uint32_t mag = p.w & 0x77777777u;
            const uint32_t w = mag | (p.w & (mag + 0x77777777u) & 0x88888888u);       // sign bits of the non-zero magnitudes only
            float out[P];
#define CCQ_PAIR(i)                                                                                  \
            if constexpr (2 * (i) < P)                                                               \
            {                                                                                        \
                const f32x2 f = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, i);                \
                out[2 * (i)] = f[0] * s;                                                             \
                out[2 * (i) + 1] = f[1] * s;                                                         \
            }
            CCQ_PAIR(0)
            CCQ_PAIR(1)
            CCQ_PAIR(2)
            CCQ_PAIR(3)
#undef CCQ_PAIR
            store_piece<DST>(dst, v * P, out);
        });
}

template <int DST, bool BLOCKSCALE>
__global__ __launch_bounds__(kThreads) void dequant4_scalar_kernel(const uint8_t* __restrict__ src, const uint8_t* __restrict__ scales,
                                                                  void* __restrict__ dst, size_t begin, size_t n, unsigned block_size, float scale)
{
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t i = begin + (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
    {
        const uint32_t byte = src[i >> 1];
        const uint32_t nib = (i & 1u) ? (byte >> 4) : (byte & 0xFu);
        const float s = BLOCKSCALE ? e4m3_to_f32(scales[i / block_size]) : scale;
        store_one<DST>(dst, i, fp4_to_f32(nib) * s);
    }
}

template <int DST, bool BLOCKSCALE>
int launch_dequant4(const void* src, const void* scales, void* dst, unsigned n, unsigned block_size, float scale, const char* what)
{
    if (n == 0) { return 0; }
    constexpr unsigned P = kPiece<DST>;
    const bool aligned = (((uintptr_t)src & 3u) | ((uintptr_t)dst & 15u)) == 0;
    const bool vec_ok = aligned && (!BLOCKSCALE || block_size % P == 0);
    const size_t n_pieces = vec_ok ? (size_t)n / P : 0;
    if (n_pieces)
    {
        dequant4_vec_kernel<DST, BLOCKSCALE><<<grid_for(n_pieces), kThreads, 0, stream()>>>((const uint8_t*)src, (const uint8_t*)scales, dst, n_pieces, block_size / P, scale);
    }
    const size_t done = n_pieces * P;
    if (done < n)
    {
        dequant4_scalar_kernel<DST, BLOCKSCALE><<<grid_for(n - done), kThreads, 0, stream()>>>((const uint8_t*)src, (const uint8_t*)scales, dst, done, n, block_size, scale);
    }
    return finish(what);
}

// ---- casts and encoders

// Truncating encoders of the reference (cccc-cuda/cuda_functions.cu:2382-2412, :2694-2724, :2796-2832)
__device__ __forceinline__ uint32_t f32_to_e5m2_trunc(float f)
{
    const uint32_t u = f32_to_bits(f);
    const uint32_t mag = u & 0x7FFFFFFFu;
    const uint32_t sign = (u >> 31) << 7;
    if (mag > 0x7F800000u) { return 0x7Cu; }
    if (mag == 0x7F800000u) { return sign | 0x7Cu; }
    const int fe = (int)((u >> 23) & 255u) - 127;
    const uint32_t fm = u & 0x7FFFFFu;
    if (fe > 15 || (fe == 15 && fm >= 0xE00000u)) { return sign | 0x7Bu; }
    const int e8 = fe + 15;
    if (e8 <= 0)
    {
        const int shift = 7 - fe;
        if (shift >= 32) { return sign; }
        return sign | (((fm | 0x800000u) >> shift) & 3u);
    }
    return sign | ((uint32_t)(e8 & 31) << 2) | (fm >> 21);
}

__device__ __forceinline__ uint32_t f32_to_e4m3_trunc(float f)
{
    const uint32_t u = f32_to_bits(f);
    const uint32_t sign = (u >> 31) << 7;
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) { return 0x7Fu; }
    const int fe = (int)((u >> 23) & 255u) - 127;
    const uint32_t fm = u & 0x7FFFFFu;
    if (fe > 8 || (fe == 8 && fm >= 0xC00000u)) { return sign | 0x7Eu; }
    const int e8 = fe + 7;
    if (e8 <= 0)
    {
        const int shift = 14 - fe;
        if (shift >= 32) { return sign; }
        return sign | (((fm | 0x800000u) >> shift) & 7u);
    }
    uint32_t m8 = fm >> 20;
    if (e8 == 15 && m8 == 7u) { m8 = 6u; }
    return sign | ((uint32_t)(e8 & 15) << 3) | m8;
}

__device__ __forceinline__ uint32_t f32_to_fp4(float f)
{
    // the reference's thresholds 0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5, each belonging to the code above it.  From 0.75 on they are the code values'
    // midpoints with one bit of mantissa: half of that bit is added to the magnitude and exponent and bit are the code (the hardware conversion
    // rounds ties to even and cannot be used).  NaN is 7, as no comparison with it holds.
    const uint32_t mag = f32_to_bits(f) & 0x7FFFFFFFu;
    const uint32_t upper = min((mag + 0x200000u) >> 22, 259u) - 252u;
    const float a = fabsf(f);
    const uint32_t lower = a < 0.25f ? 0u : a < 0.75f ? 1u : 2u;
    return (f < 0.0f ? 8u : 0u) | (a < 1.0f ? lower : upper);
}

__device__ __forceinline__ float load_plain(const void* src, int type, size_t i)
{
    if (type == DT_FLOAT) { return ((const float*)src)[i]; }
    if (type == DT_HALF) { return (float)((const _Float16*)src)[i]; }
    return bf16_bits_to_f32(((const uint16_t*)src)[i]);
}

__device__ __forceinline__ uint32_t cast_bits(float v, int dst_type)
{
    if (dst_type == DT_HALF) { return f32_to_half_bits(v); }
    return (v != v) ? ((f32_to_bits(v) >> 16) | 0x40u) : f32_to_bf16_bits(v);
}

// Plain casts (no scale): float->bf16, half->float, half->bf16, bf16->float, bf16->half.
// BF16 results round to nearest even; NaN inputs stay NaN (quiet bit forced).  One element per lane: the last few and
// misaligned pointers (2^24 misaligned floats to BF16 18.2 us; with the types as
// run-time arguments 21.7).
template <int SRC, int DST>
__global__ __launch_bounds__(kThreads) void cast_kernel(const void* __restrict__ src, void* __restrict__ dst, size_t begin, size_t n)
{
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t i = begin + (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
    {
        const float v = load_plain(src, SRC, i);
        if constexpr (DST == DT_FLOAT) { ((float*)dst)[i] = v; }
        else { ((uint16_t*)dst)[i] = (uint16_t)cast_bits(v, DST); }
    }
}

// Four consecutive values of a plain type as floats: one 16-byte or 8-byte load
template <int SRC>
struct Quad
{
    typedef u32x2 raw;
    __device__ static float at(const raw& r, int i)
    {
        const uint32_t h = (r[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
        return SRC == DT_HALF ? half_bits_to_f32(h) : bf16_bits_to_f32(h);
    }
};
template <>
struct Quad<DT_FLOAT>
{
    typedef u32x4 raw;
    __device__ static float at(const raw& r, int i) { return bits_to_f32(r[i]); }
};

// The same casts, four elements per lane and step (4096 x 12288 BF16 -> float: 95 us one element at a time).
template <int SRC, int DST>
__global__ __launch_bounds__(kThreads) void cast_vec_kernel(const void* __restrict__ src, void* __restrict__ dst, size_t n_quads)
{
    stream_pieces(n_quads,
        [&](size_t v) { return __builtin_nontemporal_load((const typename Quad<SRC>::raw*)src + v); },
        [&](size_t v, const typename Quad<SRC>::raw& r) {
            if constexpr (DST == DT_FLOAT)
            {
                ((f32x4*)dst)[v] = f32x4{ Quad<SRC>::at(r, 0), Quad<SRC>::at(r, 1), Quad<SRC>::at(r, 2), Quad<SRC>::at(r, 3) };
            }
            else
            {
                uint32_t b[4];
#pragma unroll
                for (int i = 0; i < 4; i++) { b[i] = cast_bits(Quad<SRC>::at(r, i), DST); }
                ((u32x2*)dst)[v] = u32x2{ b[0] | (b[1] << 16), b[2] | (b[3] << 16) };
            }
        });
}

template <int SRC, int DST>
int launch_cast(const void* src, void* dst, unsigned n)
{
    const bool aligned = (((uintptr_t)src | (uintptr_t)dst) & 15u) == 0;
    const size_t n_quads = aligned ? (size_t)n / 4 : 0;
    if (n_quads) { cast_vec_kernel<SRC, DST><<<grid_for(n_quads), kThreads, 0, stream()>>>(src, dst, n_quads); }
    const size_t done = n_quads * 4;
    if (done < n) { cast_kernel<SRC, DST><<<grid_for(n - done), kThreads, 0, stream()>>>(src, dst, done, n); }
    return finish("convert_cast");
}

// Quantising casts: float|bf16 -> e4m3, float -> e5m2 (value * scale, truncating encoders).
template <int DST>
__device__ __forceinline__ uint32_t encode8(float v) { return DST == DT_E5M2 ? f32_to_e5m2_trunc(v) : f32_to_e4m3_trunc(v); }

template <int SRC, int DST>
__global__ __launch_bounds__(kThreads) void encode8_kernel(const void* __restrict__ src, uint8_t* __restrict__ dst, size_t begin, size_t n, float scale)
{
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t i = begin + (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) { dst[i] = (uint8_t)encode8<DST>(load_plain(src, SRC, i) * scale); }
}

template <int SRC, int DST>
__global__ __launch_bounds__(kThreads) void encode8_vec_kernel(const void* __restrict__ src, uint8_t* __restrict__ dst, size_t n_quads, float scale)
{
    stream_pieces(n_quads,
        [&](size_t v) { return __builtin_nontemporal_load((const typename Quad<SRC>::raw*)src + v); },
        [&](size_t v, const typename Quad<SRC>::raw& r) {
            uint32_t w = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) { w |= encode8<DST>(Quad<SRC>::at(r, i) * scale) << (8 * i); }
            ((uint32_t*)dst)[v] = w;
        });
}

template <int SRC, int DST>
int launch_encode8(const void* src, void* dst, unsigned n, float scale)
{
    const bool aligned = (((uintptr_t)src & 15u) | ((uintptr_t)dst & 3u)) == 0;
    const size_t n_quads = aligned ? (size_t)n / 4 : 0;
    if (n_quads) { encode8_vec_kernel<SRC, DST><<<grid_for(n_quads), kThreads, 0, stream()>>>(src, (uint8_t*)dst, n_quads, scale); }
    const size_t done = n_quads * 4;
    if (done < n) { encode8_kernel<SRC, DST><<<grid_for(n - done), kThreads, 0, stream()>>>(src, (uint8_t*)dst, done, n, scale); }
    return finish("convert_to_fp8");
}

// float -> packed FP4 with a per-tensor scale; one lane per output byte.
__global__ __launch_bounds__(kThreads) void encode4_kernel(const float* __restrict__ src, uint8_t* __restrict__ dst, size_t n, float scale)
{
    const size_t n_bytes = (n + 1) / 2;
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t b = (size_t)blockIdx.x * kThreads + threadIdx.x; b < n_bytes; b += stride)
    {
        const size_t e0 = 2 * b;
        const uint32_t lo = f32_to_fp4(src[e0] * scale);
        const uint32_t hi = (e0 + 1 < n) ? f32_to_fp4(src[e0 + 1] * scale) : 0u;
        dst[b] = (uint8_t)(lo | (hi << 4));
    }
}

// float -> FP4 nibbles + truncating E4M3 dequant scale per block; one lane per block, blocks first_block and up.
__global__ __launch_bounds__(kThreads) void encode4_blockscale_kernel(const float* __restrict__ src, uint8_t* __restrict__ nibbles, uint8_t* __restrict__ scales,
                                                                     size_t first_block, size_t n, unsigned block_size)
{
    const size_t n_blocks = (n + block_size - 1) / block_size;
    const size_t stride = (size_t)gridDim.x * kThreads;
    for (size_t b = first_block + (size_t)blockIdx.x * kThreads + threadIdx.x; b < n_blocks; b += stride)
    {
        const size_t lo = b * block_size;
        const size_t hi = (lo + block_size < n) ? lo + block_size : n;
        float amax = 0.0f;
        for (size_t i = lo; i < hi; i++) { amax = fmaxf(amax, fabsf(src[i])); }
        const float fwd = (amax > 1e-10f) ? (6.0f / amax) : 1.0f;
        const float dq = (amax > 1e-10f) ? (amax / 6.0f) : 1.0f;
        scales[b] = (uint8_t)f32_to_e4m3_trunc(dq);
        for (size_t i = lo; i < hi; i += 2)
        {
            const uint32_t l = f32_to_fp4(src[i] * fwd);
            const uint32_t h = (i + 1 < n) ? f32_to_fp4(src[i + 1] * fwd) : 0u;
            nibbles[i >> 1] = (uint8_t)(l | (h << 4));
        }
    }
}

// Whole blocks of 16 or 32 elements: BLOCK / 4 neighbouring lanes share a block, each with one 16-byte load, and find its
// largest magnitude through lane exchanges inside their row of 16.  One lane per block read 64 bytes at a stride of 64, twice:
// 254 us for a 4096 x 12288 weight (234 MB, 0.9 TB/s).
template <int BLOCK>
__device__ __forceinline__ float block_absmax(const f32x4& x)
{
    float m = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
    m = fmaxf(m, dpp_f32<0xB1>(m));                                                   // quad_perm [1,0,3,2]
    m = fmaxf(m, dpp_f32<0x4E>(m));                                                   // quad_perm [2,3,0,1]
    if (BLOCK == 32) { m = fmaxf(m, dpp_f32<0x141>(m)); }                             // row_half_mirror
    return m;
}

__device__ __forceinline__ uint16_t encode4(const f32x4& x, float f)
{
    return (uint16_t)(f32_to_fp4(x[0] * f) | (f32_to_fp4(x[1] * f) << 4) | (f32_to_fp4(x[2] * f) << 8) | (f32_to_fp4(x[3] * f) << 12));
}

// One piece per lane, up to as many as the grid has lanes (4 M floats on 256 CUs): bound by one trip to memory, every lane divides for itself.
// 1 M floats 2.8 us, 4 M 5.5; with four pieces per lane, three of them past the end, 3.4 and 7.8, on a quarter of the workgroups 3.3 and 6.6.
template <int BLOCK>
__global__ __launch_bounds__(kThreads) void encode4_blockscale_piece_kernel(const float* __restrict__ src, uint8_t* __restrict__ nibbles, uint8_t* __restrict__ scales,
                                                                           size_t n_quads)
{
    constexpr int LANES = BLOCK / 4;
    const size_t v = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (v >= n_quads) { return; }               // whole groups of lanes: n_quads is a multiple of LANES
    const f32x4 x = __builtin_nontemporal_load((const f32x4*)src + v);
    const float amax = block_absmax<BLOCK>(x);
    ((uint16_t*)nibbles)[v] = encode4(x, (amax > 1e-10f) ? (6.0f / amax) : 1.0f);
    if (v % LANES == 0) { scales[v / LANES] = (uint8_t)f32_to_e4m3_trunc((amax > 1e-10f) ? (amax / 6.0f) : 1.0f); }
}

// More: a lane has four pieces, of four blocks; lane u of every quad takes the two divisions and the scale byte of block u and the others get the
// factor through a lane exchange (4096 x 12288 floats 45 us, 5.1 TB/s; 51 with every lane dividing for itself and seven comparisons per code).
// The pieces are walked from the last to the first: what a cast or another pass has just written last is still in the memory-side cache.
template <int BLOCK>
__global__ __launch_bounds__(kThreads) void encode4_blockscale_vec_kernel(const float* __restrict__ src, uint8_t* __restrict__ nibbles, uint8_t* __restrict__ scales,
                                                                         size_t n_quads)
{
    constexpr int LANES = BLOCK / 4;
    static_assert(kInFlight == 4, "a piece per lane of a quad");
    const size_t stride = (size_t)gridDim.x * kThreads;
    const size_t rounds = (n_quads + 4 * stride - 1) / (4 * stride);
    const uint32_t q = threadIdx.x & 3u;
    for (size_t r = rounds; r-- > 0;)
    {
        // a group of lanes is complete in every step: n_quads is a multiple of LANES, and so are the stride and a group's first lane
        const size_t v = r * 4 * stride + (size_t)blockIdx.x * kThreads + threadIdx.x;
        f32x4 x[4];
        float amax[4];
#pragma unroll
        for (int u = 0; u < 4; u++) { x[u] = __builtin_nontemporal_load((const f32x4*)src + (v + u * stride < n_quads ? v + u * stride : n_quads - LANES + threadIdx.x % LANES)); }
#pragma unroll
        for (int u = 0; u < 4; u++) { amax[u] = block_absmax<BLOCK>(x[u]); }
        const float mine = q < 2u ? (q == 0u ? amax[0] : amax[1]) : (q == 2u ? amax[2] : amax[3]);
        const float fwd = (mine > 1e-10f) ? (6.0f / mine) : 1.0f;
        const size_t at = v + q * stride;                                             // a piece of the lane's block
        if (at < n_quads && (LANES == 4 || (threadIdx.x & 4u) == 0u)) { scales[at / LANES] = (uint8_t)f32_to_e4m3_trunc((mine > 1e-10f) ? (mine / 6.0f) : 1.0f); }
        const float f[4] = { dpp_f32<0x00>(fwd), dpp_f32<0x55>(fwd), dpp_f32<0xAA>(fwd), dpp_f32<0xFF>(fwd) };      // lane u of the quad
#pragma unroll
        for (int u = 0; u < 4; u++)
        {
            const uint16_t w = encode4(x[u], f[u]);
            if (v + u * stride < n_quads) { ((uint16_t*)nibbles)[v + u * stride] = w; }
        }
    }
}

// Largest magnitude.  16-byte loads from the first 16-byte boundary on (scalar loads in front of it, behind the last one and for a pointer off
// its elements), four in flight per lane, wave reduction through lane exchanges, the sixteen waves of a workgroup through LDS, then at
// most one atomic per workgroup on the bit pattern (non-negative floats order like unsigned integers) -- and none when the value
// already stored is at least as large.  Atomics on one address are served one after the other and most workgroups start before the
// first has ended: one workgroup per CU at most, of 1024 threads.  Up to 32 K floats one workgroup, which stores its result itself.
//   us, with the launch that clears the result: 20 K floats 3.7, 1 M 6.4, 16 M 13.1, 50 M 31.3, the same one element off their 16
// bytes (up to sixteen workgroups of 256 threads per CU and a memset: 5.7, 18.5, 26.2, 36.7 and off their 16 bytes 50.4 for 50 M).
// From the last piece to the first: what a cast has just written last is still in the memory-side cache, and the encoder that
// follows begins where this ends.  NaN inputs are skipped by fmaxf.
constexpr int kMaxThreads = 1024;

static __global__ void absmax_clear_kernel(unsigned int* out) { *out = 0u; }

template <int SRC>
__global__ __launch_bounds__(kMaxThreads) void absmax_kernel(const void* __restrict__ src, size_t n, unsigned int* __restrict__ out)
{
    __shared__ float part[kMaxThreads / 64];
    const size_t stride = (size_t)gridDim.x * kMaxThreads;
    const size_t first = (size_t)blockIdx.x * kMaxThreads + threadIdx.x;
    constexpr size_t PER = SRC == DT_FLOAT ? 4 : 8;             // elements per 16-byte load
    // elements in front of the first 16-byte boundary; none is whole where the pointer is off its elements
    constexpr size_t SIZE = 16 / PER;
    const size_t head = min((size_t)(-(uintptr_t)src & 15u) / SIZE, n);
    const size_t n_vec = (uintptr_t)src % SIZE == 0 ? (n - head) / PER : 0;
    const u32x4* const body = (const u32x4*)((const uint8_t*)src + head * SIZE);
    float m = 0.0f;
    auto take = [&](const u32x4& v) {
#pragma unroll
        for (int d = 0; d < 4; d++)
        {
            if constexpr (SRC == DT_FLOAT) { m = fmaxf(m, fabsf(bits_to_f32(v[d]))); }
            else { m = fmaxf(m, fmaxf(fabsf(act_bits_to_f32<SRC>(v[d] & 0xFFFFu)), fabsf(act_bits_to_f32<SRC>(v[d] >> 16)))); }
        }
    };
    size_t rounds = n_vec / stride;                             // whole ones; the rest is at the end and comes first
    if (rounds * stride + first < n_vec) { take(body[rounds * stride + first]); }
    for (; rounds % 4; rounds--) { take(body[(rounds - 1) * stride + first]); }
    for (; rounds; rounds -= 4)
    {
        u32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) { v[u] = body[(rounds - 1 - u) * stride + first]; }
#pragma unroll
        for (int u = 0; u < 4; u++) { take(v[u]); }
    }
    for (size_t i = first; i < n - n_vec * PER; i += stride) { m = fmaxf(m, fabsf(load_plain(src, SRC, i < head || n_vec == 0 ? i : i + n_vec * PER))); }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) { m = fmaxf(m, __shfl_xor(m, off)); }
    if ((threadIdx.x & 63) == 0) { part[threadIdx.x >> 6] = m; }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        for (int w = 1; w < kMaxThreads / 64; w++) { m = fmaxf(m, part[w]); }
        const unsigned int bits = f32_to_bits(m);
        if (gridDim.x == 1) { *out = bits; }
        else if (bits > __atomic_load_n(out, __ATOMIC_RELAXED)) { atomicMax(out, bits); }
    }
}

}    // namespace

int hip_absmax(const void* src, int src_type, unsigned int n, void* d_result)
{
    if (src_type != DT_FLOAT && src_type != DT_HALF && src_type != DT_BF16) { return -1; }
    if (!d_result) { return -1; }
    // one workgroup up to eight pieces a lane, which writes its result without a launch that clears it
    const size_t want = ((size_t)n / (src_type == DT_FLOAT ? 4 : 8) + kMaxThreads - 1) / kMaxThreads;
    const unsigned grid = want <= 8 ? 1u : (unsigned)std::min(want, (size_t)cu_count());
    if (grid > 1) { absmax_clear_kernel<<<1, 1, 0, stream()>>>((unsigned int*)d_result); }
    if (src_type == DT_FLOAT) { absmax_kernel<DT_FLOAT><<<grid, kMaxThreads, 0, stream()>>>(src, n, (unsigned int*)d_result); }
    else if (src_type == DT_HALF) { absmax_kernel<DT_HALF><<<grid, kMaxThreads, 0, stream()>>>(src, n, (unsigned int*)d_result); }
    else { absmax_kernel<DT_BF16><<<grid, kMaxThreads, 0, stream()>>>(src, n, (unsigned int*)d_result); }
    return finish("absmax");
}

int hip_convert(const void* src, int src_type, void* dst, int dst_type, unsigned int n, float scale)
{
    if (src_type == dst_type && scale == 1.0f)
    {
        if (n == 0) { return 0; }
        const hipError_t err = hipMemcpyAsync(dst, src, (size_t)n, hipMemcpyDeviceToDevice, stream());
        if (err != hipSuccess)
        {
            fprintf(stderr, "convert copy failed: %s\n", hipGetErrorString(err));
            return 1;
        }
        return finish("convert");
    }
    if ((unsigned)src_type >= 7u || (unsigned)dst_type >= 7u) { return -1; }
    const int pair = src_type * 8 + dst_type;
    switch (pair)
    {
    case DT_E5M2 * 8 + DT_BF16: return launch_dequant8<DT_E5M2, DT_BF16>(src, dst, n, scale, "fp8e5m2_to_bf16");
    case DT_E5M2 * 8 + DT_FLOAT: return launch_dequant8<DT_E5M2, DT_FLOAT>(src, dst, n, scale, "fp8e5m2_to_float");
    case DT_E5M2 * 8 + DT_HALF: return launch_dequant8<DT_E5M2, DT_HALF>(src, dst, n, scale, "fp8e5m2_to_half");
    case DT_E4M3 * 8 + DT_BF16: return launch_dequant8<DT_E4M3, DT_BF16>(src, dst, n, scale, "fp8e4m3_to_bf16");
    case DT_E4M3 * 8 + DT_FLOAT: return launch_dequant8<DT_E4M3, DT_FLOAT>(src, dst, n, scale, "fp8e4m3_to_float");
    case DT_E4M3 * 8 + DT_HALF: return launch_dequant8<DT_E4M3, DT_HALF>(src, dst, n, scale, "fp8e4m3_to_half");
    case DT_FP4 * 8 + DT_BF16: return launch_dequant4<DT_BF16, false>(src, nullptr, dst, n, 1, scale, "fp4_to_bf16");
    case DT_FP4 * 8 + DT_FLOAT: return launch_dequant4<DT_FLOAT, false>(src, nullptr, dst, n, 1, scale, "fp4_to_float");
    case DT_FLOAT * 8 + DT_BF16: return launch_cast<DT_FLOAT, DT_BF16>(src, dst, n);
    case DT_HALF * 8 + DT_FLOAT: return launch_cast<DT_HALF, DT_FLOAT>(src, dst, n);
    case DT_HALF * 8 + DT_BF16: return launch_cast<DT_HALF, DT_BF16>(src, dst, n);
    case DT_BF16 * 8 + DT_FLOAT: return launch_cast<DT_BF16, DT_FLOAT>(src, dst, n);
    case DT_BF16 * 8 + DT_HALF: return launch_cast<DT_BF16, DT_HALF>(src, dst, n);
    case DT_FLOAT * 8 + DT_E4M3: return launch_encode8<DT_FLOAT, DT_E4M3>(src, dst, n, scale);
    case DT_FLOAT * 8 + DT_E5M2: return launch_encode8<DT_FLOAT, DT_E5M2>(src, dst, n, scale);
    case DT_BF16 * 8 + DT_E4M3: return launch_encode8<DT_BF16, DT_E4M3>(src, dst, n, scale);
    case DT_FLOAT * 8 + DT_FP4:
        if (n) { encode4_kernel<<<grid_for((n + 1) / 2), kThreads, 0, stream()>>>((const float*)src, (uint8_t*)dst, n, scale); }
        return finish("float_to_fp4");
    default: return -1;
    }
}

int hip_fp4_blockscale_to_bf16(const void* src_nibbles, const void* src_scales, void* dst, unsigned int n_elems, unsigned int block_size)
{
    if (block_size == 0 || !src_scales) { return -1; }
    return launch_dequant4<DT_BF16, true>(src_nibbles, src_scales, dst, n_elems, block_size, 1.0f, "fp4_blockscale_to_bf16");
}

int hip_float_to_fp4_blockscale(const void* src, void* dst_nibbles, void* dst_scales, unsigned int n_elems, unsigned int block_size)
{
    if (block_size == 0 || (block_size & 1u)) { return -1; }
    if (n_elems == 0) { return 0; }
    const size_t n_blocks = ((size_t)n_elems + block_size - 1) / block_size;
    const bool vec_ok = (((uintptr_t)src & 15u) | ((uintptr_t)dst_nibbles & 1u)) == 0 && (block_size == 16 || block_size == 32);
    const size_t whole = vec_ok ? (size_t)n_elems / block_size : 0;                 // complete blocks
    const size_t n_quads = whole * block_size / 4;
    if (whole)
    {
        const bool one = n_quads <= (size_t)cu_count() * 16 * kThreads;
        auto* const kernel = block_size == 16 ? (one ? encode4_blockscale_piece_kernel<16> : encode4_blockscale_vec_kernel<16>)
                                              : (one ? encode4_blockscale_piece_kernel<32> : encode4_blockscale_vec_kernel<32>);
        kernel<<<grid_for(one ? n_quads : (n_quads + 3) / 4), kThreads, 0, stream()>>>((const float*)src, (uint8_t*)dst_nibbles, (uint8_t*)dst_scales, n_quads);
    }
    if (whole < n_blocks)
    {
        encode4_blockscale_kernel<<<grid_for(n_blocks - whole), kThreads, 0, stream()>>>((const float*)src, (uint8_t*)dst_nibbles, (uint8_t*)dst_scales, whole, n_elems, block_size);
    }
    return finish("float_to_fp4_blockscale");
}
