// Which tile and how many k ranges a prompt GEMM takes (gemm_kernels.h has the kernels): host arithmetic on the shape, no
// device state.  A tile is 16 mb tokens x 64 nb features for one workgroup of 256 threads.
#pragma once
#include "linear_args.h"
#include <algorithm>
#include <math.h>

namespace ccq
{

enum GemmKind { GEMM_LINEAR, GEMM_PAIR, GEMM_SEGMENTS };

struct GemmWeights
{
    bool fp4, row_major, scaled;      // FP4 reads tiled copies only; scaled: an FP8 weight with a scale (any of a launch's)
};

struct GemmPlan
{
    int mb, nb, splits;
    bool small;              // FP8: a tile with weights requested three k-tiles ahead (gemm_short.h); FP4: gemm_short_fp4.hip
    int ranges;              // k ranges of the larger tile that this plan was compared with, and so of the scratch held: splits <= ranges
    bool staged = false;     // FP8: gemm_staged_kernel (gemm_staged.h), a tile of kStagedTiles; `small` is set as well
};

// Tile shape and k split of the larger tiles (tuned on MI355X with the FP8 kernel): a workgroup owns 64 NB features x
// 16 MB tokens.  A CU wants two resident workgroups (one alone reaches ~85 % of the rate), the workgroups should spread
// evenly over the CUs (384 tiles on 256 CUs leave half of them with twice the work: 36 % of peak where 512 even tiles
// reach 42 %), and 48-feature waves with 64-token tiles cost ~5 % against the larger tiles.  Too few tiles in every
// shape: the k range is split over workgroups (256-feature tiles, about one workgroup per CU, 1024 elements of k or more
// each; 512 or more up to 64 tokens) and a second kernel adds the partial sums.
//
// fp4: the FP4 kernel's costs -- the 128-token x 256-feature tile stays out of the scoring (see large_fp4), and
// 64-token tiles pay for converting every weight for half as many products (913 against 1037 TFLOP/s at equal balance).
// row_major (FP8 only): the weight is read from the file layout, where a wave's load is sixteen half cache lines; 64-token
// tiles then pay that fetch for half as many products, and a 128-token tile is worth having even at one workgroup per CU
// (4096 x 4096 at 2048 tokens: 70 us against 91; K 12288: 196 against 244; on the tiled copy the two are level).
// 64 tokens x 128 features (FP8, K < 8192, at most 2048 features) puts 256 or more workgroups on outputs as narrow as 1024
// features (2048 tokens: 29 / 35 us tiled / row-major against 33 / 40).  Wider outputs with few tiles keep the k split: with
// a long K it is far ahead (K 12288 at 512 tokens: 60 against 110 us), and on 512 tokens x 4096 x 4096, where the two
// measure the same on weights that rotate through the memory-side cache, the split is 8 us ahead inside a whole model.
inline GemmPlan large_linear(const LinearArgs& a, const GemmWeights& w, int cus, bool scratch)
{
    struct Shape { int nb, mb; double quality; };
    const double q64 = w.row_major ? 0.8 : 1.0;          // what a 64-token tile is worth against a 128-token one
    const Shape shapes[] = { { 4, 8, 1.0 }, { 4, 4, w.fp4 ? 0.88 : q64 }, { 3, 8, 1.0 }, { 3, 4, w.fp4 ? 0.84 : 0.95 * q64 }, { 2, 4, 0.9 * q64 } };
    GemmPlan plan = { 4, 4, 1, false, 1 };
    double best = -1.0;
    for (const Shape& sh : shapes)
    {
        if (sh.nb == 2 && (w.fp4 || a.K >= 8192 || a.n_out > 2048)) { continue; }
        if (sh.mb == 8 && (a.tokens <= 64 || (sh.nb == 4 && w.fp4))) { continue; }
        const long long tiles = (long long)((a.n_out + 64 * sh.nb - 1) / (64 * sh.nb)) * ((a.tokens + 16 * sh.mb - 1) / (16 * sh.mb));
        const double balance = (double)tiles / (double)(((tiles + cus - 1) / cus) * cus);
        double occupancy = tiles >= 2LL * cus ? 1.0 : (tiles > cus ? 0.95 : 0.85);
        // one 128 x 256 tile on (nearly) every CU and a long K: ahead of two 64-token tiles per CU, which convert every weight
        // twice (2048 tokens x 4096 features, K 12288, tiled copy: 160 against 168-170 us; K 4096: level)
        if (sh.nb == 4 && sh.mb == 8 && !w.row_major && a.K >= 8192 && tiles * 8 > 7LL * cus && tiles <= cus) { occupancy = 1.02; }
        const double score = sh.quality * balance * occupancy;
        if (score > best + 1e-9)
        {
            best = score;
            plan.nb = sh.nb;
            plan.mb = sh.mb;
        }
    }
    const long long n_tiles = (a.n_out + 255) / 256;
    const long long tiles8 = n_tiles * ((a.tokens + 127) / 128), tiles4 = n_tiles * ((a.tokens + 63) / 64);
    if (scratch && best < 0.6 && tiles4 * 4 < 5LL * cus && a.n_out % 4 == 0)
    {
        const long long base = a.tokens > 64 ? tiles8 : tiles4;
        // up to 64 tokens the weight bytes bound the launch and finer k ranges put more workgroups on them (32 tokens:
        // 4096 x 4096 17.3 -> 14.6 us, 1024 x 4096 16.3 -> 13.5, 4096 x 12288 28.5 -> 24.0); above that the FP32 partial
        // sums weigh more and a range keeps 1024 elements of k or more
        const long long s = std::min({ (cus + base / 2) / base, a.tokens <= 64 ? 16LL : 8LL, (long long)a.K / (a.tokens <= 64 ? 512 : 1024) });
        if (s > 1)
        {
            plan.splits = (int)s;
            plan.nb = 4;
            plan.mb = a.tokens > 64 ? 8 : (a.tokens > 32 || w.fp4 ? 4 : 2);        // FP8, up to 32 tokens: a 32-token tile
        }
    }
    return plan;
}

// FP4: the 128 x 256 tile needs the register file of a whole SIMD per wave, so a CU runs one such workgroup at a time
// and nothing hides its prologue and epilogue: it pays when every tile gets a CU of its own (1009 TFLOP/s on
// 2048 x 4096, K 14336, against 940 for 64 x 256 tiles; 767 against 1009 for 128 x 192 tiles on 2048 x 14336, where a CU
// runs three or four of them in sequence), with the k range split when the tiles are few.
inline GemmPlan large_fp4(const LinearArgs& a, const GemmWeights& w, int cus, bool scratch)
{
    const long long tiles = (long long)((a.n_out + 255) / 256) * ((a.tokens + 127) / 128);
    if (a.tokens > 64 && tiles <= cus)
    {
        const long long s = std::max(1LL, a.n_out % 4 == 0 ? std::min({ (cus + tiles / 2) / tiles, 8LL, (long long)a.K / 1024 }) : 1LL);
        if (tiles * s * 5 >= 3LL * cus) { return GemmPlan{ 8, 4, scratch ? (int)s : 1, false, 1 }; }
    }
    return large_linear(a, w, cus, scratch);
}

// k ranges of a joint or paired launch of `base` tiles: as many as leave one workgroup per CU, 512 elements of k or more each
inline int joint_splits(const LinearArgs& a, int cus, long long base, int most, bool by4, bool scratch)
{
    return scratch && by4 ? (int)std::max(1LL, std::min({ cus / base, (long long)most, (long long)a.K / 512 })) : 1;
}

// up to three linears on the same activations in one launch: 64- or 128-token x 256-feature tiles, whichever gives the CUs
// two rounds of workgroups or more evenly; few tiles (q, k, v of a 4096-wide model are 24 feature tiles): the k range split,
// every segment's partial sums laid out as its own split GEMM one after the other, and one combine launch for all
inline GemmPlan large_segments(const LinearArgs& a, const GemmWeights& w, int cus, bool scratch)
{
    long long n_tiles = 0;
    bool by4 = true;
    for (int s = 0; s < a.n_segments; s++)
    {
        n_tiles += (a.seg_n_out[s] + 255) / 256;
        by4 = by4 && a.seg_n_out[s] % 4 == 0;
    }
    const int mb = a.tokens > 64 ? 8 : (a.tokens > 32 || w.fp4 ? 4 : 2);
    const int s = joint_splits(a, cus, n_tiles * ((a.tokens + 16 * mb - 1) / (16 * mb)), mb == 8 ? 8 : 16, by4, scratch);
    if (s > 1) { return GemmPlan{ mb, 4, s, false, 1 }; }
    // on the file layout the 128-token tile is worth having from one workgroup per CU on, see large_linear
    const long long tiles8 = n_tiles * ((a.tokens + 127) / 128);
    return GemmPlan{ !w.fp4 && a.tokens > 64 && (tiles8 >= 2LL * cus || (w.row_major && tiles8 >= cus)) ? 8 : 4, 4, 1, false, 1 };
}

// gate / up pair, a tile covers 32 nb output features: FP8 128 tokens x 128 features, FP4 64 x 128; few tiles: the k range split
inline GemmPlan large_pair(const LinearArgs& a, const GemmWeights& w, int cus, bool scratch)
{
    const int mb = w.fp4 ? 4 : (a.tokens > 64 ? 8 : (a.tokens > 32 ? 4 : 2));
    const long long base = (long long)((a.n_out + 127) / 128) * ((a.tokens + 16 * mb - 1) / (16 * mb));
    const int s = joint_splits(a, cus, base, 8, a.n_out % 4 == 0, scratch);
    return GemmPlan{ s > 1 || w.fp4 ? mb : 8, 4, s, false, 1 };
}

// What a tile takes, in us:
//   fixed + per_cu x workgroups of a CU                    launch, first loads, stores
//   + k-tiles of a workgroup x us per k-tile               one workgroup on a CU: `one`, down to 0.85 of it where few of the CUs
//     (or the weight and the output at 5, FP4 4.1 MB/us,   have one; more: `each` per workgroup, and no less than `one`
//     if that is longer)
//   + 2 + 0.2 per k range + 0.3 per MB of partial sums     the combine launch
// The workgroups of a feature tile all land on XCD (tile % 8), so a CU of the fullest XCD is what counts: 20 feature tiles x 12
// workgroups are 36 on four of the XCDs, two rounds, and 24 on the others.
// Fitted to 170,000 measured launches (28 shapes x 16 token counts x every tile and k split, the four columns below, FP4 in blocks
// of 16 and 32, HALF activations, pairs, add and norm; up to 32 weights in turn), error 6.5 % rms.
struct GemmTile
{
    int mb, nb;
    double fixed, per_cu;
    double one[4], each[4];           // FP8: tiled copy, file layout, tiled copy with a scale, file layout with a scale
};

// weights requested three k-tiles ahead; 32 x 256 only with the k range split
constexpr GemmTile kSmallTiles[] = {
    { 2, 1, 2.4, 0.6, { 0.214, 0.247, 0.243, 0.261 }, { 0.132, 0.208, 0.148, 0.215 } },
    { 2, 2, 2.6, 1.1, { 0.248, 0.387, 0.302, 0.399 }, { 0.194, 0.358, 0.225, 0.362 } },
    { 2, 4, 3.2, 1.5, { 0.382, 0.686, 0.490, 0.694 }, { 0.330, 0.663, 0.405, 0.664 } },
    { 4, 1, 2.8, 0.9, { 0.240, 0.267, 0.284, 0.310 }, { 0.177, 0.213, 0.197, 0.223 } },
    { 4, 2, 3.2, 1.4, { 0.290, 0.393, 0.345, 0.406 }, { 0.224, 0.326, 0.270, 0.339 } },
    { 4, 4, 4.5, 1.7, { 0.436, 0.675, 0.583, 0.684 }, { 0.360, 0.573, 0.473, 0.594 } },
    { 8, 2, 4.5, 2.9, { 0.471, 0.507, 0.559, 0.578 }, { 0.395, 0.441, 0.454, 0.487 } },
};
// one k-tile ahead
constexpr GemmTile kLargeTiles[] = {
    { 8, 4, 6.5, 1.1, { 0.766, 0.959, 0.946, 1.116 }, { 0.638, 0.732, 0.756, 0.815 } },
    { 8, 3, 3.1, 3.7, { 0.675, 0.823, 0.818, 0.938 }, { 0.508, 0.540, 0.602, 0.625 } },
    { 4, 4, 3.9, 1.3, { 0.697, 0.831, 0.898, 0.976 }, { 0.373, 0.569, 0.501, 0.601 } },
    { 4, 3, 1.2, 2.3, { 0.630, 0.683, 0.755, 0.787 }, { 0.275, 0.417, 0.366, 0.439 } },
    { 4, 2, 1.5, 1.4, { 0.589, 0.575, 0.701, 0.637 }, { 0.222, 0.314, 0.279, 0.333 } },
};
constexpr GemmTile kSmallTilesFp4[] = {
    { 2, 1, 1.2, 1.1, { 0.376 }, { 0.133 } },
    { 2, 2, 2.2, 1.0, { 0.433 }, { 0.250 } },
    { 4, 1, 1.4, 1.5, { 0.399 }, { 0.156 } },
    { 4, 2, 3.4, 1.0, { 0.443 }, { 0.274 } },
    { 8, 2, 6.1, 0.3, { 0.553 }, { 0.423 } },
};
constexpr GemmTile kLargeTilesFp4[] = {
    { 4, 3, 4.6, 0.6, { 0.522 }, { 0.366 } },
    { 4, 4, 5.1, 1.1, { 0.634 }, { 0.476 } },
    { 8, 3, 6.8, 0.6, { 0.707 }, { 0.552 } },
    { 8, 4, 7.3, 2.1, { 0.913 }, { 0.873 } },
};

// What the estimate takes from the launch and from a tile on it, worked out once: a call asks for 20 to 200 estimates (0.7 us of host time
// for plan_gemm and staged_plan together, 1.0 with every estimate from scratch).
struct LaunchShape
{
    const LinearArgs& a;
    GemmKind kind;
    int cus, column;
    double outputs, traffic_us, partial_us;       // MB of output elements; bytes; FP32 sums, per k range

    LaunchShape(const LinearArgs& args, GemmKind k, const GemmWeights& w, int n_cus) : a(args), kind(k), cus(n_cus), column(w.fp4 ? 0 : (w.scaled ? 2 : 0) + (w.row_major ? 1 : 0))
    {
        long long features = a.n_out;
        if (kind == GEMM_SEGMENTS)
        {
            features = 0;
            for (int s = 0; s < a.n_segments; s++) { features += a.seg_n_out[s]; }
        }
        const double two = kind == GEMM_PAIR ? 2.0 : 1.0;
        outputs = 1e-6 * (double)a.tokens * (double)features;
        traffic_us = (1e-6 * two * (double)features * a.K * (w.fp4 ? 0.5625 : 1.0) + 2.0 * outputs) / (w.fp4 ? 4.1 : 5.0);
        partial_us = 0.2 + 0.3 * 4.0 * two * outputs;
    }
};

struct TileEstimate
{
    const LaunchShape& launch;
    const GemmTile& t;
    long long workgroups;       // of the fullest XCD, times eight

    TileEstimate(const LaunchShape& l, const GemmTile& tile) : launch(l), t(tile)
    {
        const int width = l.kind == GEMM_PAIR ? 32 * t.nb : 64 * t.nb;
        int n_tiles = 0;
        if (l.kind != GEMM_SEGMENTS) { n_tiles = (l.a.n_out + width - 1) / width; }
        else
        {
            for (int s = 0; s < l.a.n_segments; s++) { n_tiles += (l.a.seg_n_out[s] + width - 1) / width; }
        }
        workgroups = (n_tiles + 7LL) / 8 * 8 * ((l.a.tokens + 16 * t.mb - 1) / (16 * t.mb));
    }

    double us(int splits, double alone = 0.85) const
    {
        const double fill = (double)(workgroups * splits) / launch.cus;
        const double per_cu = fill <= 1.0 ? 1.0 : 0.1 * fill + 0.9 * (double)((workgroups * splits + launch.cus - 1) / launch.cus);
        const double one = t.one[launch.column];
        const double k_tile = fill <= 1.0 ? one * (alone + (1.0 - alone) * fill) : std::max(one, t.each[launch.column] * per_cu);
        const double time = t.fixed + t.per_cu * per_cu + std::max((double)((launch.a.K / 64 + splits - 1) / splits) * k_tile, launch.traffic_us);
        return splits > 1 ? time + 2.0 + splits * launch.partial_us : time;
    }
};

// The larger tile, or the small one with the least estimate if that is 6 % or more below.  Of 4357 measured cases 20 then take
// more than 3 % longer than on the larger tile alone (6 % at most), and the mean is 0.79 of its time; of 5785 calls of a later
// run, other shapes among them, 39 (10 % at most) and 0.76 (profiles/gemm_tiles.md).  Without scratch memory nothing splits its
// k range.
// A linear of up to 4096 features whose larger tile splits may come with the residual add and the norm behind it
// (hip_quant_gemm_add_rms_norm), and gives the same bits either way, so both take one plan.  Behind a k split the combine
// launch carries them, an unsplit launch has a row kernel to follow (3 us + 0.55 per MB of output): half of that, 6 % of the launch
// at most, is laid on the unsplit plans (of 739 cases with add and norm 3 are then more than 3 % slower than on the larger tile
// and 14 without it; linears alone 0.764 of the larger tiles' time and 0.763; a fixed share would cost launches of 5 us a third).
inline GemmPlan plan_gemm(const LinearArgs& a, GemmKind kind, const GemmWeights& w, int cus, bool scratch)
{
    GemmPlan plan = kind == GEMM_PAIR ? large_pair(a, w, cus, scratch) : kind == GEMM_SEGMENTS ? large_segments(a, w, cus, scratch)
                  : w.fp4 ? large_fp4(a, w, cus, scratch) : large_linear(a, w, cus, scratch);
    plan.ranges = plan.splits;
    const GemmTile* const small = w.fp4 ? kSmallTilesFp4 : kSmallTiles;
    const int n_small = w.fp4 ? sizeof(kSmallTilesFp4) / sizeof(GemmTile) : sizeof(kSmallTiles) / sizeof(GemmTile);
    const bool deep = !w.fp4 && plan.splits > 1 && plan.mb <= 4;      // the larger tiles that take their weights three k-tiles ahead as well
    const GemmTile* const large = w.fp4 ? kLargeTilesFp4 : deep ? kSmallTiles : kLargeTiles;
    const int n_large = w.fp4 ? sizeof(kLargeTilesFp4) / sizeof(GemmTile) : deep ? n_small : sizeof(kLargeTiles) / sizeof(GemmTile);
    const LaunchShape launch(a, kind, w, cus);
    double limit = 0.0;
    for (int i = 0; i < n_large; i++)
    {
        if (large[i].mb == plan.mb && large[i].nb == plan.nb) { limit = 0.94 * TileEstimate(launch, large[i]).us(plan.splits); }
    }
    const bool add_norm = kind == GEMM_LINEAR && plan.ranges > 1 && a.n_out <= 4096 && a.n_out % 8 == 0;
    const double row_kernel = add_norm ? 0.5 * (3.0 + 0.55 * 2e-6 * (double)a.tokens * a.n_out) : 0.0;
    for (int i = 0; i < n_small; i++)
    {
        const GemmTile& t = small[i];
        if ((t.mb == 2 && (a.tokens > 64 || t.nb == 4)) || (t.mb == 8 && (a.tokens <= 64 || (!w.fp4 && (!w.row_major || w.scaled)))) || (kind == GEMM_PAIR && t.nb == 1)) { continue; }
        const TileEstimate tile(launch, t);
        for (int s = 1; s <= plan.ranges && (s == 1 || a.K / 64 >= 4 * s); s++)
        {
            double us = tile.us(s);
            if (s == 1) { us += std::min(row_kernel, 0.06 * us); }
            if (us < limit)
            {
                limit = us;
                plan = GemmPlan{ t.mb, t.nb, s, true, plan.ranges };
            }
        }
    }
    return plan;
}

// gemm_staged_kernel, all weights: the same estimate, fitted to 10,900 launches (13 shapes x 11 token counts from 20 to 1024 x every tile
// and 1 to 8 k ranges, the four columns and HALF activations; weights in turn through up to 1.2 GB) of an earlier form of the kernel.
// On 21,700 launches of this one, at 25 token counts from 18 to 512, it is 4 to 7 % high (7 to 10 % rms per tile).  Alone on a CU a
// k-tile takes down to 0.7 of `one`: the loads share L2 and HBM with fewer others.
constexpr GemmTile kStagedTiles[] = {
    { 2, 1, 3.2, 0.6, { 0.162, 0.174, 0.208, 0.211 }, { 0.143, 0.152, 0.158, 0.167 } },
    { 2, 2, 2.3, 2.7, { 0.226, 0.240, 0.317, 0.314 }, { 0.247, 0.257, 0.302, 0.305 } },
    { 3, 2, 2.3, 3.6, { 0.223, 0.232, 0.336, 0.338 }, { 0.223, 0.231, 0.305, 0.312 } },
    { 4, 1, 2.2, 2.3, { 0.189, 0.199, 0.233, 0.233 }, { 0.145, 0.153, 0.167, 0.174 } },
    { 4, 2, 2.0, 4.1, { 0.249, 0.260, 0.353, 0.355 }, { 0.256, 0.263, 0.323, 0.334 } },
    { 5, 2, 2.3, 4.5, { 0.294, 0.301, 0.399, 0.407 }, { 0.289, 0.293, 0.360, 0.375 } },
    { 7, 2, 2.5, 5.0, { 0.361, 0.381, 0.462, 0.460 }, { 0.356, 0.360, 0.426, 0.434 } },
};

// The staged kernel in the place of `plan` from K = 1024 on (the shortest that the estimate is fitted to) and up to 512 tokens (above that
// the larger tiles are level or ahead).
// It adds the products in the order of the register-fed kernels, so only the k ranges of a launch show in its bits.  A plan of one
// range keeps one: joint and paired launches give the bits of the separate calls where none of them splits k, whichever kernel each
// of them takes.  A k-split plan may get other ranges; where the plans of the two weight layouts have the same, one decision serves
// both, the k ranges for which the staged kernel is ahead on both together, so that a weight gives the same bits from the file layout
// and from its tiled copy.  Elsewhere each layout takes what is best for it.
// Ahead: 0.3 us and 5 % (file layout) or 8 % (tiled copy, whose KiB blocks the other kernels read whole as well; 3 % in a joint decision)
// below the plan's own estimate; with less, launches of 5 us and k-split ones on tiled copies lose up to 15 %.  Of 1550
// measured calls (the 13 shapes and 25 token counts above) 278 then run it, three of them more than 3 % slower than on the plan (7 % at
// most); mean of all calls 0.94 of the plans' time on E5M2 in the file layout, 0.96 with scales, 0.98 on tiled copies.  A tile
// with sixteen tokens or more past the end is not considered, which leaves 81 to 96 and 113 to 128 tokens with smaller ones.
// An unsplit linear that may come with the add and the norm carries half of the row kernel, as in plan_gemm, and must not be behind
// with all of it either (4096 x 12288 at 512 tokens, tiled: 58 us alone on both, 64 against 55 with the norm).
// `scratch` is that of the call to plan_gemm.  The k ranges of the larger tile, and so the scratch memory, stay what they were.  FP4
// keeps its plans.
inline GemmPlan staged_plan(const LinearArgs& a, GemmKind kind, const GemmWeights& w, int cus, const GemmPlan& plan, bool scratch)
{
    if (w.fp4 || a.K < 1024 || a.tokens > 512) { return plan; }
    const GemmWeights layouts[2] = { w, { false, !w.row_major, w.scaled } };
    const GemmPlan plans[2] = { plan, plan_gemm(a, kind, layouts[1], cus, scratch) };
    const LaunchShape launches[2] = { { a, kind, layouts[0], cus }, { a, kind, layouts[1], cus } };
    constexpr int MOST = 16;                    // k ranges of any plan
    const bool joint = plans[0].splits == plans[1].splits;
    const int ranges = plan.splits == 1 ? 1 : std::min(joint ? plans[1].ranges : MOST, std::min(plan.ranges, MOST));
    const bool add_norm = kind == GEMM_LINEAR && plan.ranges > 1 && a.n_out <= 4096 && a.n_out % 8 == 0;
    const double row_kernel = add_norm ? 3.0 + 0.55 * 2e-6 * (double)a.tokens * a.n_out : 0.0;
    double limit[2] = { 0.0, 0.0 }, with_norm[2] = { 0.0, 0.0 };
    for (int l = 0; l < (joint ? 2 : 1); l++)
    {
        const GemmPlan& p = plans[l];
        const bool deep = p.small || (p.splits > 1 && p.mb <= 4);
        const GemmTile* const table = deep ? kSmallTiles : kLargeTiles;
        const int n_table = deep ? sizeof(kSmallTiles) / sizeof(GemmTile) : sizeof(kLargeTiles) / sizeof(GemmTile);
        for (int i = 0; i < n_table; i++)
        {
            if (table[i].mb == p.mb && table[i].nb == p.nb)
            {
                const double us = TileEstimate(launches[l], table[i]).us(p.splits), row = p.splits == 1 ? row_kernel : 0.0;
                limit[l] = (layouts[l].row_major ? 0.95 : joint ? 0.97 : 0.92) * (us + 0.5 * row) - 0.3;
                with_norm[l] = us + row;
            }
        }
    }
    double least[2][MOST];                      // per layout and number of ranges
    const GemmTile* least_tile[MOST] = {};      // on the layout of the launch
    for (int s = 0; s < MOST; s++) { least[0][s] = least[1][s] = 1e30; }
    for (const GemmTile& t : kStagedTiles)
    {
        if ((t.mb > 2 && 16 * (t.mb - 1) >= a.tokens) || (t.mb == 2 && a.tokens > 64) || (t.mb == 3 && a.tokens > 192)) { continue; }
        for (int l = 0; l < (joint ? 2 : 1); l++)
        {
            const TileEstimate tile(launches[l], t);
            for (int s = 1; s <= ranges && (s == 1 || a.K / 64 >= 4 * s); s++)
            {
                const double us = tile.us(s, 0.7);
                if (us >= least[l][s - 1]) { continue; }
                least[l][s - 1] = us;
                if (l == 0) { least_tile[s - 1] = &t; }
            }
        }
    }
    GemmPlan best = plan;
    double least_sum = 1e30;
    for (int s = 1; s <= ranges && least_tile[s - 1]; s++)
    {
        const double row = s == 1 ? row_kernel : 0.0;
        double sum = 0.0;
        for (int l = 0; l < (joint ? 2 : 1); l++)
        {
            const double us = least[l][s - 1];
            sum += us + 0.5 * row < limit[l] && us + row <= with_norm[l] ? us + 0.5 * row : 1e30;
        }
        if (sum < least_sum)
        {
            least_sum = sum;
            best = GemmPlan{ least_tile[s - 1]->mb, least_tile[s - 1]->nb, s, true, plan.ranges, true };
        }
    }
    return best;
}

}    // namespace ccq
