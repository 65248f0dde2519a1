// gemm_plan.h - how one dequant-GEMM call is run: which kernel takes it, how
// K is split, which 16-bit operand type f32 activations are rounded to, and
// the workspace layout. Host code only (no HIP types), so the CPU tests can
// sweep shapes through it (tests/c/plan_check.cpp).
//
// Shapes are in GEMM form: M tokens, N output features, K input features
// (BatchMatMulPC's seq_len, out_dim, in_dim, dit.c3:172-178).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "llmr_hip.h"

namespace llmr {
namespace plan {

constexpr uint32_t kF32 = LLMR_GGML_F32, kF16 = LLMR_GGML_F16, kBF16 = LLMR_GGML_BF16;
constexpr uint32_t kQ8_0 = LLMR_GGML_Q8_0, kQ4K = LLMR_GGML_Q4_K;

constexpr uint32_t kStageK = 64;          // K per stage of every MFMA kernel
constexpr uint32_t kImageBlock = 256u * 128u;  // bytes of one 256-row x 64-wide 16-bit image block
// Weights times at most this many tokens run on the GEMV kernels (an HBM-bound
// weight stream, gemv_q.hip): Q4_K always, Q8_0 where gemv_q8_fits.
constexpr uint32_t kGemvMaxTokens = 4;
// From this many tokens the weight is dequantized once per call into a
// 16-bit image (gemm_w16.hip) instead of once per 256-token tile.
constexpr uint32_t kW16MinTokens = 2048;
// The tiled kernel splits K when it has fewer than kSplitWgsPerCu
// workgroups per CU, with at least kSplitMinStages stages per split.
constexpr uint32_t kSplitWgsPerCu = 2, kSplitMinStages = 4;
// The few-token kernel (gemm_few.hip): a workgroup owns 32 tokens x
// kFewFeatures or kFewNarrow features over the whole K.
constexpr uint32_t kFewTokens = 32, kFewFeatures = 96, kFewNarrow = 32, kFewMaxTokens = 512;
constexpr uint32_t kSkinnyMaxTokens = 256;

inline uint64_t row_bytes_of(uint32_t wtype, uint32_t K) {
    return wtype == kQ8_0 ? (uint64_t)(K / 32) * 34 : (uint64_t)(K / 256) * 144;
}

inline size_t align256(size_t b) { return (b + 255u) / 256u * 256u; }

// The MFMA operand type f32 activations are rounded to. Q8_0: fp16, the
// reference's float16_t(x) of batch_matmul_q8 (llm.slang:1673). Q4_K: bf16
// (batch_matmul_q4k multiplies x in f32, llm.slang:2300-2304, so a value
// beyond fp16's 65504 stays finite there; bf16 keeps f32's range).
inline uint32_t f32_operand_type(uint32_t wtype) { return wtype == kQ4K ? kBF16 : kF16; }

// The MFMA operand type of activations of type xtype against wtype weights.
inline uint32_t operand_type(uint32_t wtype, uint32_t xtype) {
    return xtype == kF32 ? f32_operand_type(wtype) : xtype;
}

// Bytes of the 16-bit weight image of N features (SwiGLU: 128-feature
// panels of gate and up rows) for the two-pass path.
inline size_t w16_image_bytes(uint32_t N, uint32_t K, bool swiglu) {
    const uint64_t panels = swiglu ? (N + 127u) / 128u : (N + 255u) / 256u;
    return (size_t)(panels * (K / kStageK) * kImageBlock);
}

// The split count for `want` splits of S stages such that every split of
// ceil(S / splits) stages is non-empty (the kernels take split z as stages
// [z per, min(S, (z + 1) per)), per = ceil(S / splits)).
inline uint32_t nonempty_splits(uint32_t S, uint32_t want) {
    if (S == 0) return 1;
    uint32_t splits = std::max<uint32_t>(1u, std::min(want, S));
    for (;;) {
        const uint32_t per = (S + splits - 1) / splits, used = (S + per - 1) / per;
        if (used == splits) return splits;
        splits = used;
    }
}

// Whether `splits` splits of S stages are all non-empty (the launchers'
// check before a split launch).
inline bool splits_nonempty(uint32_t S, uint32_t splits) {
    if (splits == 0 || splits > S) return false;
    const uint32_t per = (S + splits - 1) / splits;
    return (S + per - 1) / per == splits;
}

// Bytes of f32 activations rounded to 16 bits for the few-token skinny
// kernel (stage-major); 16-bit activations are read in place.
inline size_t skinny_x_bytes(uint32_t xtype, uint32_t M, uint32_t K) {
    return xtype == kF32 ? align256((size_t)M * K * 2u) : 0u;
}

// The 4-wave tiled kernel's tile (64, 128 or 256 square) and K splits: the
// largest tile that still gives every CU ~1.5 workgroups; launches with fewer
// workgroups than kSplitWgsPerCu per CU split K (at least kSplitMinStages
// stages per split, M * N % 4 == 0 for the reduction, partials within ws_limit:
// as many as fit, none if fewer than two).
constexpr size_t kNoWorkspaceLimit = ~(size_t)0;
struct TilePlan {
    uint32_t bm, splits;
};
inline TilePlan plan_tiles(uint32_t wtype, uint32_t N, uint32_t K, uint32_t M, int num_cus,
                           size_t ws_limit = kNoWorkspaceLimit) {
    auto wgs = [&](uint32_t bm) { return (uint64_t)((M + bm - 1) / bm) * ((N + bm - 1) / bm); };
    const uint64_t want = (uint64_t)num_cus * 3 / 2;
    TilePlan t{64, 1};
    if (wgs(256) >= want) t.bm = 256;
    else if (wgs(128) >= want) t.bm = 128;
    if (wtype == kQ8_0 && K % kStageK) return t;  // the generic kernel
    const uint64_t w = wgs(t.bm), target = (uint64_t)num_cus * kSplitWgsPerCu;
    const uint32_t S = K / kStageK;
    if (w < target && S >= 2 * kSplitMinStages && ((uint64_t)M * N) % 4 == 0)
        t.splits = nonempty_splits(S, (uint32_t)std::min<uint64_t>((target + w - 1) / w, S / kSplitMinStages));
    const size_t fit = ws_limit / ((size_t)M * N * sizeof(float));
    if (t.splits > fit) t.splits = fit >= 2 ? nonempty_splits(S, (uint32_t)fit) : 1u;
    return t;
}

// Whether the few-token kernel can take M x N x K: at most kFewMaxTokens
// tokens, whole stages, 32-bit buffer offsets.
inline bool few_fits(uint32_t wtype, uint32_t N, uint32_t K, uint32_t M) {
    if (M == 0 || M > kFewMaxTokens || K % kStageK || K == 0) return false;
    // the f32 activation rows and the weight rows past N that a last tile addresses
    return (uint64_t)(M + kFewTokens) * K * 4u < (1ull << 31) &&
           (uint64_t)(N + kFewFeatures) * row_bytes_of(wtype, K) < (1ull << 32);
}

// The few-token kernel's tile width up to kSkinnyMaxTokens tokens (0: the
// skinny kernel, or the tiled one where N % 4). 96-feature tiles read the fewest
// bytes per CU but hold it alone (102 KiB of LDS), so their cost is whole rounds
// over the CUs; 32-feature tiles share a CU two at a time and cost by their number
// (f32 activations, re-read by every tile, more so past K = 8192, as 16-bit ones a
// little), plus a fixed part of a round. In units of a 32-feature tile; measured on
// 256 CUs, 96 -> 32 features: 77 x 9216 x 3072 Q4_K bf16 27.2 -> 19.2 us, 200 x 3840
// x 3840 31.0 -> 22.7, 64 x 9216 x 3072 15.2 / 15.7, 200 x 3072 x 3072 15.2 / 15.4,
// Q8_0 f32 15.7 / 21.0, 200 x 21504 x 15360 Q8_0 bf16 414 / 508, 150 x 21504 x 8192
// 155 / 170; where both come close, within a quarter (113 x 9368 x 10240 72 / 93, 256
// x 2048 x 8192 31 / 26, the 32-feature tiles both).
// Below half the CUs' worth of 96-feature tiles the 32-feature tiles take 77 x 3072
// x 4096 Q4_K bf16 in 12.8 us against the skinny kernel's 19.5 (packed activations,
// K splits, partial sums: three launches), 32 x 3840 x 3840 8.7 against 19.6, 5 x
// 9216 x 3072 10.5 against 43. The skinny kernel is the better one where a wave's K
// stages, one after the other, are most of the time: f32 activations with long rows
// (77 x 3072 x 12288 43 against 48 us; from 14336 with few features too, 150 x 64 x
// 15360 28 against 34, tiled 23), 16-bit ones from 14336 with 257 to 1024 features
// (few-token : skinny at 512 features 0.98 at K = 12288, 1.02-1.13 at 14336,
// 1.03-1.20 at 15360; at 64 and 256 0.9-1.0 up to 16384, 1.0-1.1 past it), and long
// rows where some CUs get a second tile (200 x 1536 x 8192 26 against 35, 150 x
// 2048 x 15360 bf16 36 against 48).
inline uint32_t few_features(uint32_t xtype, uint32_t N, uint32_t K, uint32_t M, int num_cus) {
    const uint64_t tm = (M + kFewTokens - 1) / kFewTokens, c = (uint64_t)num_cus;
    const uint64_t wide = tm * ((N + kFewFeatures - 1) / kFewFeatures), narrow = tm * ((N + kFewNarrow - 1) / kFewNarrow);
    const bool f32 = xtype == kF32;
    if (2 * wide < c) {
        const bool skinny = N % 4 == 0 && ((f32 && K > 8192 && N >= 512) || (narrow > c && K >= 8192 && N < 3072) ||
                                           (!f32 && K >= 14336 && N > 256 && N <= 1024) ||
                                           (!f32 && K > 16384 && N <= 1024));
        return skinny || (f32 && K >= 14336 && N < 512) ? 0u : kFewNarrow;
    }
    const double f = f32 ? (K > 8192 ? 1.6 : 1.3) : K >= 8192 ? 1.14 : 1.03;
    return f * narrow + 0.7 * c < 3.0 * c * ((wide + c - 1) / c) ? kFewNarrow : kFewFeatures;
}
// Time in us of the 32-feature tiles past kSkinnyMaxTokens tokens, for the choice
// against plan_split and the tiled kernel: a wave's K / 512 stages one after
// the other, or the tiles a CU has times their stages (with f32 activations a
// second tile on a CU doubles the time), more past K = 8192, where the activation
// rows leave the L2. Measured: 300 x 3072 x 3072 Q4_K bf16 19 us, 257 x 9216 x 256
// Q8_0 12.6, 288 x 64 x 15360 f32 34.
inline double few_us(uint32_t xtype, uint32_t N, uint32_t K, uint32_t M, int num_cus) {
    const bool f32 = xtype == kF32;
    double q = (double)((M + kFewTokens - 1) / kFewTokens) * ((N + kFewNarrow - 1) / kFewNarrow) / num_cus;
    if (f32 && q < 2.0) q = q <= 1.0 ? 1.0 : 2.0;
    const double stages = K / 512.0, far = std::max(0.0, (K - 8192.0) / 4096.0), n = (K + 511) / 512;
    const double tiles = 4.0 + q * (0.5 + (f32 ? 1.03 : 0.68) * std::max(stages, 0.5) + (f32 ? 7.7 : 3.2) * far);
    return std::max({7.6, tiles, f32 ? 1.16 * n : 1.4 + 0.79 * n});
}
// Time in us of the tiled kernel: two of its workgroups per CU run at full
// speed, its 64 x 64 tiles four at a time (three with f32 activations).
inline double tiled_us(uint32_t wtype, uint32_t xtype, uint32_t N, uint32_t K, uint32_t M, int num_cus,
                       size_t ws_limit) {
    const TilePlan t = plan_tiles(wtype, N, K, M, num_cus, ws_limit);
    const bool f32 = xtype == kF32;
    const double wgs = (double)((M + t.bm - 1) / t.bm) * ((N + t.bm - 1) / t.bm) * t.splits, c = (double)num_cus;
    const double rounds = wgs <= 2 * c ? 1.0 : wgs <= (f32 ? 3 : 4) * c ? 1.8 : std::max(3.1, 0.55 * wgs / c);
    const double per_k = (t.bm == 64 ? 1.0 : t.bm == 128 ? 2.8 : 8.0) * (wtype == kQ8_0 ? 0.0105 : 0.0090) *
                         (!f32 ? 1.0 : K < 8192 ? 1.05 : 1.26);
    return 6.0 + rounds * ((double)K / t.splits) * per_k;
}
// What its split-K sum (the output's stores where it has none) adds to that.
inline double tiled_sum_us(uint32_t wtype, uint32_t N, uint32_t K, uint32_t M, int num_cus, size_t ws_limit) {
    const TilePlan t = plan_tiles(wtype, N, K, M, num_cus, ws_limit);
    const double y = (double)M * N * sizeof(float) / 5e6;
    return t.splits > 1 ? 3.0 + 0.25 * t.splits + y * (t.splits + 1) : 0.3 * y;
}

// Launches below kW16MinTokens tokens, or with too few tiles for the persistent
// kernels, whose 256 x 256 tiles leave CUs idle in their last round: the whole
// rounds of tiles run as they are (`full` of them) and every tile of the last
// round is cut along K into `splits` workgroups, whose partial tiles a second
// launch adds up. The times are estimates in us on MI355X (256 CUs), fitted to
// 1500 launches of 257-9000 tokens x 64-21504 features: a K stage of a tile takes
// 2.0 us on the 8-wave kernel that also runs the splits (1.93 and 1.7 for Q8_0 and
// Q4_K where tiles follow each other in the persistent kernels, down to three
// quarters of it where most CUs have none), a workgroup 8 us around its stages,
// the partial tiles are written and read at ~5 TB/s, and f32 activations, which
// the tiled kernel reads in place, are rounded by a launch of their own. Measured,
// whole launch before -> after: 1101 x 3840 x 3840 Q8_0 (75 tiles x 3) 129 ->
// 60 us, x 10240 348 -> 117; 520 x 9216 x 3072 Q4_K (108 x 2) 99 -> 60; 1536 x
// 11520 x 3840 Q8_0 (256 whole tiles + 14 x 15) 236 -> 160; 2000 x 9216 x
// 3072 Q4_K (256 + 32 x 8) 165 -> 139; 2048 x 3840 x 3840 Q8_0 (120 x 2) 123
// -> 88, x 10240 256 -> 169. Where the estimates are within 3%
// the launch stays whole (2000 x 12288 x 3072 Q4_K, 128 tiles in its last
// round: 168 whole, 177 split).
constexpr size_t kPartTile = 256u * 256u * sizeof(float);  // one partial tile
constexpr uint32_t kSplitMax = 16;
// Fewer K stages than this run whole: a workgroup's fixed 8 us are then as
// long as all of a tile's stages.
constexpr uint32_t kSplitTileMinStages = 16;
struct SplitPlan {
    uint32_t full, splits;  // splits 1: no split
    size_t x16;             // bytes of f32 activations rounded to 16 bits, before the partial tiles
    double us;              // of the launch, split or whole
    size_t ws(uint64_t tiles) const { return x16 + (size_t)(tiles - full) * splits * kPartTile; }
};
inline SplitPlan plan_split(uint32_t wtype, uint32_t xtype, uint32_t N, uint32_t K, uint32_t M, int num_cus,
                            bool persistent, size_t ws_limit, bool cut_tiles) {
    const uint64_t tiles = (uint64_t)((M + 255) / 256) * ((N + 255) / 256);
    const uint32_t S = K / kStageK;
    const uint64_t full = tiles / num_cus * num_cus, rem = tiles - full;
    SplitPlan p{(uint32_t)full, 1, xtype == kF32 ? align256((size_t)M * K * 2u) : 0u, 0.0};
    const double whole = persistent
                             ? (full == 0 ? 0.75 + 0.25 * rem / num_cus : (double)((tiles + num_cus - 1) / num_cus)) *
                                       S * (wtype == kQ8_0 ? 1.93 : 1.7) + 6.0
                             : tiled_us(wtype, xtype, N, K, M, num_cus, ws_limit);
    p.us = whole;
    double best = 0.97 * whole;
    const double round_x = xtype == kF32 && !persistent ? (double)M * K * 6.0 / 8e6 : 0.0;
    for (uint32_t s = 2; cut_tiles && rem && S >= kSplitTileMinStages && s <= std::min(kSplitMax, S / kSplitMinStages); s++) {
        if (nonempty_splits(S, s) != s || p.x16 + (size_t)rem * s * kPartTile > ws_limit) continue;
        const double rounds = (double)((rem * s + num_cus - 1) / num_cus);
        const double us = (double)(full / num_cus) * (S * 2.0 + 8.0) + rounds * ((S + s - 1) / s * 2.0 + 8.0) + 3.0 +
                          (double)rem * kPartTile * (s + 1) / 5e6 + round_x;
        if (us < best) best = p.us = us, p.splits = s;
    }
    return p;
}

// How one GEMM runs.
//  * few: the few-token kernel (f32 / 16-bit activations read in place, no
//    workspace), to kSkinnyMaxTokens tokens as few_features says, past them
//    where few_us is the least;
//  * skinny: the few-token kernel with K splits (where few_features is 0):
//    workspace = [f32 activations as 16 bits | split partials];
//  * persistent: the 256 x 256 persistent kernels (at least half the CUs'
//    worth of tiles, whole stages, N % 4 == 0, 31-bit buffer offsets), f32
//    activations rounded to operand_type() into the workspace first; from
//    kW16MinTokens tokens two-pass (the 16-bit weight image after them in
//    the workspace);
//  * split: below kW16MinTokens tokens or where not persistent, where plan_split finds that cutting
//    the last round's tiles along K pays: [x16 | partial tiles];
//  * otherwise the tiled kernel, split-K partials in the workspace.
// With a workspace limit (the no-allocation entry point's fixed array) the
// plan keeps within it: the two-pass path only when its image fits, as many
// splits as fit (none if fewer than two), and the kernels that read f32
// activations in place (tiled, few-token) when the 16-bit copy of f32
// activations for the others does not fit. The estimates are of what fits: with
// 32 MiB, 323 x 3072 x 15360 Q8_0 f16 ran the tiled kernel, 1.5 times the
// few-token kernel's time, as the split it was compared with did not fit.
// Without cut_tiles (a stream being captured, which allocates and waits for
// nothing) no tile is cut along K: such a launch needs a workspace where the tiled
// kernel mostly needs none.
struct GemmPlan {
    bool persistent, two_pass, convert_x, skinny, few;
    uint32_t xt;                  // activation type the kernel reads
    TilePlan tiles;               // the tiled kernel's tile and splits (not persistent)
    uint32_t splits;              // the skinny kernel's K splits
    uint32_t few_features;        // few: features of a tile
    uint32_t split, split_full;   // split > 1: 256 x 256 tiles, those past split_full cut along K into `split`
    size_t x16_off, img_off, ws;  // workspace: [x16 | image] (persistent), [packed x | partials]
                                  // (skinny), split-K partials (tiled)
};
inline GemmPlan plan_gemm(uint32_t wtype, uint32_t xtype, uint32_t N, uint32_t K, uint32_t M, int num_cus,
                          size_t ws_limit = kNoWorkspaceLimit, bool cut_tiles = true) {
    GemmPlan p{};
    p.xt = xtype;
    p.tiles = TilePlan{64, 1};
    p.splits = 1;
    p.split = 1;
    const uint64_t rb = row_bytes_of(wtype, K);
    const bool offsets31 = (uint64_t)M * K * 2u < (1ull << 31) && (uint64_t)N * rb < (1ull << 31);
    const uint64_t tiles = (uint64_t)((M + 255) / 256) * ((N + 255) / 256);
    p.persistent = K % kStageK == 0 && N % 4 == 0 && 2 * tiles >= (uint64_t)num_cus && offsets31 &&
                   (xtype != kF32 || align256((size_t)M * K * 2u) <= ws_limit);
    const bool few_ok = !p.persistent && few_fits(wtype, N, K, M);
    if (few_ok && M <= kSkinnyMaxTokens) {
        p.few_features = few_features(xtype, N, K, M, num_cus);
        if (p.few_features) {
            p.few = true;
            return p;
        }
    }
    if (!p.persistent && M <= kSkinnyMaxTokens && K % kStageK == 0 && N % 4 == 0 && offsets31) {
        // few tokens over few features: the skinny kernel (one workgroup per
        // CU: its LDS), K split so the launch fills the CUs in one round (at
        // least kSplitMinStages stages per split), as far as the partials fit
        // the workspace
        const size_t x16 = skinny_x_bytes(xtype, M, K), part = (size_t)M * N * sizeof(float);
        if (x16 <= ws_limit) {
            const uint32_t S = K / kStageK, tn = (N + 63) / 64;
            uint32_t want = std::max<uint32_t>(1u, std::min<uint32_t>((uint32_t)num_cus / tn, S / kSplitMinStages));
            if (want > 1 && x16 + want * part > ws_limit)
                want = std::max<uint32_t>(1u, (uint32_t)((ws_limit - x16) / part));
            p.skinny = true;
            p.xt = operand_type(wtype, xtype);
            p.splits = nonempty_splits(S, want);
            p.ws = x16 + (p.splits > 1 ? p.splits * part : 0u);
            return p;
        }
    }
    if (K % kStageK == 0 && N % 4 == 0 && offsets31 && (M < kW16MinTokens || !p.persistent)) {
        const SplitPlan sp = plan_split(wtype, xtype, N, K, M, num_cus, p.persistent, ws_limit, cut_tiles);
        const double sum = sp.splits > 1 ? 0.0 : tiled_sum_us(wtype, N, K, M, num_cus, ws_limit);
        if (few_ok && few_us(xtype, N, K, M, num_cus) < 0.9 * (sp.us + sum)) {
            p.few = true;
            p.few_features = kFewNarrow;
            return p;
        }
        if (sp.splits > 1) {
            p.persistent = false;
            p.split = sp.splits;
            p.split_full = sp.full;
            p.convert_x = xtype == kF32;
            p.xt = operand_type(wtype, xtype);
            p.img_off = sp.x16;  // the partial tiles
            p.ws = sp.ws(tiles);
            return p;
        }
    }
    if (!p.persistent) {
        p.tiles = plan_tiles(wtype, N, K, M, num_cus, ws_limit);
        p.ws = p.tiles.splits > 1 ? (size_t)p.tiles.splits * M * N * sizeof(float) : 0u;
        return p;
    }
    p.convert_x = xtype == kF32;
    p.xt = operand_type(wtype, xtype);
    p.x16_off = 0;
    p.img_off = p.convert_x ? align256((size_t)M * K * 2u) : 0u;
    p.two_pass = M >= kW16MinTokens && p.img_off + w16_image_bytes(N, K, false) <= ws_limit;
    p.ws = p.img_off + (p.two_pass ? w16_image_bytes(N, K, false) : 0u);
    return p;
}

}  // namespace plan
}  // namespace llmr
