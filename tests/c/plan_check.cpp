// plan_check.cpp - sweeps GEMM shapes through the dispatcher's planner
// (llm-runner_amd/csrc/gemm_plan.h, host code only) and checks what every
// launch relies on:
//  * a split launch gives every split at least one K stage (the kernels
//    load their first stage unconditionally);
//  * the workspace a plan asks for stays within the limit it was given;
//  * f32 activations are rounded to fp16 against Q8_0 (the reference's
//    float16_t(x), llm.slang:1673) and to bf16 against Q4_K (whose reference
//    keeps x in f32, llm.slang:2300-2304).
// Prints "plan_check: N plans ok" and exits 0, or prints the first failing
// case and exits 1.
#include <cstdio>
#include <cstdlib>

#include "gemm_plan.h"

using namespace llmr::plan;

static long n_checked = 0;

static void fail(const char* what, uint32_t wt, uint32_t xt, uint32_t N, uint32_t K, uint32_t M, int cus,
                 size_t limit) {
    std::printf("FAIL %s: wtype %u xtype %u N %u K %u M %u cus %d limit %zu\n", what, wt, xt, N, K, M, cus, limit);
    std::exit(1);
}

static void check(uint32_t wt, uint32_t xt, uint32_t N, uint32_t K, uint32_t M, int cus, size_t limit) {
    const GemmPlan p = plan_gemm(wt, xt, N, K, M, cus, limit);
    const uint32_t S = K / kStageK;
    n_checked++;
    const GemmPlan w = plan_gemm(wt, xt, N, K, M, cus, limit, false);
    if (w.split > 1 || w.ws > limit) fail("plan without cut tiles", wt, xt, N, K, M, cus, limit);
    if (p.split <= 1 && (w.ws != p.ws || w.few != p.few || w.persistent != p.persistent || w.skinny != p.skinny))
        fail("cut_tiles changes a plan that cuts none", wt, xt, N, K, M, cus, limit);
    if (p.few + p.skinny + p.persistent + (p.split > 1) > 1) fail("more than one kernel", wt, xt, N, K, M, cus, limit);
    if (p.ws > limit) fail("workspace beyond the limit", wt, xt, N, K, M, cus, limit);
    if (p.few) {
        if (M > kFewMaxTokens || K % kStageK || p.ws != 0) fail("few-token plan", wt, xt, N, K, M, cus, limit);
        if (p.few_features != kFewNarrow && p.few_features != kFewFeatures)
            fail("few-token tile width", wt, xt, N, K, M, cus, limit);
        return;
    }
    if (p.skinny) {
        if (!splits_nonempty(S, p.splits)) fail("skinny split without stages", wt, xt, N, K, M, cus, limit);
        if (p.splits > 1 && N % 4) fail("skinny split reduction needs N % 4", wt, xt, N, K, M, cus, limit);
        if (xt == kF32 && p.xt != f32_operand_type(wt)) fail("skinny f32 operand type", wt, xt, N, K, M, cus, limit);
        return;
    }
    if (p.persistent) {
        if (xt == kF32 && (!p.convert_x || p.xt != f32_operand_type(wt)))
            fail("persistent f32 operand type", wt, xt, N, K, M, cus, limit);
        if (p.two_pass && M < kW16MinTokens) fail("two-pass below its token count", wt, xt, N, K, M, cus, limit);
        return;
    }
    if (p.split > 1) {
        const uint64_t tiles = (uint64_t)((M + 255) / 256) * ((N + 255) / 256);
        if (!splits_nonempty(S, p.split)) fail("tile cut without stages", wt, xt, N, K, M, cus, limit);
        if (p.split_full >= tiles || p.split_full % cus || tiles - p.split_full > (uint64_t)cus)
            fail("tiles cut are not the last round's", wt, xt, N, K, M, cus, limit);
        if (N % 4 || K % kStageK) fail("tile cut of a ragged launch", wt, xt, N, K, M, cus, limit);
        const size_t x16 = xt == kF32 ? align256((size_t)M * K * 2) : 0;
        if (p.convert_x != (xt == kF32) || p.xt != operand_type(wt, xt) || p.img_off != x16)
            fail("tile cut's activations", wt, xt, N, K, M, cus, limit);
        if (p.ws != x16 + (tiles - p.split_full) * p.split * kPartTile)
            fail("tile cut's workspace", wt, xt, N, K, M, cus, limit);
        return;
    }
    // the tiled kernel: where the few-token kernel could run instead, not by much the slower of the two
    if (M > kSkinnyMaxTokens && few_fits(wt, N, K, M) && N % 4 == 0 &&
        few_us(xt, N, K, M, cus) < 0.8 * tiled_us(wt, xt, N, K, M, cus, limit))
        fail("tiled in place of the few-token kernel", wt, xt, N, K, M, cus, limit);
    // the tiled kernel (or, Q8_0 with K % 64 == 32, the generic one: no splits)
    if (wt == kQ8_0 && K % kStageK) {
        if (p.tiles.splits != 1) fail("generic kernel split", wt, xt, N, K, M, cus, limit);
        return;
    }
    if (p.tiles.splits > 1) {
        if (!splits_nonempty(S, p.tiles.splits)) fail("tiled split without stages", wt, xt, N, K, M, cus, limit);
        if (((uint64_t)M * N) % 4) fail("tiled split reduction needs M N % 4", wt, xt, N, K, M, cus, limit);
        if (p.ws != (size_t)p.tiles.splits * M * N * 4) fail("tiled split workspace", wt, xt, N, K, M, cus, limit);
    }
}

int main() {
    // the splitting rule on its own
    for (uint32_t S = 1; S <= 300; S++)
        for (uint32_t want = 1; want <= 80; want++) {
            const uint32_t s = nonempty_splits(S, want);
            n_checked++;
            if (s < 1 || s > want || !splits_nonempty(S, s)) {
                std::printf("FAIL nonempty_splits(%u, %u) = %u\n", S, want, s);
                return 1;
            }
        }
    // the case that had an empty split: M 320, N 640, K 3072 on 256 CUs
    {
        const TilePlan t = plan_tiles(kQ8_0, 640, 3072, 320, 256);
        n_checked++;
        if (!splits_nonempty(3072 / kStageK, t.splits)) {
            std::printf("FAIL plan_tiles(320 x 640 x 3072): %u splits\n", t.splits);
            return 1;
        }
    }
    if (f32_operand_type(kQ8_0) != kF16 || f32_operand_type(kQ4K) != kBF16) {
        std::printf("FAIL f32 operand types\n");
        return 1;
    }
    // launches of either kernel that the estimates once took for the other's
    // (measured few-token : tiled, 15.5 : 8.9 us, 65 : 45, 34.9 : 25, 8.9 : 12.7)
    {
        struct {
            uint32_t wt, xt, N, K, M;
            bool few;
        } const c[] = {{kQ8_0, kF16, 12288, 256, 257, false}, {kQ8_0, kF32, 1024, 15360, 257, false},
                       {kQ4K, kF32, 64, 15360, 288, false}, {kQ8_0, kF32, 128, 3840, 350, true}};
        for (const auto& s : c) {
            n_checked++;
            if (plan_gemm(s.wt, s.xt, s.N, s.K, s.M, 256).few != s.few) {
                std::printf("FAIL %u x %u x %u: few-token kernel %d\n", s.M, s.N, s.K, !s.few);
                return 1;
            }
        }
    }
    // up to 256 tokens: which of the two few-token kernels, and its tile width (0: not the few-token kernel;
    // measured the other way: 35 : 26 us, 48 : 36, 508 : 414, 34 : 28, 23.6 : 19.6, 17.2 : 20.5)
    {
        struct {
            uint32_t wt, xt, N, K, M, features;
        } const c[] = {{kQ8_0, kF32, 1536, 8192, 200, 0},   {kQ8_0, kBF16, 2048, 15360, 150, 0},
                       {kQ8_0, kBF16, 21504, 15360, 200, 96}, {kQ8_0, kF32, 64, 15360, 150, 0},
                       {kQ8_0, kF16, 512, 15360, 5, 0},     {kQ4K, kBF16, 128, 10240, 64, 32}};
        for (const auto& s : c) {
            const GemmPlan p = plan_gemm(s.wt, s.xt, s.N, s.K, s.M, 256);
            n_checked++;
            if (p.skinny != (s.features == 0) || (p.few ? p.few_features : 0u) != s.features) {
                std::printf("FAIL %u x %u x %u: few-token tiles of %u features\n", s.M, s.N, s.K, p.few_features);
                return 1;
            }
        }
    }
    // what the GPU tests' launches run, so that each reaches the kernel it names
    {
        enum Route { kTiled, kFew32, kFew96, kSkinny, kCut, kPersist };
        const size_t none = kNoWorkspaceLimit, scratch = LLMR_NOALLOC_SCRATCH_BYTES;
        struct {
            uint32_t wt, xt, N, K, M;
            size_t limit;
            Route route;
            bool ws;
        } const c[] = {
            // test_gpu_gemm.py: test_gemm_parity, test_few_token_tiles, test_split_tiles
            {kQ8_0, kF32, 516, 8256, 33, none, kSkinny, true},    {kQ4K, kF32, 512, 8448, 100, none, kSkinny, true},
            {kQ8_0, kF16, 640, 14400, 17, none, kSkinny, true},   {kQ4K, kBF16, 1540, 8192, 200, none, kSkinny, true},
            {kQ4K, kBF16, 3077, 1024, 77, none, kFew32, false},   {kQ4K, kF32, 1028, 768, 300, none, kFew32, false},
            {kQ8_0, kBF16, 1024, 1088, 512, none, kFew32, false}, {kQ8_0, kBF16, 3072, 640, 250, none, kFew96, false},
            {kQ8_0, kF32, 3840, 3840, 1101, none, kCut, true},    {kQ4K, kF32, 3072, 3072, 1101, none, kCut, true},
            {kQ8_0, kBF16, 2052, 5120, 513, none, kCut, true},    {kQ4K, kF16, 2052, 5120, 513, none, kCut, true},
            {kQ8_0, kBF16, 11520, 1088, 1536, none, kCut, true},  {kQ4K, kBF16, 9216, 3072, 2047, none, kCut, true},
            {kQ8_0, kF16, 2052, 2048, 2049, none, kCut, true},
            {kQ4K, kF32, 256, 512, 100, none, kFew32, false},     {kQ4K, kF32, 512, 8448, 77, none, kSkinny, true},
            {kQ4K, kF32, 520, 512, 600, none, kTiled, true},
            // test_zz_no_alloc.py
            {kQ8_0, kF32, 3072, 3072, 64, scratch, kFew32, false},
            {kQ4K, kF32, 3840, 10240, 64, scratch, kSkinny, true}, {kQ4K, kF32, 3840, 10240, 33, scratch, kSkinny, true},
            {kQ4K, kF32, 4096, 1024, 2304, scratch, kPersist, true}, {kQ4K, kBF16, 12288, 3072, 2560, scratch, kPersist, false},
            {kQ4K, kBF16, 3072, 3072, 4608, scratch, kPersist, true}, {kQ4K, kBF16, 3072, 3072, 2048, scratch, kTiled, false},
            {kQ8_0, kF16, 1000, 14400, 200, scratch, kSkinny, true}, {kQ8_0, kF16, 1000, 14400, 40, scratch, kSkinny, true},
            {kQ8_0, kBF16, 3840, 5120, 600, scratch, kCut, true},  {kQ8_0, kBF16, 3840, 5120, 513, scratch, kCut, true},
            {kQ4K, kF32, 512, 10240, 64, scratch, kSkinny, true},  {kQ4K, kF32, 4096, 4096, 4608, scratch, kTiled, false},
        };
        for (const auto& s : c) {
            const GemmPlan p = plan_gemm(s.wt, s.xt, s.N, s.K, s.M, 256, s.limit);
            const Route r = p.few ? (p.few_features == kFewNarrow ? kFew32 : kFew96)
                            : p.skinny ? kSkinny : p.split > 1 ? kCut : p.persistent ? kPersist : kTiled;
            n_checked++;
            if (r != s.route || (p.ws > 0) != s.ws) {
                std::printf("FAIL %u x %u x %u: a test's launch runs kernel %d (%zu bytes), not %d\n", s.M, s.N, s.K, r,
                            p.ws, s.route);
                return 1;
            }
        }
    }
    // a limit that holds fewer parts than the launch is cut into without one
    {
        const GemmPlan a = plan_gemm(kQ8_0, kBF16, 3840, 3840, 1101, 256);
        const GemmPlan b = plan_gemm(kQ8_0, kBF16, 3840, 3840, 1101, 256, (size_t)40 << 20);
        n_checked++;
        if (a.split != 3 || b.split != 2) {
            std::printf("FAIL 1101 x 3840 x 3840: cut into %u, %u with 40 MiB\n", a.split, b.split);
            return 1;
        }
    }
    const uint32_t Ms[] = {1, 2, 4, 5, 17, 31, 32, 33, 64, 100, 200, 255, 256, 257, 320, 500, 512, 1000,
                           1024, 2047, 2048, 3000, 4096, 4352, 4608, 9000};
    const uint32_t Ns[] = {4, 60, 64, 96, 100, 256, 320, 640, 1000, 1536, 3072, 3840, 10240, 11520, 21504};
    const uint32_t Ks[] = {256, 512, 768, 1024, 3072, 3840, 10240, 15360, 32, 96, 3104};
    const int cus[] = {256, 304, 80, 8};
    const size_t limits[] = {kNoWorkspaceLimit, (size_t)32 << 20, (size_t)1 << 20, 0};
    for (uint32_t wt : {kQ8_0, kQ4K})
        for (uint32_t xt : {kF32, kF16, kBF16})
            for (uint32_t M : Ms)
                for (uint32_t N : Ns)
                    for (uint32_t K : Ks) {
                        if (wt == kQ4K && K % 256) continue;
                        if (K % 32) continue;
                        for (int c : cus)
                            for (size_t lim : limits) check(wt, xt, N, K, M, c, lim);
                    }
    std::printf("plan_check: %ld plans ok\n", n_checked);
    return 0;
}
