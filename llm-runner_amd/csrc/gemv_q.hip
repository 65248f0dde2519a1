// gemv_q.hip - dequant-GEMM for a handful of tokens (M <= 4): the
// modulation and timestep projections of a DiT step (M = 1) stream a whole
// weight matrix for a few dot products, so they are bound by HBM reads of the
// packed weight. Here every weight byte is read once and used for all M tokens.
//
// gemv_i8_kernel (below) takes Q4_K and Q8_0 weights as long as the activations
// fit its LDS; gemv_q4k_kernel is the Q4_K form for longer rows: a wave covers
// 16 weight rows, lane t (of 16) walks superblocks t, t+16, ..., and each lane
// serves 4 of the rows with one register copy of the activations it needs (a
// 64-element slice per token at a time); the 16 partial sums of a row are
// reduced with lane shuffles. Arithmetic is f32 throughout, as the reference's
// batch_matmul_q4k (llm.slang:2264-2365) with activations in f32: each weight
// is (d*sc)*q - dmin*mn with one rounding (the FMA; both products are exact).
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "llmr_device.h"
#include "llmr_internal.h"

namespace llmr {
namespace {

template <uint32_t XT>
__device__ __forceinline__ f32x4 load_x4(const void* X, uint64_t e) {
    if constexpr (XT == kGgmlF32) {
        return *(const f32x4*)((const float*)X + e);
    } else {
        const u32x2 v = *(const u32x2*)((const uint16_t*)X + e);
        if constexpr (XT == kGgmlBF16) {
            return f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                         __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
        } else {
            // the halves go through scalars: this compiler's __builtin_bit_cast
            // of a vector element (bit_cast(f16x2, v.y)) reads element 0's bits
            const uint32_t lo = v.x, hi = v.y;
            const f16x2 a = __builtin_bit_cast(f16x2, lo), b = __builtin_bit_cast(f16x2, hi);
            return f32x4{(float)a.x, (float)a.y, (float)b.x, (float)b.y};
        }
    }
}

template <uint32_t XT, int MM>
__global__ void __launch_bounds__(256) gemv_q4k_kernel(const uint8_t* __restrict__ W, const void* __restrict__ X,
                                                        float* __restrict__ Y, uint32_t N, uint32_t K, uint32_t M,
                                                        uint32_t row_offset) {
    // lane t = l % 16 walks superblocks t, t+16, ...; lane group r = l / 16
    // owns rows r, r+4, r+8, r+12 of the wave's 16: one 64-element slice of
    // the activations (per token) is loaded once and used for all four rows
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t t = lane & 15u, r = lane >> 4;
    const uint32_t n0 = blockIdx.x * 64u + wave * 16u + r;  // rows n0 + 4i, i < 4
    const uint32_t nsb = K / 256u;
    const uint64_t rb = (uint64_t)nsb * 144u;
    float acc[4][MM];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int m = 0; m < MM; ++m) acc[i][m] = 0.0f;
    for (uint32_t sb = t; sb < nsb; sb += 16u) {
        const uint64_t xb = (uint64_t)sb * 256u;
        u32x4 hdr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t n = n0 + 4u * i;
            hdr[i] = n < N ? *(const u32x4_a4*)(W + (uint64_t)(row_offset + n) * rb + (uint64_t)sb * 144u)
                           : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // activations of elements 64j .. 64j+63 of this superblock, per token
            f32x4 xl[MM][8], xh[MM][8];
#pragma unroll
            for (int m = 0; m < MM; ++m) {
                if (m < (int)M) {
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const uint64_t e = (uint64_t)m * K + xb + 64u * j + 4u * c;
                        xl[m][c] = load_x4<XT>(X, e);
                        xh[m][c] = load_x4<XT>(X, e + 32u);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t n = n0 + 4u * i;
                if (n >= N) continue;
                const uint32_t* b = (const uint32_t*)(W + (uint64_t)(row_offset + n) * rb + (uint64_t)sb * 144u);
                const u32x4 q0 = *(const u32x4_a4*)(b + 4 + 8 * j), q1 = *(const u32x4_a4*)(b + 8 + 8 * j);
                const float d = f16_bits_to_f32(hdr[i].x & 0xffffu), dmin = f16_bits_to_f32(hdr[i].x >> 16);
                uint32_t sc0, mn0, sc1, mn1;
                q4k_scale_min(2u * j, hdr[i].y, hdr[i].z, hdr[i].w, sc0, mn0);
                q4k_scale_min(2u * j + 1u, hdr[i].y, hdr[i].z, hdr[i].w, sc1, mn1);
                const float d0 = d * (float)sc0, m0 = dmin * (float)mn0;
                const float d1 = d * (float)sc1, m1 = dmin * (float)mn1;
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    // bytes 4c .. 4c+3 of the pair's 32 quant bytes: elements
                    // 64j + 4c + k (low nibble) and 64j + 32 + 4c + k (high)
                    const uint32_t word = c < 4 ? q0[c] : q1[c - 4];
                    f32x4 wl, wh;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t q = (word >> (8 * k)) & 0xffu;
                        wl[k] = __builtin_fmaf((float)(q & 15u), d0, -m0);
                        wh[k] = __builtin_fmaf((float)(q >> 4), d1, -m1);
                    }
#pragma unroll
                    for (int m = 0; m < MM; ++m) {
                        if (m < (int)M) {
                            const f32x4 a = xl[m][c], h = xh[m][c];
                            acc[i][m] += (wl.x * a.x + wl.y * a.y) + (wl.z * a.z + wl.w * a.w) +
                                         ((wh.x * h.x + wh.y * h.y) + (wh.z * h.z + wh.w * h.w));
                        }
                    }
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int m = 0; m < MM; ++m) {
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) acc[i][m] += __shfl_xor(acc[i][m], o, 64);
        }
    if (t == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t n = n0 + 4u * i;
            if (n < N) {
#pragma unroll
                for (int m = 0; m < MM; ++m)
                    if (m < (int)M) Y[(uint64_t)m * N + n] = acc[i][m];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// gemv_i8_kernel: the same products on the integer matrix cores.
//
// What bounds a projection of 1-4 tokens is the weight stream, if the vector
// ALU keeps up: one FMA per weight on the nibble as a float took 3.6 VALU
// instructions per weight and lane (18 us for the 31.9 MB of 18432 x 3072).
// Here a 4x4x4 int8 MFMA (16 blocks of 4 x 4 outputs over 4 k each) multiplies
// the quants as they are with the activations cut into four int8 digits:
//  * a Q4_K nibble masked in place is an int8 (3 instructions for 8 weights), a
//    Q8_0 quant is one already;
//  * each activation, scaled by a power of two so that its 32-element
//    sub-block's largest lies in [2^29, 2^30) and rounded to an integer (31
//    bits under the largest), is the sum of four signed base-256 digits; sums of
//    quant x digit over a sub-block are exact in int32, and the four of them
//    make one f32 with a single rounding (Q8_0, whose pairs of sums pass 2^24:
//    with up to three);
//  * Q4_K: acc += (d sc) sum (q - c) x - (dmin mn - c d sc) sum x with c the quant
//    whose weight is nearest zero; the first sum is exact (c times the
//    activations' digit sums off the products). Both terms are then of the size of
//    the weights times x, and a zero weight's activation is in neither: one 300
//    times the rest of its sub-block leaves 0.9-2.1e-7 (8 for every c: 2-7e-6).
// That is at least as exact as f32 FMAs on f32 activations (18432 x 3072: 1.4e-7
// relative to 64 bits, the FMA kernel 2.5e-7), as long as the digits hold what is
// multiplied. Where they do not, a workgroup multiplies in f32 (gemv_f32_rows): an
// infinite or NaN activation; f16 and bf16 values, other than zeros, that are not
// whole (below 2^10 and 2^7 units of the digits); f32 values below 2^20 units, 2^9
// to 2^10 under their sub-block's largest, that fill a quarter of it, or one below
// 2^8; a sub-block under 2^-97, for which no scale is a normal number. With an
// activation 2^k times the rest of its sub-block under a zero weight the digits'
// error is, for k = 8, 10, 12 and 20, 1.1e-7, 3.5e-7, 9.6e-7 and 7.7e-4, the
// FMAs' 0.9e-7; with activations of 1e-33 2.8e-6 and 1.8e-7. (Of 3072 normal
// deviates one lies below 2^8 units in 1 of 500 draws.)
// A wave owns 16 weight rows and walks them 4 units at a time: lane l = 16 rq +
// 4 g + j has row 4 rq + j and unit g, so the four lanes of an MFMA block share
// a unit. One token: the block's four rows of A are the token's digits; two to
// four tokens: A's rows are the tokens, one MFMA per digit. The weight bytes are
// loaded 16 bytes a lane along the rows (whole lines) a step ahead and change
// lanes through the wave's own LDS region (a lane reads its 144 or 136 bytes at
// conflict-free strides); no barrier in the loop. At one token and K = 3072 the
// LDS holds three workgroups per CU. KS waves share 16 rows (each takes every
// KS-th step), so that launches of few rows still put work on every CU.
// Measured per call, before -> after (one token, FMA kernel; Q8_0, the few-token
// GEMMs): 18432 x 3072 Q4_K 19.5 -> 8.9 us (3.6 TB/s), 38 of them grouped 328
// -> 210 us (5.8 TB/s), 3072 x 15360 76 -> 12, two and four tokens of 18432 x
// 3072 31 -> 14 and 56 -> 17 us; 11520 x 3840 Q8_0 54 -> 9.8 us (4.8 TB/s).
// At three and four tokens over more rows than 64 a CU the Q8_0 few-token GEMM is
// the faster one from K = 4096 on (18432 x 6144 27 against 31 us), with the
// activations rounded to fp16: 2e-4 against 64 bits where this leaves 1e-7.
// ---------------------------------------------------------------------------

// Up to CAP projections of one shape [N, K] (each its own weight, input
// and output rows, ldy apart): workgroup b serves rows (64 / KS) (b % bpj) .. of
// job b / bpj. CAP = 1 for one projection, kGemvMaxJobs for a group.
constexpr uint32_t kGemvMaxJobs = 64;
template <uint32_t CAP>
struct GemvJobs {
    const uint8_t* w[CAP];
    const void* x[CAP];
    float* y[CAP];
    uint32_t m[CAP], row_offset[CAP];
};

// A lane's unit: a Q4_K super-block (256 k, 144 bytes) or four Q8_0 blocks
// (128 k, 136 bytes; eight would keep the third workgroup off the CU). A step of
// a wave is 16 rows x 4 units, loaded as 16-byte pieces along the rows.
template <uint32_t WT>
struct GemvW {
    static constexpr uint32_t kK = WT == kGgmlQ4K ? 256u : 128u, kBytes = WT == kGgmlQ4K ? 144u : 136u;
    static constexpr uint32_t kStep = 64u * kBytes, kRowPieces = 4u * kBytes / 16u;
    static constexpr uint32_t kLoads = (16u * kRowPieces + 63u) / 64u;  // pieces per lane (Q8_0: half of the last)
};

// LDS of the activations per unit, T token slots (1, 2 or 4). Digits: 16 k at a
// time, [digit][token][16 bytes]. Then per sub-block and token: Q4_K, the sums of
// its two upper and two lower digits, 1 / scale, activation sum; Q8_0, 1 / scale.
// Units are padded so the four a wave reads together lie 64 bytes apart in the
// banks.
template <uint32_t WT, int T>
struct GemvX {
    static constexpr uint32_t kSub = GemvW<WT>::kK / 32u;
    static constexpr uint32_t kDigits = GemvW<WT>::kK / 16u * (64u * T);
    static constexpr uint32_t kTok = WT == kGgmlQ4K ? 16u : 8u, kSubBytes = kTok * T;
    static constexpr uint32_t kUsed = kDigits + kSub * kSubBytes, kUnit = kUsed + (320u - kUsed % 256u) % 256u;
};
// the activations as f32 in the same region: 16 bytes of padding every 64 k, so
// that pieces 256 bytes apart lie in other banks
constexpr uint32_t gemv_xs(uint32_t k) { return k + k / 64u * 4u; }
template <uint32_t WT, int T>
constexpr bool gemv_xs_fits = gemv_xs(GemvW<WT>::kK) * T * 4u <= GemvX<WT, T>::kUnit;
static_assert(gemv_xs_fits<kGgmlQ4K, 1> && gemv_xs_fits<kGgmlQ4K, 2> && gemv_xs_fits<kGgmlQ4K, 4> &&
              gemv_xs_fits<kGgmlQ8_0, 1> && gemv_xs_fits<kGgmlQ8_0, 2> && gemv_xs_fits<kGgmlQ8_0, 4>);
constexpr uint32_t kGemvLdsLimit = 160u * 1024u;
template <uint32_t WT, int T>
constexpr uint32_t gemv_lds_bytes(uint32_t K, uint32_t waves) {
    const uint32_t nu4 = (K / GemvW<WT>::kK + 3u) / 4u * 4u;
    return nu4 * GemvX<WT, T>::kUnit + waves * GemvW<WT>::kStep + 16u;
}

// The same rows in f32, for activations that have no digits: each weight with
// one rounding ((d sc) q - dmin mn; d q), one FMA per token. xs: the token's
// activations as f32 in LDS, [token][gemv_xs(K)]. 16 lanes per row, RPL rows a lane, a piece
// of 32 weights at a time (Q4_K: 16 bytes of quants, their low nibbles one
// sub-block's and the high ones the next's; Q8_0: a block), the next piece's
// bytes in flight. Bound by the vector ALU: one infinite activation, 18432 x
// 3072 Q4_K 206 -> 19 us (a byte-wise load per weight, a row per wave before), four
// tokens 984 -> 59, 11520 x 3840 Q8_0 390 -> 16.
template <uint32_t WT>
struct GemvPiece {
    u32x4 a, b;
    uint32_t c;  // Q8_0: the block's last two quants
    __device__ __forceinline__ void load(const uint8_t* row, uint32_t p) {
        if constexpr (WT == kGgmlQ4K) {
            const uint8_t* const w = row + p / 8u * 144u;
            a = *(const u32x4_a4*)w;
            b = *(const u32x4_a4*)(w + 16u + 16u * (p % 8u));
        } else {  // from the dword that holds the scale: 36 bytes, never past the row
            const uint8_t* const w = row + 34u * p - 2u * (p & 1u);
            a = *(const u32x4_a4*)w;
            b = *(const u32x4_a4*)(w + 16u);
            c = *(const uint32_t*)(w + 32u);
        }
    }
};
template <uint32_t WT, int T, int RPL>
__device__ __forceinline__ void gemv_f32_rows(const uint8_t* W, const float* xs, float* Y, uint32_t n0, uint32_t N,
                                              uint32_t K, uint32_t rb, uint32_t M, uint32_t ldy, uint32_t lane) {
    const uint32_t t = lane & 15u, pieces = K / 32u;
    n0 += lane >> 4;  // rows n0 + 4 i; those past N read row N - 1 and are not stored
    const uint8_t* row[RPL];
    GemvPiece<WT> nxt[RPL];
    float acc[T][RPL];
#pragma unroll
    for (int i = 0; i < RPL; i++) {
        row[i] = W + (uint64_t)min(n0 + 4u * i, N - 1u) * rb;
        nxt[i].load(row[i], min(t, pieces - 1u));
#pragma unroll
        for (int m = 0; m < T; m++) acc[m][i] = 0.0f;
    }
    for (uint32_t p = t; p < pieces; p += 16u) {
        GemvPiece<WT> w[RPL];
        float d[RPL][2], mn[RPL][2], sum[T][RPL];  // Q4_K: of the low and the high nibbles
#pragma unroll
        for (int i = 0; i < RPL; i++) {
            w[i] = nxt[i];
            nxt[i].load(row[i], min(p + 16u, pieces - 1u));
            if constexpr (WT == kGgmlQ4K) {
                const u32x4 h = w[i].a;
#pragma unroll
                for (uint32_t e = 0; e < 2; e++) {
                    uint32_t sc, mi;
                    q4k_scale_min(2u * (p % 8u / 2u) + e, h.y, h.z, h.w, sc, mi);
                    d[i][e] = f16_bits_to_f32(h.x & 0xffffu) * (float)sc;
                    mn[i][e] = f16_bits_to_f32(h.x >> 16) * (float)mi;
                }
            } else {
                d[i][0] = f16_bits_to_f32(p & 1u ? w[i].a.x >> 16 : w[i].a.x & 0xffffu);
            }
#pragma unroll
            for (int m = 0; m < T; m++) sum[m][i] = 0.0f;
        }
        // elements 4 c .. of the piece: Q4_K c < 4 the low nibbles, then the high ones, 32 k on
        const uint32_t k0 = WT == kGgmlQ4K ? p / 2u * 64u + 16u * (p % 2u) : 32u * p;
#pragma unroll
        for (uint32_t c = 0; c < 8; c++) {
            f32x4 wv[RPL];
#pragma unroll
            for (int i = 0; i < RPL; i++) {
                if constexpr (WT == kGgmlQ4K) {
                    const uint32_t q = (w[i].b[c % 4u] >> (c < 4 ? 0 : 4)) & 0x0f0f0f0fu;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        wv[i][e] = __builtin_fmaf((float)((q >> (8 * e)) & 0xffu), d[i][c / 4u], -mn[i][c / 4u]);
                } else {
                    const uint32_t w9[9] = {w[i].a.x, w[i].a.y, w[i].a.z, w[i].a.w, w[i].b.x,
                                            w[i].b.y, w[i].b.z, w[i].b.w, w[i].c};
                    const uint32_t q = p & 1u ? w9[c + 1] : __builtin_amdgcn_alignbyte(w9[c + 1], w9[c], 2);
#pragma unroll
                    for (int e = 0; e < 4; e++) wv[i][e] = (float)(int8_t)(q >> (8 * e)) * d[i][0];
                }
            }
            const uint32_t k = k0 + (WT == kGgmlQ4K ? (c & 3u) * 4u + (c >> 2) * 32u : 4u * c);
#pragma unroll
            for (int m = 0; m < T; m++) {
                if ((uint32_t)m >= M) continue;
                const f32x4 x = *(const f32x4*)(xs + m * gemv_xs(K) + gemv_xs(k));
#pragma unroll
                for (int i = 0; i < RPL; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) sum[m][i] = __builtin_fmaf(wv[i][e], x[e], sum[m][i]);
            }
        }
#pragma unroll
        for (int m = 0; m < T; m++)
#pragma unroll
            for (int i = 0; i < RPL; i++) acc[m][i] += sum[m][i];
    }
#pragma unroll
    for (int m = 0; m < T; m++)
#pragma unroll
        for (int i = 0; i < RPL; i++) {
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) acc[m][i] += __shfl_xor(acc[m][i], o, 64);
            if (t == 0 && n0 + 4u * i < N && (uint32_t)m < M) Y[(uint64_t)m * ldy + n0 + 4u * i] = acc[m][i];
        }
}

typedef int i32x4 __attribute__((ext_vector_type(4)));

// v of lane ^ 1 or lane ^ 2, without the LDS round trip of a shuffle
template <int X, typename V>
__device__ __forceinline__ V quad_xor(V v) {
    static_assert(X == 1 || X == 2, "within a quad");
    return __builtin_bit_cast(
        V, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), X == 1 ? 0xb1 : 0x4e, 15, 15, false));
}

// `waves`: of a workgroup, 4 to 8 (KS == 1; gemv_waves), else 4.
template <uint32_t WT, uint32_t XT, int T, uint32_t CAP, uint32_t KS>
__global__ void __launch_bounds__(512, T == 1 ? 3 : 2) gemv_i8_kernel(const GemvJobs<CAP> jobs, uint32_t N, uint32_t K,
                                                          uint32_t ldy, uint32_t bpj, uint32_t waves) {
    static_assert(T == 1 || T == 2 || T == 4, "one token, two, or up to four");
    typedef GemvW<WT> GW;
    typedef GemvX<WT, T> GX;
    const uint32_t job = CAP == 1u ? 0u : blockIdx.x / bpj;
    const uint32_t blk = CAP == 1u ? blockIdx.x : blockIdx.x - job * bpj;
    const void* __restrict__ X = jobs.x[job];
    float* __restrict__ Y = jobs.y[job];
    const uint32_t M = jobs.m[job];
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t nu = K / GW::kK, steps = (nu + 3u) / 4u, nu4 = 4u * steps;
    const uint32_t nw = KS == 1u ? waves : 4u, threads = 64u * nw, rows = 16u * nw / KS;  // of the workgroup
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const wsb = smem + nu4 * GX::kUnit;
    uint8_t* const ws = wsb + wave * GW::kStep;           // the wave's weight bytes of a step
    uint32_t* const odd = (uint32_t*)(wsb + nw * GW::kStep);  // the activations have no digits: f32 rows
    if (tid == 0) *odd = 0u;

    // activations: thread -> 8 k of one token, four neighbours a sub-block; the
    // first pieces (all of them up to K = 4096) are requested before the weights
    // (loads return in order: behind the weights they would wait for them)
    const uint32_t pieces = nu4 * (GW::kK / 8u), total = pieces * (uint32_t)T;
    struct X8 {
        f32x4 a, b;
    };
    auto load_x = [&](uint32_t i) __attribute__((always_inline)) {
        X8 v{};
        const uint32_t m = T == 1 ? 0u : i / pieces, k = 8u * (T == 1 ? i : i - m * pieces);
        if (i < total && m < M && k < K) {
            v.a = load_x4<XT>(X, (uint64_t)m * K + k);
            v.b = load_x4<XT>(X, (uint64_t)m * K + k + 4u);
        }
        return v;
    };
    constexpr uint32_t kAhead = T == 1 ? 2u : T == 2 ? 4u : 8u;
    X8 xa[kAhead];
#pragma unroll
    for (uint32_t q = 0; q < kAhead; q++) xa[q] = load_x(tid + threads * q);

    // the wave's 16 rows as a buffer: rows past N read as zero
    const uint32_t n0 = blk * rows + wave / KS * 16u, rb = nu * GW::kBytes;
    const uint8_t* const W = jobs.w[job] + (uint64_t)jobs.row_offset[job] * rb;
    const uint32_t wbytes = n0 < N ? min(16u, N - n0) * rb : 0u;
    uint32_t voff[GW::kLoads];  // piece c = 64 i + lane of a step: row c / kRowPieces, 16 (c % kRowPieces) bytes in
#pragma unroll
    for (uint32_t i = 0; i < GW::kLoads; i++) {
        const uint32_t c = 64u * i + lane, r = c / GW::kRowPieces;
        voff[i] = r < 16u ? r * rb + 16u * (c - r * GW::kRowPieces) : 0x80000000u;
    }
    struct Set {
        u32x4 v[GW::kLoads];
    };
    // (the last step may read into the next row: those units are masked below; past
    // the last row the buffer ends, and there the step's offset is added to the
    // lane's, as the range check need not cover a scalar offset. Added at every step
    // it took 3% longer, 9216 x 12288 Q8_0 22.4 -> 23.0 us, a descriptor moved by it
    // 28.7; with 16 rows shared by the waves the branch costs more, 3072 x 8192 8.0
    // -> 8.7)
    auto load_w = [&](uint32_t s) __attribute__((always_inline)) {
        Set w;
        const uint32_t at = 4u * GW::kBytes * s;
        const rsrc_t r = make_rsrc(W + (uint64_t)n0 * rb, s < steps ? wbytes : 0u);
        if (KS > 1u || 4u * (s + 1u) > nu) {
#pragma unroll
            for (uint32_t i = 0; i < GW::kLoads; i++)
                w.v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff[i] + at, 0, 0));
        } else {
#pragma unroll
            for (uint32_t i = 0; i < GW::kLoads; i++)
                w.v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff[i], at, 0));
        }
        return w;
    };
    const uint32_t s0 = wave % KS;
    Set set = load_w(s0);
    __syncthreads();  // odd is cleared

    bool bad = false;
    constexpr float kLow = XT == kGgmlF32 ? 0x1p20f : XT == kGgmlF16 ? 0x1p10f : 0x1p7f;
    constexpr float kTiny = XT == kGgmlF32 ? 0x1p8f : kLow;
    auto stage_x = [&](uint32_t i, const X8& v) __attribute__((always_inline)) {
        const float x[8] = {v.a.x, v.a.y, v.a.z, v.a.w, v.b.x, v.b.y, v.b.z, v.b.w};
        float mx = 0.0f, sum = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        bad = bad || !(__builtin_fabsf(sum) < INFINITY);  // (sums that overflow: the f32 rows too)
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, __builtin_fabsf(x[e]));
        mx = fmaxf(mx, quad_xor<1>(mx));
        sum += quad_xor<1>(sum);
        mx = fmaxf(mx, quad_xor<2>(mx));
        sum += quad_xor<2>(sum);
        // scale 2^e with 2^e mx in [2^29, 2^30), e kept where 2^e and 2^-e are normal
        const int e = min(126, max(-126, 156 - (int)((__float_as_uint(mx) >> 23) & 0xffu)));
        const float up = __uint_as_float((uint32_t)(127 + e) << 23), down = __uint_as_float((uint32_t)(127 - e) << 23);
        // values whose digits hold too few of their bits, zeros aside (magnitude
        // bits less one: a zero's are the largest)
        const uint32_t low_bits = 2u * __float_as_uint(kLow * down) - 1u;
        uint32_t low = 0u, least = ~0u;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const uint32_t b = 2u * __float_as_uint(x[q]) - 1u;
            low += b < low_bits ? 1u : 0u;
            least = min(least, b);
        }
        low += quad_xor<1>(low);
        low += quad_xor<2>(low);
        bad = bad || low >= 8u || least < 2u * __float_as_uint(kTiny * down) - 1u || (mx > 0.0f && mx < 0x1p-97f);
        uint32_t dg[2][4];  // [four k][digit, lowest first]: a byte per k
        int sums[4] = {0, 0, 0, 0};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t v4[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                // |v| < 2^30 + 1: adding 0x808080 and flipping those bits turns the
                // three low bytes into signed digits (the carries go up)
                const int i32 = (int)rintf(x[4 * h + q] * up);
                v4[q] = ((uint32_t)i32 + 0x00808080u) ^ 0x00808080u;
            }
            // 4 x 4 byte transpose
            const uint32_t a0 = __builtin_amdgcn_perm(v4[1], v4[0], 0x05010400u);  // b0 b0' b1 b1'
            const uint32_t a1 = __builtin_amdgcn_perm(v4[1], v4[0], 0x07030602u);  // b2 b2' b3 b3'
            const uint32_t c0 = __builtin_amdgcn_perm(v4[3], v4[2], 0x05010400u);
            const uint32_t c1 = __builtin_amdgcn_perm(v4[3], v4[2], 0x07030602u);
            dg[h][0] = __builtin_amdgcn_perm(c0, a0, 0x05040100u);
            dg[h][1] = __builtin_amdgcn_perm(c0, a0, 0x07060302u);
            dg[h][2] = __builtin_amdgcn_perm(c1, a1, 0x05040100u);
            dg[h][3] = __builtin_amdgcn_perm(c1, a1, 0x07060302u);
            if constexpr (WT == kGgmlQ4K)
#pragma unroll
                for (int p = 0; p < 4; p++) sums[p] = __builtin_amdgcn_sdot4((int)dg[h][p], 0x01010101, sums[p], false);
        }
        if constexpr (WT == kGgmlQ4K)
#pragma unroll
            for (int p = 0; p < 4; p++) {
                sums[p] += quad_xor<1>(sums[p]);
                sums[p] += quad_xor<2>(sums[p]);
            }
        if (i >= total) return;
        const uint32_t m = T == 1 ? 0u : i / pieces, c = T == 1 ? i : i - m * pieces;  // chunk of 8 k
        const uint32_t u = c / (GW::kK / 8u), cu = c % (GW::kK / 8u);
        uint8_t* const dst = smem + u * GX::kUnit + cu / 2u * (64u * T) + m * 16u + 8u * (cu & 1u);
#pragma unroll
        for (int p = 0; p < 4; p++) *(u32x2*)(dst + p * (16u * T)) = u32x2{dg[0][p], dg[1][p]};
        if (cu % 4u == 0u) {
            uint8_t* const sb = smem + u * GX::kUnit + GX::kDigits + cu / 4u * GX::kSubBytes + GX::kTok * m;
            if constexpr (WT == kGgmlQ4K)
                *(f32x4*)sb = f32x4{(float)(sums[3] * 256 + sums[2]), (float)(sums[1] * 256 + sums[0]), down, sum};
            else
                *(float*)sb = down;
        }
    };
#pragma unroll
    for (uint32_t q = 0; q < kAhead; q++)
        if (threads * q < total) stage_x(tid + threads * q, xa[q]);
    for (uint32_t i = threads * kAhead; i < total; i += threads) stage_x(i + tid, load_x(i + tid));  // (whole waves)
    if (bad) *odd = 1u;
    __syncthreads();
    if (*odd != 0u) {  // a whole workgroup's branch: nothing below waits for it
        // (the last read of odd and of the digits lies behind every thread's barrier)
        float* const xs = (float*)smem;
        for (uint32_t i = 4u * tid; i < M * K; i += 4u * threads) *(f32x4*)(xs + gemv_xs(i)) = load_x4<XT>(X, i);
        __syncthreads();
        gemv_f32_rows<WT, T, 4 / KS>(W, xs, Y, blk * rows + wave * (16u / KS), N, K, rb, M, ldy, lane);
        return;
    }

    const uint32_t j = lane & 3u, g = (lane >> 2) & 3u, rq = lane >> 4;
    const uint8_t* const wl = ws + ((4u * rq + j) * 4u + g) * GW::kBytes;
    float acc[T];
#pragma unroll
    for (int m = 0; m < T; m++) acc[m] = 0.0f;
    constexpr int P = T == 1 ? 1 : 4;  // accumulator tiles: [digits] of one token, or [tokens] per digit

    // D += A B for 16 k of two sub-blocks at once (independent accumulators, so
    // the MFMAs follow each other): w the lane's quants (16 bytes), xb the
    // unit's digits of these 16 k; this lane's row of A is digit j (one token)
    // or token j
    auto mul16 = [&](i32x4 (&d)[P], const uint8_t* xb, u32x4 w, i32x4 (&d2)[P], const uint8_t* xb2, u32x4 w2)
        __attribute__((always_inline)) {
        u32x4 a[P], a2[P];
#pragma unroll
        for (int p = 0; p < P; p++) {
            const uint32_t at = 16u * T * p + (T == 1 ? 16u * j : 16u * (j % T));
            a[p] = *(const u32x4*)(xb + at);
            a2[p] = *(const u32x4*)(xb2 + at);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
#pragma unroll
            for (int p = 0; p < P; p++) d[p] = __builtin_amdgcn_mfma_i32_4x4x4i8((int)a[p][q], (int)w[q], d[p], 0, 0, 0);
#pragma unroll
            for (int p = 0; p < P; p++)
                d2[p] = __builtin_amdgcn_mfma_i32_4x4x4i8((int)a2[p][q], (int)w2[q], d2[p], 0, 0, 0);
        }
    };
    // acc += ds (sum (q - c) x) - dm (sum x) of one sub-block
    auto add = [&](const i32x4 (&d)[P], const uint8_t* sb, float ds, float dm, float c) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < T; m++) {
            const int d0 = T == 1 ? d[0].x : d[0][m], d1 = T == 1 ? d[0].y : d[1 % P][m];
            const int d2 = T == 1 ? d[0].z : d[2 % P][m], d3 = T == 1 ? d[0].w : d[3 % P][m];
            float hi = (float)(d3 * 256 + d2), lo = (float)(d1 * 256 + d0);
            if constexpr (WT == kGgmlQ4K) {
                // quants to 15: both pairs, c times the digits' and the differences
                // are whole numbers below 2^24, so only t rounds
                const f32x4 s = *(const f32x4*)(sb + GX::kTok * m);
                const float t = __builtin_fmaf(__builtin_fmaf(-c, s.x, hi), 65536.0f, __builtin_fmaf(-c, s.y, lo));
                acc[m] = __builtin_fmaf(-dm, s.w, __builtin_fmaf(ds * t, s.z, acc[m]));
            } else {  // (quants to 127: the pairs reach 2^27 and round)
                const float down = *(const float*)(sb + GX::kTok * m);
                acc[m] = __builtin_fmaf(ds * __builtin_fmaf(hi, 65536.0f, lo), down, acc[m]);
            }
        }
    };

    for (uint32_t s = s0; s < steps; s += KS) {
        // the step's bytes into the wave's region (its reads of the step before
        // are done: a wave's LDS accesses run in order), the next step's loads out
#pragma unroll
        for (uint32_t i = 0; i < GW::kLoads; i++)
            if (64u * i + 63u < 16u * GW::kRowPieces || 64u * i + lane < 16u * GW::kRowPieces)
                *(u32x4*)(ws + 1024u * i + 16u * lane) = set.v[i];
        set = load_w(s + KS);
        const uint32_t u = 4u * s + g;
        const bool live = u < nu;  // (a unit past the row adds 0)
        const uint8_t* const xb = smem + u * GX::kUnit;
        const uint8_t* const sb = xb + GX::kDigits;
        if constexpr (WT == kGgmlQ4K) {
            const u32x4 h = *(const u32x4*)wl;
            const uint32_t s0w = h.y, s1w = h.z, s2w = h.w;
            const float dd = live ? f16_bits_to_f32(h.x & 0xffffu) : 0.0f;
            const float dmin = live ? f16_bits_to_f32(h.x >> 16) : 0.0f;
            // get_scale_min_k4 of the eight sub-blocks, four bytes at a time
            const uint32_t sc4[2] = {s0w & 0x3f3f3f3fu, (s2w & 0x0f0f0f0fu) | ((s0w >> 2) & 0x30303030u)};
            const uint32_t mn4[2] = {s1w & 0x3f3f3f3fu, ((s2w >> 4) & 0x0f0f0f0fu) | ((s1w >> 2) & 0x30303030u)};
            float ds[8], dm[8], c[8];
#pragma unroll
            for (int b = 0; b < 8; b++) {
                ds[b] = dd * (float)((sc4[b >> 2] >> (8u * (b & 3u))) & 0xffu);
                dm[b] = dmin * (float)((mn4[b >> 2] >> (8u * (b & 3u))) & 0xffu);
                // (any c from 0 to 15 gives the same sum: a ds of 0 may take either end)
                c[b] = (float)(uint32_t)__builtin_amdgcn_fmed3f(
                    __builtin_fmaf(dm[b], __builtin_amdgcn_rcpf(ds[b]), 0.5f), 0.0f, 15.5f);
                dm[b] = __builtin_fmaf(-c[b], ds[b], dm[b]);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {  // sub-blocks 2q (low nibbles) and 2q + 1 (high)
                __builtin_amdgcn_sched_barrier(0);  // one quarter's operands at a time
                const u32x4 qa = *(const u32x4*)(wl + 16u + 32u * q), qb = *(const u32x4*)(wl + 32u + 32u * q);
                const u32x4 m4 = {0x0f0f0f0fu, 0x0f0f0f0fu, 0x0f0f0f0fu, 0x0f0f0f0fu};
                i32x4 lo[P], hi[P];
#pragma unroll
                for (int p = 0; p < P; p++) lo[p] = hi[p] = i32x4{0, 0, 0, 0};
                mul16(lo, xb + (4u * q) * (64u * T), qa & m4, hi, xb + (4u * q + 2u) * (64u * T), (qa >> 4) & m4);
                mul16(lo, xb + (4u * q + 1u) * (64u * T), qb & m4, hi, xb + (4u * q + 3u) * (64u * T), (qb >> 4) & m4);
#pragma unroll
                for (int e = 0; e < 2; e++)
                    add(e ? hi : lo, sb + (2u * q + e) * GX::kSubBytes, ds[2 * q + e], dm[2 * q + e], c[2 * q + e]);
            }
        } else {
            // four blocks of 34 bytes: block b's scale at byte 34 b, its quants two bytes on
            uint32_t wd[34];
#pragma unroll
            for (int i = 0; i < 17; i++) {
                const u32x2 v = *(const u32x2*)(wl + 8u * i);
                wd[2 * i] = v.x;
                wd[2 * i + 1] = v.y;
            }
#pragma unroll
            for (int b = 0; b < 4; b += 2) {  // block b's quants lie two bytes past a dword, block b + 1's on one
                __builtin_amdgcn_sched_barrier(0);
                const int dw = 17 * (b / 2);
                uint32_t q[8], q2[8];  // quant bytes 4 i .. 4 i + 3 of each block
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    q[i] = __builtin_amdgcn_alignbyte(wd[dw + i + 1], wd[dw + i], 2);
                    q2[i] = wd[dw + 9 + i];
                }
                i32x4 t[P], t2[P];
#pragma unroll
                for (int p = 0; p < P; p++) t[p] = t2[p] = i32x4{0, 0, 0, 0};
#pragma unroll
                for (int h = 0; h < 2; h++)
                    mul16(t, xb + (2u * b + h) * (64u * T), u32x4{q[4 * h], q[4 * h + 1], q[4 * h + 2], q[4 * h + 3]},
                          t2, xb + (2u * b + 2u + h) * (64u * T),
                          u32x4{q2[4 * h], q2[4 * h + 1], q2[4 * h + 2], q2[4 * h + 3]});
                add(t, sb + b * GX::kSubBytes, live ? f16_bits_to_f32(wd[dw] & 0xffffu) : 0.0f, 0.0f, 0.0f);
                add(t2, sb + (b + 1) * GX::kSubBytes, live ? f16_bits_to_f32(wd[dw + 8] >> 16) : 0.0f, 0.0f, 0.0f);
            }
        }
    }

    // the four unit lanes of a row, then the KS waves, in wave order
    const uint32_t r = 4u * rq + j;
#pragma unroll
    for (int m = 0; m < T; m++) {
        acc[m] += __shfl_xor(acc[m], 4, 64);
        acc[m] += __shfl_xor(acc[m], 8, 64);
    }
    if constexpr (KS > 1) {
        float* const red = (float*)wsb;  // [wave][token][row], over the waves' weight regions
        __syncthreads();
        if (g == 0)
#pragma unroll
            for (int m = 0; m < T; m++) red[(wave * T + m) * 16u + r] = acc[m];
        __syncthreads();
        for (uint32_t i = tid; i < rows * T; i += threads) {
            const uint32_t row = i % rows, m = i / rows, w0 = row / 16u * KS, n = blk * rows + row;
            float v = red[(w0 * T + m) * 16u + row % 16u];
#pragma unroll
            for (uint32_t w = 1; w < KS; w++) v += red[((w0 + w) * T + m) * 16u + row % 16u];
            if (n < N && m < M) Y[(uint64_t)m * ldy + n] = v;
        }
    } else {
#pragma unroll
        for (int m = 0; m < T; m++)
            if (g == 0 && n0 + r < N && (uint32_t)m < M) Y[(uint64_t)m * ldy + n0 + r] = acc[m];
    }
}

// Whether gemv_i8_kernel takes M tokens x K: whole super-blocks (Q8_0 rows in
// whole 16-byte pieces) and the digits in LDS.
template <uint32_t WT>
bool gemv_fits(uint32_t K, uint32_t M) {
    if (M == 0 || M > kGemvMaxTokens || K % 256u || K == 0 || K > (1u << 20)) return false;
    return (M == 1 ? gemv_lds_bytes<WT, 1>(K, 4u) : M == 2 ? gemv_lds_bytes<WT, 2>(K, 4u) : gemv_lds_bytes<WT, 4>(K, 4u)) <=
           kGemvLdsLimit;
}

// Waves of a workgroup, 16 rows each, for one projection: as few from 4 on as
// give every CU at most one workgroup (beside the activations' digits the LDS holds
// one to three of 4 waves, and each cuts the digits anew), 4 where 8 do not.
// 18432 rows are 288 workgroups of 4 and 231 of 5: x 3072 Q8_0 at one, two and four
// tokens 13.8, 18.2, 29.5 -> 12.3, 15.6, 18.5 us, x 6144 24, 44, 55 -> 22, 28, 34, x
// 12288 Q4_K at one 47 -> 30. With two full rounds more waves gain nothing (36864 x
// 3072 Q4_K, two tokens: 24.5 us with 4, 28.6 with 5).
template <uint32_t WT, int T>
uint32_t gemv_waves(uint32_t N, uint32_t K, int num_cus) {
    for (uint32_t w = 4; w <= 8 && gemv_lds_bytes<WT, T>(K, w) <= kGemvLdsLimit; w++)
        if ((N + 16u * w - 1u) / (16u * w) <= (uint32_t)num_cus) return w;
    return 4;
}

template <uint32_t WT, uint32_t XT, int T, uint32_t CAP, uint32_t KS>
hipError_t launch_gemv_k(const GemvJobs<CAP>& jobs, uint32_t n_jobs, uint32_t N, uint32_t K, uint32_t ldy,
                         uint32_t waves, hipStream_t st) {
    auto kern = gemv_i8_kernel<WT, XT, T, CAP, KS>;
    // more than 64 KiB of LDS: an attribute of the kernel on each device
    static std::atomic<uint64_t> allowed{0};  // by device
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = dev < 64 ? 1ull << dev : 0ull;
    if (!(allowed.load(std::memory_order_acquire) & bit)) {
        e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGemvLdsLimit);
        if (e != hipSuccess) return e;
        allowed.fetch_or(bit, std::memory_order_release);
    }
    const uint32_t rows = 16u * waves / KS, bpj = (N + rows - 1u) / rows;
    hipLaunchKernelGGL(kern, dim3(bpj * n_jobs), dim3(64u * waves), (gemv_lds_bytes<WT, T>(K, waves)), st, jobs, N, K,
                       ldy, bpj, waves);
    return hipGetLastError();
}

// Fewer than 128 workgroups of 64 rows leave half the CUs without one: the
// four waves then share 16 rows (one token, 3072 x 15360 Q4_K: 24 -> 12 us; four
// tokens, 3072 x 3072: 13.6 -> 8.4). From 128 on it costs more, as every
// workgroup cuts the activations into digits (four tokens, 9216 x 3072: 13.4
// against 25 us; one token, 18432 x 3072: 9.7 against 11.1 before gemv_waves).
template <uint32_t WT, uint32_t XT, int T, uint32_t CAP>
hipError_t launch_gemv_t(const GemvJobs<CAP>& jobs, uint32_t n_jobs, uint32_t N, uint32_t K, uint32_t ldy,
                         int num_cus, hipStream_t st) {
    if ((N + 63u) / 64u * n_jobs < 128u) return launch_gemv_k<WT, XT, T, CAP, 4>(jobs, n_jobs, N, K, ldy, 4u, st);
    const uint32_t waves = CAP == 1u ? gemv_waves<WT, T>(N, K, num_cus) : 4u;
    return launch_gemv_k<WT, XT, T, CAP, 1>(jobs, n_jobs, N, K, ldy, waves, st);
}

template <uint32_t WT, uint32_t CAP>
hipError_t launch_gemv(uint32_t xtype, const GemvJobs<CAP>& jobs, uint32_t n_jobs, uint32_t N, uint32_t K, uint32_t ldy,
                       uint32_t max_m, int num_cus, hipStream_t st) {
    auto by_x = [&](auto xt) {
        constexpr uint32_t XT = decltype(xt)::value;
        return max_m <= 1   ? launch_gemv_t<WT, XT, 1, CAP>(jobs, n_jobs, N, K, ldy, num_cus, st)
               : max_m <= 2 ? launch_gemv_t<WT, XT, 2, CAP>(jobs, n_jobs, N, K, ldy, num_cus, st)
                            : launch_gemv_t<WT, XT, 4, CAP>(jobs, n_jobs, N, K, ldy, num_cus, st);
    };
    switch (xtype) {
        case kGgmlF32: return by_x(std::integral_constant<uint32_t, kGgmlF32>{});
        case kGgmlF16: return by_x(std::integral_constant<uint32_t, kGgmlF16>{});
        default: return by_x(std::integral_constant<uint32_t, kGgmlBF16>{});
    }
}

template <uint32_t XT>
hipError_t launch_t(const void* w, const void* x, float* y, uint32_t N, uint32_t K, uint32_t M, uint32_t row_offset,
                    hipStream_t st) {
    const dim3 grid((N + 63u) / 64u), block(256);
    const uint8_t* W = (const uint8_t*)w;
    if (M <= 1) hipLaunchKernelGGL((gemv_q4k_kernel<XT, 1>), grid, block, 0, st, W, x, y, N, K, M, row_offset);
    else if (M <= 2) hipLaunchKernelGGL((gemv_q4k_kernel<XT, 2>), grid, block, 0, st, W, x, y, N, K, M, row_offset);
    else hipLaunchKernelGGL((gemv_q4k_kernel<XT, 4>), grid, block, 0, st, W, x, y, N, K, M, row_offset);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemv_q4k_multi(uint32_t xtype, const GemmJob* jobs, uint32_t n_jobs, uint32_t N, uint32_t K,
                                 uint32_t ldy, hipStream_t st) {
    if (n_jobs == 0 || N == 0) return hipSuccess;
    if (n_jobs > kGemvMaxJobs) return hipErrorNotSupported;
    GemvJobs<kGemvMaxJobs> t{};
    uint32_t max_m = 0;
    for (uint32_t q = 0; q < n_jobs; q++) {
        t.w[q] = (const uint8_t*)jobs[q].w;
        t.x[q] = jobs[q].x;
        t.y[q] = jobs[q].y;
        t.m[q] = jobs[q].M;
        t.row_offset[q] = jobs[q].row_offset;
        max_m = max(max_m, jobs[q].M);
    }
    if (max_m == 0) return hipSuccess;
    if (!gemv_fits<kGgmlQ4K>(K, max_m)) return hipErrorNotSupported;
    return launch_gemv<kGgmlQ4K>(xtype, t, n_jobs, N, K, ldy, max_m, 0, st);
}

hipError_t launch_gemv_q4k(const void* w, uint32_t xtype, const void* x, float* y, uint32_t N, uint32_t K,
                           uint32_t M, uint32_t row_offset, int num_cus, hipStream_t st) {
    if (M == 0 || N == 0) return hipSuccess;
    if (M > kGemvMaxTokens) return hipErrorInvalidValue;
    if (gemv_fits<kGgmlQ4K>(K, M)) {
        const GemvJobs<1> one{{(const uint8_t*)w}, {x}, {y}, {M}, {row_offset}};
        return launch_gemv<kGgmlQ4K>(xtype, one, 1u, N, K, N, M, num_cus, st);
    }
    switch (xtype) {
        case kGgmlF32: return launch_t<kGgmlF32>(w, x, y, N, K, M, row_offset, st);
        case kGgmlF16: return launch_t<kGgmlF16>(w, x, y, N, K, M, row_offset, st);
        default: return launch_t<kGgmlBF16>(w, x, y, N, K, M, row_offset, st);
    }
}

bool gemv_q8_fits(uint32_t K, uint32_t M) { return gemv_fits<kGgmlQ8_0>(K, M); }

hipError_t launch_gemv_q8(const void* w, uint32_t xtype, const void* x, float* y, uint32_t N, uint32_t K, uint32_t M,
                          uint32_t row_offset, int num_cus, hipStream_t st) {
    if (M == 0 || N == 0) return hipSuccess;
    if (!gemv_fits<kGgmlQ8_0>(K, M)) return hipErrorInvalidValue;
    const GemvJobs<1> one{{(const uint8_t*)w}, {x}, {y}, {M}, {row_offset}};
    return launch_gemv<kGgmlQ8_0>(xtype, one, 1u, N, K, N, M, num_cus, st);
}

}  // namespace llmr
