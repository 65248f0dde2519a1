// lora.hip - LoRA adapters on the DiT linears, in the reference's two forms:
//
//  * the runtime two-hop correction appended to a base batch_matmul output
//    (dispatch_lora_correction, dit.c3:1319-1364): hop 1 scratch = x . A^T
//    (batch_matmul_simple, llm.slang:1146-1180), hop 2 output += scale *
//    scratch . B^T (batch_matmul_add_scaled, llm.slang:1262-1294);
//  * the load-time merge into a Q8_0 weight with per-block requantization
//    (q8_lora_merge, llm.slang:1337-1420; host merge_one_site,
//    lora_merge.c3:36-73).
//
// The dot products are fused multiply-adds (the reference's `partial += a *
// b` leaves contraction to its shader compiler), every other f32 operation
// rounds where the reference's source writes it, and every sum is formed in
// the reference's order, so the results are bit-identical to the CPU
// restatement: hop 1's sums as a 256-thread workgroup forms them (strided
// partials, then the tree), hop 2's and the merge's in rank order.
//
// Work layout (MI355X): hop 1 gives each wave 4 tokens x 8 ranks (A is read
// once per 4 tokens instead of once per (token, rank) sum) with the tree across
// its lanes; hop 2 gives each workgroup 256 output features x 16 or 32 tokens.
// Hop 2's read-modify-write of the f32 output is the dominant traffic.
#include <hip/hip_runtime.h>

#include "llmr_device.h"
#include "llmr_internal.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace llmr {
namespace {

constexpr uint32_t kDownTokens = 4;   // tokens per hop-1 workgroup
constexpr uint32_t kDownRanks = 8;    // rank outputs per hop-1 pass
constexpr uint32_t kDownTree = 32;    // sums per LDS tree round
constexpr uint32_t kUpTokens = 32;    // tokens per hop-2 workgroup
constexpr uint32_t kUpChunk = 32;     // ranks per hop-2 LDS pass

template <uint32_t XT>
__device__ __forceinline__ float load_act(const void* X, uint64_t i) {
    if constexpr (XT == kGgmlF32) {
        return ((const float*)X)[i];
    } else if constexpr (XT == kGgmlBF16) {
        return __uint_as_float((uint32_t)((const uint16_t*)X)[i] << 16);
    } else {
        return (float)__builtin_bit_cast(_Float16, ((const uint16_t*)X)[i]);
    }
}

// scratch[s, r] = sum_k A[r, k] * X[s, k]: thread gi accumulates k = gi,
// gi + 256, ... in order, then the tree s = 128 .. 1 of batch_matmul_simple.
template <uint32_t XT>
__global__ void __launch_bounds__(256) lora_down_kernel(const float* __restrict__ A, const void* __restrict__ X,
                                                         float* __restrict__ scratch, uint32_t rank, uint32_t in_dim,
                                                         uint32_t seq_len) {
    constexpr uint32_t Q = kDownTokens * kDownRanks;  // sums per pass, reduced kDownTree at a time
    __shared__ float red[kDownTree][256];
    const uint32_t gi = threadIdx.x;
    const uint32_t s0 = blockIdx.x * kDownTokens;
    for (uint32_t r0 = 0; r0 < rank; r0 += kDownRanks) {
        float part[kDownTokens][kDownRanks];
#pragma unroll
        for (uint32_t t = 0; t < kDownTokens; t++)
#pragma unroll
            for (uint32_t r = 0; r < kDownRanks; r++) part[t][r] = 0.0f;
#pragma unroll 4
        for (uint32_t k = gi; k < in_dim; k += 256u) {
            float x[kDownTokens];
#pragma unroll
            for (uint32_t t = 0; t < kDownTokens; t++)
                x[t] = s0 + t < seq_len ? load_act<XT>(X, (uint64_t)(s0 + t) * in_dim + k) : 0.0f;
#pragma unroll
            for (uint32_t r = 0; r < kDownRanks; r++) {
                const float a = r0 + r < rank ? A[(uint64_t)(r0 + r) * in_dim + k] : 0.0f;
#pragma unroll
                for (uint32_t t = 0; t < kDownTokens; t++) part[t][r] = __builtin_fmaf(a, x[t], part[t][r]);
            }
        }
#pragma unroll
        for (uint32_t h = 0; h < Q / kDownTree; h++) {
#pragma unroll
            for (uint32_t q = 0; q < kDownTree; q++)
                red[q][gi] = part[(h * kDownTree + q) / kDownRanks][(h * kDownTree + q) % kDownRanks];
            __syncthreads();
#pragma unroll
            for (uint32_t ls = 7; ls < 8; ls--) {  // s = 2^ls = 128, 64, ..., 1
                const uint32_t s = 1u << ls;
                for (uint32_t item = gi; item < kDownTree * s; item += 256u) {
                    const uint32_t q = item >> ls, i = item & (s - 1u);
                    red[q][i] += red[q][i + s];
                }
                __syncthreads();
            }
            if (gi < kDownTree) {
                const uint32_t qq = h * kDownTree + gi, t = qq / kDownRanks, r = qq % kDownRanks;
                if (s0 + t < seq_len && r0 + r < rank) scratch[(uint64_t)(s0 + t) * rank + r0 + r] = red[gi][0];
            }
            __syncthreads();  // red is rewritten by the next half
        }
    }
}

// The same sums, a wave per 4 tokens x 8 ranks with no LDS: lane l carries the
// partial sums gi = 4 l .. 4 l + 3 (16-byte loads of A and x), and the tree
// s = 128 .. 4 runs across lanes l + 32, 16, .., 1, s = 2 and 1 in the lane. Each
// cross-lane level adds two sums at once (the lanes with the level's bit clear
// keep one, the others the other), so 32 sums cost 128 exchanges instead of
// 768. What bounds it is A from L2 (rank x in_dim floats per 4 tokens); through
// LDS with a barrier per tree level it was 55 us for 1536 x 3072 x 32, this is
// 16. Needs 16-byte aligned A and x, in_dim % 4 == 0.
constexpr uint32_t kWaveTokens = 4, kWaveRanks = 8;
__device__ __forceinline__ float tree_pair(float a, float b, uint32_t lane, uint32_t bit) {
    // lanes with `bit` clear: a[l] + a[l ^ bit]; set: b[l] + b[l ^ bit]
    const bool up = (lane & bit) != 0u;
    return (up ? b : a) + __shfl_xor(up ? a : b, (int)bit, 64);
}
template <uint32_t XT>
__global__ void __launch_bounds__(256, 2) lora_down_wave_kernel(const float* __restrict__ A, const void* __restrict__ X,
                                                                 float* __restrict__ scratch, uint32_t rank,
                                                                 uint32_t in_dim, uint32_t seq_len, uint32_t rank_groups) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t id = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r0 = id % rank_groups * kWaveRanks, s0 = id / rank_groups * kWaveTokens;
    if (s0 >= seq_len) return;
    f32x4 acc[kWaveTokens][kWaveRanks];
#pragma unroll
    for (uint32_t t = 0; t < kWaveTokens; t++)
#pragma unroll
        for (uint32_t r = 0; r < kWaveRanks; r++) acc[t][r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // rows past seq_len or rank read the last row and are not stored
    struct In {
        f32x4 x[kWaveTokens], a[kWaveRanks];
    };
    auto load = [&](uint32_t k) __attribute__((always_inline)) {
        In v;
#pragma unroll
        for (uint32_t t = 0; t < kWaveTokens; t++) {
            const uint64_t e = (uint64_t)min(s0 + t, seq_len - 1u) * in_dim + k;
            if constexpr (XT == kGgmlF32) {
                v.x[t] = *(const f32x4*)((const float*)X + e);
            } else {
                const u32x2 w = *(const u32x2*)((const uint16_t*)X + e);
                const uint32_t lo = w.x, hi = w.y;
                if constexpr (XT == kGgmlBF16) {
                    v.x[t] = f32x4{__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u),
                                   __uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u)};
                } else {
                    const f16x2 p = __builtin_bit_cast(f16x2, lo), q = __builtin_bit_cast(f16x2, hi);
                    v.x[t] = f32x4{(float)p.x, (float)p.y, (float)q.x, (float)q.y};
                }
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < kWaveRanks; r++)
            v.a[r] = *(const f32x4*)(A + (uint64_t)min(r0 + r, rank - 1u) * in_dim + k);
        return v;
    };
    const uint32_t k0 = 4u * lane;
    if (k0 < in_dim) {
        In cur = load(k0);
        for (uint32_t k = k0; k < in_dim; k += 256u) {
            In nxt;
            const bool more = k + 256u < in_dim;
            if (more) nxt = load(k + 256u);
#pragma unroll
            for (uint32_t t = 0; t < kWaveTokens; t++)
#pragma unroll
                for (uint32_t r = 0; r < kWaveRanks; r++)
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        acc[t][r][c] = __builtin_fmaf(cur.a[r][c], cur.x[t][c], acc[t][r][c]);
            if (more) cur = nxt;
        }
    }
    // sum q = 8 t + r; after the five pairing levels lane l holds sum 16 b5 +
    // 8 b4 + 4 b3 + 2 b2 + b1 of its bits, after the sixth both lanes of a pair
    f32x4 v16[16], v8[8], v4[4], v2[2], v1;
#pragma unroll
    for (int q = 0; q < 16; q++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[q / 8][q % 8][c]),
                                                            __float_as_uint(acc[2 + q / 8][q % 8][c]), false, false);
            v16[q][c] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
        }
#pragma unroll
    for (int q = 0; q < 8; q++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v16[q][c]), __float_as_uint(v16[8 + q][c]),
                                                            false, false);
            v8[q][c] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
        }
#pragma unroll
    for (int c = 0; c < 4; c++) {
#pragma unroll
        for (int q = 0; q < 4; q++) v4[q][c] = tree_pair(v8[q][c], v8[4 + q][c], lane, 8u);
#pragma unroll
        for (int q = 0; q < 2; q++) v2[q][c] = tree_pair(v4[q][c], v4[2 + q][c], lane, 4u);
        v1[c] = tree_pair(v2[0][c], v2[1][c], lane, 2u);
        v1[c] += __shfl_xor(v1[c], 1, 64);
    }
    const float sum = (v1.x + v1.z) + (v1.y + v1.w);
    const uint32_t q = (lane >> 5 & 1u) * 16u + (lane >> 4 & 1u) * 8u + (lane >> 3 & 1u) * 4u + (lane >> 2 & 1u) * 2u +
                       (lane >> 1 & 1u);
    const uint32_t t = s0 + q / kWaveRanks, r = r0 + q % kWaveRanks;
    if ((lane & 1u) == 0u && t < seq_len && r < rank) scratch[(uint64_t)t * rank + r] = sum;
}

// out[s * out_dim + row_offset + o] += scale * sum_r B[(wro + o) * rank + r] *
// scratch[s * rank + r] for o < b_rows, the sum in rank order. A workgroup
// takes 512 outputs (thread gi: o0 + gi and o0 + 256 + gi) x kUpTokens
// tokens; B's rows for its outputs pass through LDS in chunks of kUpChunk
// ranks (read coalesced, stored transposed with a pad so thread gi reads its
// columns without bank conflicts) and stay in registers while the tokens'
// scratch rows are read as 16-byte broadcasts.
__global__ void __launch_bounds__(256) lora_up_kernel(const float* __restrict__ B, const float* __restrict__ scratch,
                                                       float* __restrict__ out, uint32_t rank, uint32_t out_dim,
                                                       uint32_t seq_len, float scale, uint32_t row_offset,
                                                       uint32_t weight_row_offset, uint32_t b_rows) {
    __shared__ __attribute__((aligned(16))) float sc[kUpTokens][kUpChunk];
    __shared__ float bs[kUpChunk][513];
    const uint32_t gi = threadIdx.x;
    const uint32_t o0 = blockIdx.x * 512u, s0 = blockIdx.y * kUpTokens;
    const uint32_t nt = min(kUpTokens, seq_len - s0), no = min(512u, b_rows - o0);
    float acc[2][kUpTokens];
#pragma unroll
    for (uint32_t h = 0; h < 2; h++)
#pragma unroll
        for (uint32_t t = 0; t < kUpTokens; t++) acc[h][t] = 0.0f;
    for (uint32_t r0 = 0; r0 < rank; r0 += kUpChunk) {
        const uint32_t nr = min(kUpChunk, rank - r0);
        if (nr == kUpChunk && rank % 4u == 0u) {
            // whole chunks: 16-byte loads (B rows and scratch rows are 16-byte
            // aligned: rank % 4 == 0), indices by shifts
            for (uint32_t i = gi; i < no * (kUpChunk / 4u); i += 256u) {
                const uint32_t o = i >> 3, r = (i & 7u) * 4u;
                const f32x4 v = *(const f32x4*)(B + (uint64_t)(weight_row_offset + o0 + o) * rank + r0 + r);
                bs[r][o] = v.x;
                bs[r + 1][o] = v.y;
                bs[r + 2][o] = v.z;
                bs[r + 3][o] = v.w;
            }
            for (uint32_t i = gi; i < nt * (kUpChunk / 4u); i += 256u) {
                const uint32_t t = i >> 3, r = (i & 7u) * 4u;
                *(f32x4*)&sc[t][r] = *(const f32x4*)(scratch + (uint64_t)(s0 + t) * rank + r0 + r);
            }
        } else {
            for (uint32_t i = gi; i < no * nr; i += 256u) {
                const uint32_t o = i / nr, r = i % nr;
                bs[r][o] = B[(uint64_t)(weight_row_offset + o0 + o) * rank + r0 + r];
            }
            for (uint32_t i = gi; i < nt * nr; i += 256u) {
                const uint32_t t = i / nr, r = i % nr;
                sc[t][r] = scratch[(uint64_t)(s0 + t) * rank + r0 + r];
            }
        }
        __syncthreads();
        if (nr == kUpChunk) {
            float bv[2][kUpChunk];
#pragma unroll
            for (uint32_t h = 0; h < 2; h++)
#pragma unroll
                for (uint32_t r = 0; r < kUpChunk; r++) bv[h][r] = bs[r][h * 256u + gi];
#pragma unroll
            for (uint32_t t = 0; t < kUpTokens; t++) {
                float a0 = acc[0][t], a1 = acc[1][t];
#pragma unroll
                for (uint32_t r = 0; r < kUpChunk; r++) {
                    const float sv = sc[t][r];
                    a0 = __builtin_fmaf(bv[0][r], sv, a0);
                    a1 = __builtin_fmaf(bv[1][r], sv, a1);
                }
                acc[0][t] = a0;
                acc[1][t] = a1;
            }
        } else {  // the last, partial chunk of ranks
            for (uint32_t r = 0; r < nr; r++) {
                const float b0 = bs[r][gi], b1 = bs[r][256u + gi];
#pragma unroll
                for (uint32_t t = 0; t < kUpTokens; t++) {
                    acc[0][t] = __builtin_fmaf(b0, sc[t][r], acc[0][t]);
                    acc[1][t] = __builtin_fmaf(b1, sc[t][r], acc[1][t]);
                }
            }
        }
        __syncthreads();  // bs and sc are refilled by the next chunk
    }
    // (columns past b_rows and tokens past seq_len are neither read nor
    // written; their acc entries hold LDS leftovers). All of the thread's
    // output reads are issued before any write, so their latencies overlap
    // instead of one read-modify-write waiting per token.
    float* const ybase = out + (uint64_t)s0 * out_dim + row_offset + o0 + gi;
    float yv[2][kUpTokens];
#pragma unroll
    for (uint32_t h = 0; h < 2; h++)
#pragma unroll
        for (uint32_t t = 0; t < kUpTokens; t++)
            yv[h][t] = (h * 256u + gi < no && t < nt) ? ybase[(uint64_t)t * out_dim + h * 256u] : 0.0f;
#pragma unroll
    for (uint32_t h = 0; h < 2; h++)
#pragma unroll
        for (uint32_t t = 0; t < kUpTokens; t++)
            if (h * 256u + gi < no && t < nt) ybase[(uint64_t)t * out_dim + h * 256u] = yv[h][t] + scale * acc[h][t];
}

// Hop 2 for ranks 4, 8, .. 32 (R) and multiples of 32 (R = 32, chunks of it):
// thread gi owns output column o0 + gi, whose B row stays in registers (a chunk
// at a time) for the workgroup's T tokens; their scratch rows are the same for
// the whole wave, so they come as scalar loads and are scalar operands of the
// FMAs, and all the output values are requested before the first sum. The buffer
// ends at seq_len: rows past it read zero and are not stored. Their offset is the
// lane's, which the range check covers on its own (whether it covers a scalar
// offset past the buffer's end is not documented). Same arithmetic
// as lora_up_kernel: the sum over ranks in rank order from 0, then y + scale *
// sum. What bounds it is the output's read and write. With the scratch rows
// through LDS (a broadcast read per 4 FMAs is as slow as they are), 16 tokens at
// a time and 128 a workgroup, 1536 x 9216 x 32 took 59 us (1.9 TB/s), 4608 x
// 21504 x 32 240 us; this takes 32 and 190 (4.2 TB/s). B through LDS instead of
// each lane reading its own row: 15 us slower. Both hops of 1536 x 9216 x 3072:
// 110 -> 49 us at rank 32, 191 -> 78 at rank 64.
template <uint32_t R, uint32_t T, bool CHUNKS>
__global__ void __launch_bounds__(256) lora_up_reg_kernel(const float* __restrict__ B,
                                                           const float* __restrict__ scratch, float* __restrict__ out,
                                                           uint32_t rank, uint32_t out_dim, uint32_t seq_len,
                                                           float scale, uint32_t row_offset, uint32_t weight_row_offset,
                                                           uint32_t b_rows) {
    typedef __attribute__((address_space(4))) const float cfloat;
    const uint32_t o = blockIdx.x * 256u + threadIdx.x;
    const uint32_t group = blockIdx.z * gridDim.y + blockIdx.y;  // of T tokens
    if (group >= (seq_len + T - 1u) / T) return;
    const uint32_t s0 = group * T, nt = min(T, seq_len - s0);
    const rsrc_t yr = make_rsrc(out + (uint64_t)s0 * out_dim, (uint64_t)nt * out_dim * 4u);
    const uint32_t yo = o < b_rows ? (row_offset + o) * 4u : 0x80000000u;
    float yv[T];
#pragma unroll
    for (uint32_t t = 0; t < T; t++)
        yv[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(yr, yo + t * out_dim * 4u, 0, 0));
    const uint32_t ld = CHUNKS ? rank : R;
    const float* const brow = B + (uint64_t)(weight_row_offset + min(o, b_rows - 1u)) * ld;
    float bv[R];
    auto load_b = [&](uint32_t c) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t r = 0; r < R; r += 4) {
            const f32x4 v = *(const f32x4*)(brow + c * R + r);
            bv[r] = v.x;
            bv[r + 1] = v.y;
            bv[r + 2] = v.z;
            bv[r + 3] = v.w;
        }
    };
    auto sum = [&](uint32_t t, uint32_t c, float a) __attribute__((always_inline)) {
        cfloat* const sc = (cfloat*)(scratch + (uint64_t)min(s0 + t, seq_len - 1u) * ld + c * R);
#pragma unroll
        for (uint32_t r = 0; r < R; r++) a = __builtin_fmaf(bv[r], sc[r], a);
        return a;
    };
    auto store = [&](uint32_t t, float a) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(yv[t] + scale * a), yr, yo + t * out_dim * 4u, 0, 0);
    };
    if constexpr (!CHUNKS) {
        load_b(0);
#pragma unroll
        for (uint32_t t = 0; t < T; t++) store(t, sum(t, 0, 0.0f));
    } else {
        float a[T];
#pragma unroll
        for (uint32_t t = 0; t < T; t++) a[t] = 0.0f;
        for (uint32_t c = 0; c < rank / R; c++) {
            load_b(c);
#pragma unroll
            for (uint32_t t = 0; t < T; t++) a[t] = sum(t, c, a[t]);
        }
#pragma unroll
        for (uint32_t t = 0; t < T; t++) store(t, a[t]);
    }
}

// One 256-element chunk (8 Q8_0 blocks = 272 bytes) of LoRA row blockIdx.y:
// thread gi owns element k = 256 blockIdx.x + gi.
__global__ void __launch_bounds__(256) q8_lora_merge_kernel(uint8_t* __restrict__ base, const float* __restrict__ A,
                                                             const float* __restrict__ B, uint32_t in_dim,
                                                             uint32_t dst_row_offset, uint32_t rank, float scale) {
    __shared__ float brow[kMaxLoraRank];
    __shared__ float amax[256];
    const uint32_t gi = threadIdx.x, j = blockIdx.y;
    const uint32_t blk = gi / 32u, e = gi % 32u;
    const uint32_t k = blockIdx.x * 256u + gi;
    for (uint32_t r = gi; r < rank; r += 256u) brow[r] = B[(uint64_t)j * rank + r];
    uint8_t* const b = base + (uint64_t)(dst_row_offset + j) * (in_dim / 32u) * 34u +
                       (uint64_t)(blockIdx.x * 8u + blk) * 34u;
    const float d = f16_bits_to_f32((uint32_t)b[0] | ((uint32_t)b[1] << 8));
    const float base_val = d * (float)(int8_t)b[2 + e];
    __syncthreads();
    float delta = 0.0f;
    for (uint32_t r = 0; r < rank; r++) delta = __builtin_fmaf(brow[r], A[(uint64_t)r * in_dim + k], delta);
    delta *= scale;
    const float u = base_val + delta;
    amax[gi] = fabsf(u);
    __syncthreads();
    for (uint32_t s = 16; s > 0; s >>= 1) {
        if (e < s) amax[gi] = fmaxf(amax[gi], amax[gi + s]);
        __syncthreads();
    }
    float dn = amax[blk * 32u] / 127.0f;
    if (dn < 1e-8f) dn = 1e-8f;
    const float qf = u / dn;
    int q = qf >= 0.0f ? (int)(qf + 0.5f) : (int)(qf - 0.5f);
    q = q < -127 ? -127 : (q > 127 ? 127 : q);
    b[2 + e] = (uint8_t)(int8_t)q;  // every read of this chunk precedes the barriers above
    if (e == 0) {
        const uint16_t h = __builtin_bit_cast(uint16_t, (_Float16)dn);
        b[0] = (uint8_t)(h & 0xffu);
        b[1] = (uint8_t)(h >> 8);
    }
}

}  // namespace

hipError_t launch_lora_correction(const float* A, const float* B, uint32_t rank, float scale, float* scratch,
                                  const void* x, uint32_t xtype, float* out, uint32_t in_dim, uint32_t out_dim,
                                  uint32_t seq_len, uint32_t b_rows, uint32_t row_offset, uint32_t weight_row_offset,
                                  hipStream_t st) {
    if (rank == 0 || seq_len == 0) return hipSuccess;
    // One wave walks a whole row for 8 ranks, so with one such group of ranks (two,
    // with long rows and many tokens) a workgroup of the LDS form is the faster one
    // where the walk is long and waves are few: both hops at rank 8, LDS : wave, 1 x
    // 3072 22 : 32 us at K = 15360, 2048 x 1024 1.0 : 1.2 at 3072, 4608 x 1024 1.0 :
    // 0.95, 1.0 : 1.0 or less at K = 1024; rank 16, 4608 tokens 1.0 : 1.14 at 15360,
    // 1.0 : 0.89 at 8192; rank 12, one token 1.0 : 0.89 at 3072.
    const bool few_waves = rank <= 8u    ? in_dim >= 2048u && (in_dim > 4096u || seq_len < 4096u)
                           : rank <= 16u ? in_dim > 12288u && seq_len >= 4096u
                                         : false;
    const bool wide = !few_waves && in_dim % 4u == 0u && ((uintptr_t)A & 15u) == 0u && ((uintptr_t)x & 15u) == 0u;
    auto down = [&](auto xt) {
        constexpr uint32_t XT = decltype(xt)::value;
        if (wide) {
            const uint32_t rg = (rank + kWaveRanks - 1u) / kWaveRanks;
            const uint64_t waves = (uint64_t)rg * ((seq_len + kWaveTokens - 1u) / kWaveTokens);
            hipLaunchKernelGGL(lora_down_wave_kernel<XT>, dim3((uint32_t)((waves + 3u) / 4u)), dim3(256), 0, st, A, x,
                               scratch, rank, in_dim, seq_len, rg);
        } else {
            hipLaunchKernelGGL(lora_down_kernel<XT>, dim3((seq_len + kDownTokens - 1) / kDownTokens), dim3(256), 0, st,
                               A, x, scratch, rank, in_dim, seq_len);
        }
    };
    switch (xtype) {
        case kGgmlF32: down(std::integral_constant<uint32_t, kGgmlF32>{}); break;
        case kGgmlF16: down(std::integral_constant<uint32_t, kGgmlF16>{}); break;
        default: down(std::integral_constant<uint32_t, kGgmlBF16>{}); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || b_rows == 0) return e;
    // (32 rows of the output within a buffer's 31-bit offsets)
    if (rank % 4u == 0u && (rank <= 32u || rank % 32u == 0u) && (uint64_t)out_dim * 32u * 4u < (1ull << 31)) {
        // 32 tokens a workgroup (B read half as often) where that still gives
        // every CU 16 workgroups: 4608 x 21504 x 32 both hops 235 against 257 us
        // with 16, 1536 x 9216 x 32 52 against 49, 300 x 3072 x 16 23 against 17
        const uint32_t cols = (b_rows + 255u) / 256u;
        const bool wide_t = (uint64_t)cols * ((seq_len + 31u) / 32u) >= 4096u;
        // (a grid's y ends at 65535 workgroups: 1048560 tokens of 16)
        auto grid = [&](uint32_t t) {
            const uint32_t groups = (seq_len - 1u) / t + 1u, y = min(groups, 65535u);
            return dim3(cols, y, (groups + y - 1u) / y);
        };
        auto go = [&](auto r) {
            constexpr uint32_t R = decltype(r)::value;
            if (rank > R)
                hipLaunchKernelGGL((lora_up_reg_kernel<R, 16, true>), grid(16u), dim3(256), 0,
                                   st, B, (const float*)scratch, out, rank, out_dim, seq_len, scale, row_offset,
                                   weight_row_offset, b_rows);
            else if (wide_t)
                hipLaunchKernelGGL((lora_up_reg_kernel<R, 32, false>), grid(32u), dim3(256), 0, st, B,
                                   (const float*)scratch, out, rank, out_dim, seq_len, scale, row_offset,
                                   weight_row_offset, b_rows);
            else
                hipLaunchKernelGGL((lora_up_reg_kernel<R, 16, false>), grid(16u), dim3(256), 0, st, B,
                                   (const float*)scratch, out, rank, out_dim, seq_len, scale, row_offset,
                                   weight_row_offset, b_rows);
        };
        switch (rank) {
            case 4: go(std::integral_constant<uint32_t, 4>{}); break;
            case 8: go(std::integral_constant<uint32_t, 8>{}); break;
            case 12: go(std::integral_constant<uint32_t, 12>{}); break;
            case 16: go(std::integral_constant<uint32_t, 16>{}); break;
            case 20: go(std::integral_constant<uint32_t, 20>{}); break;
            case 24: go(std::integral_constant<uint32_t, 24>{}); break;
            case 28: go(std::integral_constant<uint32_t, 28>{}); break;
            default: go(std::integral_constant<uint32_t, 32>{}); break;
        }
        return hipGetLastError();
    }
    const dim3 gu((b_rows + 511u) / 512u, (seq_len + kUpTokens - 1) / kUpTokens);
    hipLaunchKernelGGL(lora_up_kernel, gu, dim3(256), 0, st, B, (const float*)scratch, out, rank, out_dim, seq_len,
                       scale, row_offset, weight_row_offset, b_rows);
    return hipGetLastError();
}

hipError_t launch_q8_lora_merge(void* base, const float* A, const float* B, uint32_t in_dim, uint32_t b_rows,
                                uint32_t dst_row_offset, uint32_t rank, float scale, hipStream_t st) {
    if (b_rows == 0) return hipSuccess;
    hipLaunchKernelGGL(q8_lora_merge_kernel, dim3(in_dim / 256u, b_rows), dim3(256), 0, st, (uint8_t*)base, A, B,
                       in_dim, dst_row_offset, rank, scale);
    return hipGetLastError();
}

}  // namespace llmr
