// Fused attention for the bf16 transformer stage: P = softmax(Q K^T / sqrt(d)), ctx = P V, and its
// backward pass, without ever writing the [batch, heads, seq, seq] score / probability tensors:
// the forward keeps one number per query (log2 of the softmax denominator, shifted), the backward
// recomputes P from it.  Three kernels: forward, backward query side (dQ), backward key side
// (dK, dV).
//
// The reference's checked-out branch has no transformer stage (PipeDream-2BW lives on another
// branch, README.md:7-8); the kernels do for such a stage's attention what cuBLAS + ATen do for the
// torch.nn layers of the reference's stages (runtime/runtime.py:529-530 forward, :606-608 backward).
//
// Bound: MFMA bf16 / vector ALU (seq * seq exponentials per head); algorithmic HBM traffic = qkv
// (and ctx, dctx in the backward) read once per kernel, ctx / dqkv written once.
//
// Forward at seq 128 and 256 (all else: "any sequence length" below): one block = one (batch, head)
// pair x 128 queries, 8 waves of 16, K and V of the head staged in LDS once
// per block with a row pitch of 72 bf16, which serves both the 128-bit fragment reads (8 consecutive
// k per lane) and the transposing reads.  Everything is computed in the orientation in which no accumulator ever has to change layout; shown for the
// forward (v_mfma_f32_16x16x32_bf16: lane l holds A row / B column l % 16, k-slots 8 (l / 16) + 0..7,
// and accumulator column l % 16, rows 4 (l / 16) + 0..3):
//   S^T = K Q^T   A = K rows from LDS (k = head dimension), B = this wave's Q rows straight from
//                 global memory; the accumulator of key tile t holds, in lane l, query l % 16 and
//                 keys 16 t + 4 (l / 16) + e, e = 0..3
//   softmax       over the keys of a query = over a lane's registers and the lanes l ^ 16, l ^ 32,
//                 l ^ 48: two shuffles per reduction
//   O^T = V^T P^T the B operand (8 keys per lane) is exactly the packed accumulators of key tiles 2u
//                 and 2u+1, so P goes from the softmax into the second product without touching
//                 LDS; a sum over keys does not care in which order the MFMA visits them, and the A
//                 operand (V^T) is fetched with the transposing LDS read ds_read_b64_tr_b16 at the
//                 matching keys.
// The backward kernels use the same two moves: "first product lands in the layout of the second
// product's B operand" and "transposed A operand through ds_read_b64_tr_b16".
#include <cfloat>

#include "pd_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef short short8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int AT_D = 64;               // head dimension
constexpr int AT_THREADS = 512;        // 8 waves x 16 queries (keys)
constexpr int AT_QB = 128;             // queries (keys) per block
constexpr int AT_P = AT_D + 8;         // LDS row pitch (bf16)
constexpr float AT_LOG2E = 1.44269504088896340736f;

__device__ __forceinline__ uint16_t at_f2bf(float f) { return pd_f2bf(f); }
__device__ __forceinline__ float at_bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// rows [0, S) x 64 columns of a [.][ld] bf16 matrix -> LDS with pitch AT_P
template <int S>
__device__ __forceinline__ void at_stage(uint16_t* lds, const uint16_t* __restrict__ g, int ld, int tid) {
    constexpr int ITERS = S * (AT_D / 8) / AT_THREADS;
    static_assert(S * (AT_D / 8) % AT_THREADS == 0, "rows divide over the block");
    u16x8 r[ITERS];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {         // all loads in flight before the first LDS store
        const int id = tid + it * AT_THREADS;
        r[it] = *(const u16x8*)(g + (size_t)(id / (AT_D / 8)) * ld + (id % (AT_D / 8)) * 8);
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        const int id = tid + it * AT_THREADS;
        *(u16x8*)(lds + (id / (AT_D / 8)) * AT_P + (id % (AT_D / 8)) * 8) = r[it];
    }
}

// MFMA operand with 8 consecutive head-dimension values: row `row` of an LDS matrix, k-step s
__device__ __forceinline__ bf16x8 at_frag(const uint16_t* lds, int row, int s, int g) {
    return __builtin_bit_cast(bf16x8, *(const u16x8*)(lds + row * AT_P + 32 * s + 8 * g));
}

// Transposed MFMA A operand for the product over rows (keys or queries) 32u .. 32u+31 of an LDS matrix
// [row][64]: lane (li, g) receives column 16 dt + li at rows 32u + 4g + (0..3) (slots 0-3) and the
// same + 16 (slots 4-7), matching two packed 16-row accumulator tiles.  Inside a 16-lane group, input
// lane i addresses [row0 + i/4][col0 + 4 (i % 4)] and output lane j receives column col0 + j at rows
// row0 .. row0 + 3.
__device__ __forceinline__ bf16x8 at_frag_t(const uint16_t* lds, int u, int dt, int li, int g) {
    typedef __attribute__((address_space(3))) short4_t* lds_ptr;
    const uint16_t* p = lds + (32 * u + 4 * g + li / 4) * AT_P + 16 * dt + 4 * (li % 4);
    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p);
    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 16 * AT_P));
    const short8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ void at_store4(uint16_t* p, const float4_t& v) {
    *(u16x4*)p = u16x4{at_f2bf(v[0]), at_f2bf(v[1]), at_f2bf(v[2]), at_f2bf(v[3])};
}

// ---- forward ---------------------------------------------------------------------------------------
// lse2[bh][q] = m * c + log2(sum_k 2^((s_k - m) c)), c = log2(e) / sqrt(d): P[q][k] = 2^(s_k c - lse2[q]).
template <int S, bool WRITE_P>
__global__ __launch_bounds__(AT_THREADS) void attention_fwd_kernel(const uint16_t* __restrict__ qkv,
                                                                  uint16_t* __restrict__ ctx,
                                                                  uint16_t* __restrict__ probs,
                                                                  float* __restrict__ lse2, int heads, float c) {
    constexpr int NT = S / 16;          // key tiles of 16
    __shared__ __attribute__((aligned(16))) uint16_t k_lds[S * AT_P];
    __shared__ __attribute__((aligned(16))) uint16_t v_lds[S * AT_P];

    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int li = lane % 16, g = lane / 16;
    const int bh = blockIdx.y, b = bh / heads, h = bh % heads;
    const int H = heads * AT_D, ld = 3 * H;
    const uint16_t* base = qkv + (size_t)b * S * ld + h * AT_D;     // Q of this head; K at +H, V at +2H
    at_stage<S>(k_lds, base + H, ld, tid);
    at_stage<S>(v_lds, base + 2 * H, ld, tid);

    const int q = blockIdx.x * AT_QB + wave * 16 + li;              // this lane's query (always < S)
    bf16x8 qf[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
        qf[s] = __builtin_bit_cast(bf16x8, *(const u16x8*)(base + (size_t)q * ld + 32 * s + 8 * g));
    __syncthreads();

    float4_t sc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at_frag(k_lds, 16 * t + li, s, g), qf[s], acc, 0, 0, 0);
        sc[t] = acc;
    }

    float m = -INFINITY;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, sc[t][e]);
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sc[t][e] = __builtin_amdgcn_exp2f((sc[t][e] - m) * c);      // hardware exp2
            sum += sc[t][e];
        }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float inv = 1.0f / sum;
    if (lse2 && g == 0) lse2[(size_t)bh * S + q] = m * c + __builtin_amdgcn_logf(sum);   // v_log_f32 is log2

    uint16_t* prow = WRITE_P ? probs + ((size_t)bh * S + q) * S + 4 * g : nullptr;
    float4_t oacc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) oacc[dt] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NT / 2; ++u) {
        u16x8 p;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p[e] = at_f2bf(sc[2 * u][e] * inv);
            p[4 + e] = at_f2bf(sc[2 * u + 1][e] * inv);
        }
        if (WRITE_P) {
            *(u16x4*)(prow + 32 * u) = u16x4{p[0], p[1], p[2], p[3]};
            *(u16x4*)(prow + 32 * u + 16) = u16x4{p[4], p[5], p[6], p[7]};
        }
        const bf16x8 pf = __builtin_bit_cast(bf16x8, p);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
            oacc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at_frag_t(v_lds, u, dt, li, g), pf, oacc[dt], 0, 0, 0);
    }

    uint16_t* crow = ctx + ((size_t)b * S + q) * H + h * AT_D + 4 * g;      // ctx[b*S + q][h*64 + 16 dt + 4 g + e]
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) at_store4(crow + 16 * dt, oacc[dt]);
}

// ---- any sequence length: forward, backward -----------------------------------------------------------------
// The other side's rows pass through LDS in chunks of AT_CH (the next chunk is on its way to the registers while one is
// used), so seq is a run-time number: a multiple of 8, rows past it are zeros in LDS and masked.  A wave has QT times 16
// queries (keys).
// Forward: a running maximum and sum per query; what is there is rescaled when the maximum rises.  It starts at the lowest
// finite number, so that keys whose scores are all -inf count as zeros until another one comes (and a query that has no
// other keys ends as 0 / 0, as in a softmax).
// Backward, query side: P^T = 2^(K Q^T c - lse2), dP^T = V dO^T, dS^T = P^T o (dP^T - delta) / sqrt(d) with
// delta_q = sum_d dO[q][d] O[q][d] (= sum_k dP[q][k] P[q][k]), dQ^T = K^T dS^T; delta is also written out for the key side.
// Backward, key side: S = Q K^T and dP = dO V^T have the queries on the MFMA rows (A operands = Q and dO rows from LDS, B =
// this wave's K and V rows from global memory), so lane l holds key l % 16 and queries 16 t + 4 (l / 16) + e: P and dS land
// packed as B operands of the sums over queries dV^T = dO^T P and dK^T = Q^T dS, whose A operands are transposing reads.
//
// Bound: fragment reads from LDS, a kilobyte per MFMA of 16 cycles with QT = 1 (256 bytes a cycle for four SIMDs), half of
// that with QT = 2; registers (116-161 and 163-213) leave three and two blocks of four waves a CU.
// Three blocks, by what keeps one on every CU (at_block): four waves of 16 rows; eight of 16 and chunks of 256 rows, which
// need half the barriers; four of 32.  us forward / backward: 512 keys for 32 heads 10.5 / 30, 10.0 / 28, 12 / 31; for 48
// (384 blocks of 64 or 192 of 128) 14.5 / 36, 11.1 / 31, 13 / 34; for 96 22 / 53, 24 / 56, 20 / 52; 328 keys for 56 9.9 / 28,
// 9.2 / 24, 9.9 / 25; 200 keys for 64 (256 blocks of 64) 5.9 / 15, 6.2 / 16, 7.5 / 18; for 96 7.4 / 20, 6.3 / 17, 7.7 / 19;
// 1024 keys for 24 22 / 57, 21 / 55, 23 / 58.
// 8 x 16 heads x 512 24 / 62 (105 / 183 as batched products with softmax kernels), 8 x 16 x 640 37 / 90 (115 / 192),
// 3 x 12 x 200 6 / 14 (23 / 31 with launches).  Error of the context (2-norm) 2.2e-3, as batched products, whose scores go
// through bf16, 4.2e-3.

// chunk of rows [r0, r0 + THREADS / 2) x 64 columns: global -> registers, registers -> LDS
template <int THREADS>
struct AtChunk {
    static constexpr int ITERS = THREADS / 2 * (AT_D / 8) / THREADS;
    u16x8 r[ITERS];
    __device__ __forceinline__ void load(const uint16_t* __restrict__ g, int ld, int r0, int rows, int tid) {
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int id = tid + it * THREADS;
            r[it] = *(const u16x8*)(g + (size_t)min(r0 + id / (AT_D / 8), rows - 1) * ld + (id % (AT_D / 8)) * 8);
        }
    }
    __device__ __forceinline__ void store(uint16_t* lds, int r0, int rows, int tid) const {
        const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int id = tid + it * THREADS;
            *(u16x8*)(lds + (id / (AT_D / 8)) * AT_P + (id % (AT_D / 8)) * 8) = r0 + id / (AT_D / 8) < rows ? r[it] : zero;
        }
    }
};

// WRITE_P: the probabilities, which need the sums, by a second pass over the keys (the first pass' bits stay the same).
template <int QT, int WAVES, bool WRITE_P>
__global__ __launch_bounds__(64 * WAVES, QT == 1 && WAVES == 4 ? 3 : 2) void attention_any_fwd_kernel(const uint16_t* __restrict__ qkv,
                                                                                   uint16_t* __restrict__ ctx,
                                                                                   uint16_t* __restrict__ probs,
                                                                                   float* __restrict__ lse2, int S, int heads,
                                                                                   float c) {
    constexpr int AT_CH = 32 * WAVES, NT = AT_CH / 16;
    __shared__ __attribute__((aligned(16))) uint16_t k_lds[AT_CH * AT_P];
    __shared__ __attribute__((aligned(16))) uint16_t v_lds[AT_CH * AT_P];

    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int li = lane % 16, g = lane / 16;
    const int bh = blockIdx.y, b = bh / heads, h = bh % heads;
    const int H = heads * AT_D, ld = 3 * H;
    const uint16_t* base = qkv + (size_t)b * S * ld + h * AT_D;
    AtChunk<64 * WAVES> kc, vc;
    kc.load(base + H, ld, 0, S, tid);
    vc.load(base + 2 * H, ld, 0, S, tid);

    const int q0 = (blockIdx.x * WAVES + wave) * 16 * QT + li;            // tile j of the wave: query q0 + 16 j
    bf16x8 qf[QT][2];
#pragma unroll
    for (int j = 0; j < QT; ++j)
#pragma unroll
        for (int s = 0; s < 2; ++s)
            qf[j][s] = __builtin_bit_cast(bf16x8, *(const u16x8*)(base + (size_t)min(q0 + 16 * j, S - 1) * ld + 32 * s + 8 * g));

    float m[QT], sum[QT];
    float4_t oacc[QT][4];
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        m[j] = -FLT_MAX;
        sum[j] = 0.f;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) oacc[j][dt] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (int k0 = 0; k0 < S; k0 += AT_CH) {
        if (k0) __syncthreads();                       // the last chunk's fragments are read
        kc.store(k_lds, k0, S, tid);
        vc.store(v_lds, k0, S, tid);
        __syncthreads();
        if (k0 + AT_CH < S) {
            kc.load(base + H, ld, k0 + AT_CH, S, tid);
            vc.load(base + 2 * H, ld, k0 + AT_CH, S, tid);
        }
        float4_t sc[QT][NT];
        float top[QT];
#pragma unroll
        for (int j = 0; j < QT; ++j) top[j] = m[j];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int j = 0; j < QT; ++j) sc[j][t] = float4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            if (k0 + 16 * t >= S) continue;
            float4_t acc[QT];
#pragma unroll
            for (int j = 0; j < QT; ++j) acc[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const bf16x8 kf = at_frag(k_lds, 16 * t + li, s, g);
#pragma unroll
                for (int j = 0; j < QT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[j][s], acc[j], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < QT; ++j) {
                if (k0 + 16 * t + 4 * g < S) sc[j][t] = acc[j];       // (seq is a multiple of 4)
#pragma unroll
                for (int e = 0; e < 4; ++e) top[j] = fmaxf(top[j], sc[j][t][e]);
            }
        }
#pragma unroll
        for (int j = 0; j < QT; ++j) {
            top[j] = fmaxf(top[j], __shfl_xor(top[j], 16, 64));
            top[j] = fmaxf(top[j], __shfl_xor(top[j], 32, 64));
            const float fade = __builtin_amdgcn_exp2f((m[j] - top[j]) * c);
            m[j] = top[j];
            sum[j] *= fade;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) oacc[j][dt] *= fade;
        }
#pragma unroll
        for (int u = 0; u < NT / 2; ++u) {
            if (k0 + 32 * u >= S) continue;
            bf16x8 pf[QT];
#pragma unroll
            for (int j = 0; j < QT; ++j) {
                u16x8 p;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = __builtin_amdgcn_exp2f((sc[j][2 * u + e / 4][e % 4] - m[j]) * c);
                    sum[j] += v;
                    p[e] = at_f2bf(v);
                }
                pf[j] = __builtin_bit_cast(bf16x8, p);
            }
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const bf16x8 vt = at_frag_t(v_lds, u, dt, li, g);
#pragma unroll
                for (int j = 0; j < QT; ++j)
                    oacc[j][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt, pf[j], oacc[j][dt], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        const int q = q0 + 16 * j;
        sum[j] += __shfl_xor(sum[j], 16, 64);
        sum[j] += __shfl_xor(sum[j], 32, 64);
        if (q >= S) continue;
        const float inv = 1.0f / sum[j];
        if (lse2 && g == 0) lse2[(size_t)bh * S + q] = m[j] * c + __builtin_amdgcn_logf(sum[j]);
        uint16_t* crow = ctx + ((size_t)b * S + q) * H + h * AT_D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) at_store4(crow + 16 * dt, oacc[j][dt] * inv);
    }
    if (!WRITE_P) return;
    for (int k0 = 0; k0 < S; k0 += AT_CH) {
        __syncthreads();
        kc.load(base + H, ld, k0, S, tid);
        kc.store(k_lds, k0, S, tid);
        __syncthreads();
        for (int t = 0; t < NT; ++t) {
            const int key = k0 + 16 * t + 4 * g;
#pragma unroll
            for (int j = 0; j < QT; ++j) {
                float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at_frag(k_lds, 16 * t + li, s, g), qf[j][s], acc, 0, 0, 0);
                const float inv = 1.0f / sum[j];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = __builtin_amdgcn_exp2f((acc[e] - m[j]) * c) * inv;
                if (key < S && q0 + 16 * j < S) at_store4(probs + ((size_t)bh * S + q0 + 16 * j) * S + key, acc);
            }
        }
    }
}

template <int QT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, QT == 1 && WAVES == 4 ? 3 : 2) void attention_any_bwd_q_kernel(const uint16_t* __restrict__ qkv,
                                                                                     const uint16_t* __restrict__ ctx,
                                                                                     const uint16_t* __restrict__ dctx,
                                                                                     const float* __restrict__ lse2,
                                                                                     float* __restrict__ delta_out,
                                                                                     uint16_t* __restrict__ dqkv, int S,
                                                                                     int heads, float c, float scale) {
    constexpr int AT_CH = 32 * WAVES, NT = AT_CH / 16;
    __shared__ __attribute__((aligned(16))) uint16_t k_lds[AT_CH * AT_P];
    __shared__ __attribute__((aligned(16))) uint16_t v_lds[AT_CH * AT_P];

    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int li = lane % 16, g = lane / 16;
    const int bh = blockIdx.y, b = bh / heads, h = bh % heads;
    const int H = heads * AT_D, ld = 3 * H;
    const uint16_t* base = qkv + (size_t)b * S * ld + h * AT_D;
    AtChunk<64 * WAVES> kc, vc;
    kc.load(base + H, ld, 0, S, tid);
    vc.load(base + 2 * H, ld, 0, S, tid);

    const int q0 = (blockIdx.x * WAVES + wave) * 16 * QT + li;
    bf16x8 qf[QT][2], dof[QT][2];
    float delta[QT], l2[QT];
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        const int q = q0 + 16 * j, qr = min(q, S - 1);
        const size_t orow = ((size_t)b * S + qr) * H + h * AT_D;
        delta[j] = 0.f;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            qf[j][s] = __builtin_bit_cast(bf16x8, *(const u16x8*)(base + (size_t)qr * ld + 32 * s + 8 * g));
            const u16x8 d8 = *(const u16x8*)(dctx + orow + 32 * s + 8 * g);
            const u16x8 o8 = *(const u16x8*)(ctx + orow + 32 * s + 8 * g);
            dof[j][s] = __builtin_bit_cast(bf16x8, d8);
#pragma unroll
            for (int e = 0; e < 8; ++e) delta[j] += at_bf2f(d8[e]) * at_bf2f(o8[e]);
        }
        delta[j] += __shfl_xor(delta[j], 16, 64);
        delta[j] += __shfl_xor(delta[j], 32, 64);
        l2[j] = lse2[(size_t)bh * S + qr];
        if (g == 0 && q < S) delta_out[(size_t)bh * S + q] = delta[j];
    }

    float4_t qacc[QT][4];
#pragma unroll
    for (int j = 0; j < QT; ++j)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) qacc[j][dt] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < S; k0 += AT_CH) {
        if (k0) __syncthreads();
        kc.store(k_lds, k0, S, tid);
        vc.store(v_lds, k0, S, tid);
        __syncthreads();
        if (k0 + AT_CH < S) {
            kc.load(base + H, ld, k0 + AT_CH, S, tid);
            vc.load(base + 2 * H, ld, k0 + AT_CH, S, tid);
        }
#pragma unroll 2
        for (int u = 0; u < NT / 2; ++u) {
            if (k0 + 32 * u >= S) break;
            u16x8 dsp[QT];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int t = 2 * u + half;
                float4_t sa[QT], da[QT];
#pragma unroll
                for (int j = 0; j < QT; ++j) sa[j] = da[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const bf16x8 kf = at_frag(k_lds, 16 * t + li, s, g), vf = at_frag(v_lds, 16 * t + li, s, g);
#pragma unroll
                    for (int j = 0; j < QT; ++j) {
                        sa[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[j][s], sa[j], 0, 0, 0);
                        da[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, dof[j][s], da[j], 0, 0, 0);
                    }
                }
                const bool live = k0 + 16 * t + 4 * g < S;            // (keys past the sequence: P = 0)
#pragma unroll
                for (int j = 0; j < QT; ++j) {
                    const float l = live ? l2[j] : INFINITY;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        // (P in bf16, as the forward pass uses it at 128 and 256; in chunks that rounds P times the sum)
                        const float p = at_bf2f(at_f2bf(__builtin_amdgcn_exp2f(sa[j][e] * c - l)));
                        dsp[j][4 * half + e] = at_f2bf(scale * p * (da[j][e] - delta[j]));
                    }
                }
            }
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const bf16x8 kt = at_frag_t(k_lds, u, dt, li, g);
#pragma unroll
                for (int j = 0; j < QT; ++j)
                    qacc[j][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt, __builtin_bit_cast(bf16x8, dsp[j]), qacc[j][dt], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        const int q = q0 + 16 * j;
        if (q >= S) continue;
        uint16_t* qrow = dqkv + ((size_t)b * S + q) * ld + h * AT_D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) at_store4(qrow + 16 * dt, qacc[j][dt]);
    }
}

template <int QT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, QT == 1 && WAVES == 4 ? 3 : 2) void attention_any_bwd_kv_kernel(const uint16_t* __restrict__ qkv,
                                                                                      const uint16_t* __restrict__ dctx,
                                                                                      const float* __restrict__ lse2,
                                                                                      const float* __restrict__ delta,
                                                                                      uint16_t* __restrict__ dqkv, int S,
                                                                                      int heads, float c, float scale) {
    constexpr int AT_CH = 32 * WAVES, NT = AT_CH / 16;
    __shared__ __attribute__((aligned(16))) uint16_t q_lds[AT_CH * AT_P];
    __shared__ __attribute__((aligned(16))) uint16_t do_lds[AT_CH * AT_P];
    __shared__ __attribute__((aligned(16))) float row_lds[2 * AT_CH];       // lse2, delta of the chunk's queries

    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int li = lane % 16, g = lane / 16;
    const int bh = blockIdx.y, b = bh / heads, h = bh % heads;
    const int H = heads * AT_D, ld = 3 * H;
    const uint16_t* base = qkv + (size_t)b * S * ld + h * AT_D;
    const uint16_t* dbase = dctx + (size_t)b * S * H + h * AT_D;
    const float* rows = (tid < AT_CH ? lse2 : delta) + (size_t)bh * S;
    AtChunk<64 * WAVES> qc, dc;
    float row;
    auto load = [&](int r0) {
        qc.load(base, ld, r0, S, tid);
        dc.load(dbase, H, r0, S, tid);
        // (queries past the sequence: P = 0)
        row = r0 + tid % AT_CH < S ? rows[r0 + tid % AT_CH] : tid < AT_CH ? INFINITY : 0.f;
    };
    load(0);

    const int key0 = (blockIdx.x * WAVES + wave) * 16 * QT + li;
    bf16x8 kf[QT][2], vf[QT][2];
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        const uint16_t* krow = base + (size_t)min(key0 + 16 * j, S - 1) * ld + H;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            kf[j][s] = __builtin_bit_cast(bf16x8, *(const u16x8*)(krow + 32 * s + 8 * g));
            vf[j][s] = __builtin_bit_cast(bf16x8, *(const u16x8*)(krow + H + 32 * s + 8 * g));
        }
    }

    float4_t kacc[QT][4], vacc[QT][4];
#pragma unroll
    for (int j = 0; j < QT; ++j)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) kacc[j][dt] = vacc[j][dt] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int q0 = 0; q0 < S; q0 += AT_CH) {
        if (q0) __syncthreads();
        qc.store(q_lds, q0, S, tid);
        dc.store(do_lds, q0, S, tid);
        row_lds[tid] = row;
        __syncthreads();
        if (q0 + AT_CH < S) load(q0 + AT_CH);
#pragma unroll 2
        for (int u = 0; u < NT / 2; ++u) {
            if (q0 + 32 * u >= S) break;
            u16x8 pp[QT], dsp[QT];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int t = 2 * u + half;
                float4_t sa[QT], da[QT];
#pragma unroll
                for (int j = 0; j < QT; ++j) sa[j] = da[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const bf16x8 qf = at_frag(q_lds, 16 * t + li, s, g), df = at_frag(do_lds, 16 * t + li, s, g);
#pragma unroll
                    for (int j = 0; j < QT; ++j) {
                        sa[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf, kf[j][s], sa[j], 0, 0, 0);
                        da[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(df, vf[j][s], da[j], 0, 0, 0);
                    }
                }
                const float4_t l2 = *(const float4_t*)(row_lds + 16 * t + 4 * g);
                const float4_t dl = *(const float4_t*)(row_lds + AT_CH + 16 * t + 4 * g);
#pragma unroll
                for (int j = 0; j < QT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint16_t pb = at_f2bf(__builtin_amdgcn_exp2f(sa[j][e] * c - l2[e]));
                        pp[j][4 * half + e] = pb;
                        dsp[j][4 * half + e] = at_f2bf(scale * at_bf2f(pb) * (da[j][e] - dl[e]));
                    }
            }
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const bf16x8 dot = at_frag_t(do_lds, u, dt, li, g), qt = at_frag_t(q_lds, u, dt, li, g);
#pragma unroll
                for (int j = 0; j < QT; ++j) {
                    vacc[j][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dot, __builtin_bit_cast(bf16x8, pp[j]), vacc[j][dt], 0, 0, 0);
                    kacc[j][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qt, __builtin_bit_cast(bf16x8, dsp[j]), kacc[j][dt], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < QT; ++j) {
        const int key = key0 + 16 * j;
        if (key >= S) continue;
        uint16_t* krow = dqkv + ((size_t)b * S + key) * ld + H + h * AT_D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            at_store4(krow + 16 * dt, kacc[j][dt]);
            at_store4(krow + H + 16 * dt, vacc[j][dt]);
        }
    }
}

int at_check(const char* who, int batch, int seq, int heads, int head_dim) {
    PD_REQUIRE(batch > 0 && heads > 0, PD_ESHAPE, "%s: batch and heads must be positive", who);
    PD_REQUIRE(pd_attention_fwd_supported(seq, head_dim), PD_ESHAPE,
               "%s: needs head_dim 64 and seq a multiple of 8 (got %d, %d)", who, head_dim, seq);
    PD_REQUIRE((long long)batch * heads <= 65535, PD_ESHAPE, "%s: too many (batch, head) pairs", who);
    return PD_OK;
}

// What a block takes: 64 queries (keys) by four waves of 16, 128 by eight waves of 16, or 128 by four waves of 32.
enum AtBlock { AT_64, AT_128, AT_128_WIDE };
AtBlock at_block(int batch, int seq, int heads) {
    const long pairs = (long)batch * heads;
    if ((seq + 63) / 64 * pairs <= 256) return AT_64;
    return (seq + 127) / 128 * pairs <= 256 ? AT_128 : AT_128_WIDE;
}

}  // namespace

extern "C" int pd_attention_fwd_supported(int seq, int head_dim) {
    return head_dim == AT_D && seq > 0 && seq % 8 == 0 && seq <= 65536;
}

extern "C" int pd_attention_fwd_bf16(const uint16_t* qkv, uint16_t* ctx, uint16_t* probs, float* lse2, int batch,
                                     int seq, int heads, int head_dim, void* stream) {
    int rc = at_check("pd_attention_fwd_bf16", batch, seq, heads, head_dim);
    if (rc != PD_OK) return rc;
    PD_REQUIRE(qkv && ctx, PD_EINVAL, "pd_attention_fwd_bf16: NULL pointer");
    PD_REQUIRE(pd_aligned(qkv, 16) && pd_aligned(ctx, 8) && (!probs || pd_aligned(probs, 8)), PD_EINVAL,
               "pd_attention_fwd_bf16: qkv must be 16-byte, ctx and probs 8-byte aligned");
    const float c = AT_LOG2E / sqrtf((float)head_dim);
    const dim3 grid(seq / AT_QB, batch * heads);
    hipStream_t s = (hipStream_t)stream;
    PD_REQUIRE(!probs || seq == 512 || seq == 256 || seq == 128, PD_ESHAPE,
               "pd_attention_fwd_bf16: probabilities only for seq 128, 256 and 512");
    // A head's K and V whole in LDS where they fit: us, whole / in chunks, 1 x 16 heads of 128 4.1 / 3.9, 8 x 16 4.4 / 4.2,
    // 16 x 16 4.7 / 5.7, 32 x 16 7.0 / 7.7, 64 x 16 15.4 / 16.1; of 256 1 x 16 5.9 / 5.8, 8 x 16 6.8 / 8.3, 32 x 16 23 / 26.
    if (seq == 128 && probs) attention_fwd_kernel<128, true><<<grid, AT_THREADS, 0, s>>>(qkv, ctx, probs, lse2, heads, c);
    else if (seq == 128) attention_fwd_kernel<128, false><<<grid, AT_THREADS, 0, s>>>(qkv, ctx, probs, lse2, heads, c);
    else if (seq == 256 && probs) attention_fwd_kernel<256, true><<<grid, AT_THREADS, 0, s>>>(qkv, ctx, probs, lse2, heads, c);
    else if (seq == 256) attention_fwd_kernel<256, false><<<grid, AT_THREADS, 0, s>>>(qkv, ctx, probs, lse2, heads, c);
    else {
        const AtBlock block = at_block(batch, seq, heads);
        const dim3 blocks(block == AT_64 ? (seq + 63) / 64 : (seq + 127) / 128, batch * heads);
        if (block == AT_64 && probs) attention_any_fwd_kernel<1, 4, true><<<blocks, 256, 0, s>>>(qkv, ctx, probs, lse2, seq, heads, c);
        else if (block == AT_64) attention_any_fwd_kernel<1, 4, false><<<blocks, 256, 0, s>>>(qkv, ctx, probs, lse2, seq, heads, c);
        else if (block == AT_128 && probs) attention_any_fwd_kernel<1, 8, true><<<blocks, 512, 0, s>>>(qkv, ctx, probs, lse2, seq, heads, c);
        else if (block == AT_128) attention_any_fwd_kernel<1, 8, false><<<blocks, 512, 0, s>>>(qkv, ctx, probs, lse2, seq, heads, c);
        else if (probs) attention_any_fwd_kernel<2, 4, true><<<blocks, 256, 0, s>>>(qkv, ctx, probs, lse2, seq, heads, c);
        else attention_any_fwd_kernel<2, 4, false><<<blocks, 256, 0, s>>>(qkv, ctx, probs, lse2, seq, heads, c);
    }
    PD_CHECK_LAUNCH("pd_attention_fwd_bf16");
    return PD_OK;
}

extern "C" int pd_attention_bwd_bf16(const uint16_t* qkv, const uint16_t* ctx, const uint16_t* dctx, const float* lse2,
                                     float* delta, uint16_t* dqkv, int batch, int seq, int heads, int head_dim,
                                     void* stream) {
    int rc = at_check("pd_attention_bwd_bf16", batch, seq, heads, head_dim);
    if (rc != PD_OK) return rc;
    PD_REQUIRE(qkv && ctx && dctx && lse2 && delta && dqkv, PD_EINVAL, "pd_attention_bwd_bf16: NULL pointer");
    PD_REQUIRE(pd_aligned(qkv, 16) && pd_aligned(ctx, 16) && pd_aligned(dctx, 16) && pd_aligned(lse2, 16) &&
                   pd_aligned(delta, 16) && pd_aligned(dqkv, 8),
               PD_EINVAL, "pd_attention_bwd_bf16: qkv, ctx, dctx, lse2, delta must be 16-byte, dqkv 8-byte aligned");
    const float scale = 1.0f / sqrtf((float)head_dim), c = AT_LOG2E * scale;
    hipStream_t s = (hipStream_t)stream;
    const AtBlock block = at_block(batch, seq, heads);
    const dim3 blocks(block == AT_64 ? (seq + 63) / 64 : (seq + 127) / 128, batch * heads);
    if (block == AT_64) attention_any_bwd_q_kernel<1, 4><<<blocks, 256, 0, s>>>(qkv, ctx, dctx, lse2, delta, dqkv, seq, heads, c, scale);
    else if (block == AT_128) attention_any_bwd_q_kernel<1, 8><<<blocks, 512, 0, s>>>(qkv, ctx, dctx, lse2, delta, dqkv, seq, heads, c, scale);
    else attention_any_bwd_q_kernel<2, 4><<<blocks, 256, 0, s>>>(qkv, ctx, dctx, lse2, delta, dqkv, seq, heads, c, scale);
    PD_CHECK_LAUNCH("pd_attention_bwd_bf16(dQ)");
    if (block == AT_64) attention_any_bwd_kv_kernel<1, 4><<<blocks, 256, 0, s>>>(qkv, dctx, lse2, delta, dqkv, seq, heads, c, scale);
    else if (block == AT_128) attention_any_bwd_kv_kernel<1, 8><<<blocks, 512, 0, s>>>(qkv, dctx, lse2, delta, dqkv, seq, heads, c, scale);
    else attention_any_bwd_kv_kernel<2, 4><<<blocks, 256, 0, s>>>(qkv, dctx, lse2, delta, dqkv, seq, heads, c, scale);
    PD_CHECK_LAUNCH("pd_attention_bwd_bf16(dK, dV)");
    return PD_OK;
}
