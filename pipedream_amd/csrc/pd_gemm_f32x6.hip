// fp32 GEMM on the gfx950 bf16 matrix pipes: C = op(A) op(B) with fp32 operands, fp32 accumulation and fp32
// accuracy, for the Linear / LSTM / projection layers of a stage (the same products as pd_gemm.hip, which see for
// what they replace in the reference).
//
// An fp32 value is the exact sum of three bf16 values (x1 = bf16(x), x2 = bf16(x - x1), x3 = bf16(x - x1 - x2)), a
// product of two bf16 values is exact in fp32, and v_mfma_f32_32x32x16_bf16 runs at sixteen times the rate of the
// fp32 MFMA, so  a b = a1 b1 + a1 b2 + a2 b1 + a2 b2 + a1 b3 + a3 b1  (the three products left out are below
// 2^-24 a b) costs six sixteenths of the fp32 MFMA time.
//
// The operands are split on their way into LDS: a thread fetches 8 consecutive k of one row (two 16-byte loads, or
// eight 4-byte loads where the reduction index is the row index of the stored matrix), splits them in registers
// (5.5 vector instructions a value, once per block and value) and writes one 16-byte unit to each of three planes in
// LDS, in the order in which the MFMA fragments are read.  Nothing but the fp32 operands is read from memory, and
// a fragment in LDS feeds one to three of the six products.
//
// Bound: the bf16 MFMA rate over six products, which on this part is a power limit: 8192^3 takes 5.8 ms = 187 TFLOP/s
// of fp32 products = 1.12 PFLOP/s of MFMAs (the library's bf16 product of that size 1.2-1.3), and 4.2 ms on operands
// of zeros.  Before (the better of the fp32 MFMA kernel and of six bf16 slots per operand written to memory and
// multiplied by the bf16 GEMM) 7.3 ms; LSTM products of 6400 rows: projection 6400 x 4096 x 1024 375 -> 294 us, its
// input gradient 432 -> 298, its weight gradient 401 -> 281; of 1240 rows 112 -> 79, 119 -> 76, 119 -> 64; the
// 32320-word classifier 2.47 / 3.17 / 2.73 -> 2.26 / 2.28 / 2.26 ms.
//
// 128 x 128 of C per block and work item, two persistent blocks of four waves on a CU (49 KB of LDS, 221-229
// registers), so that one block's epilogue and waits run beside the other's loop; the chunks of a block's items form
// one sequence, so only its first item waits for memory (K = 64, 6272 items: 157 -> 125 us).  128 x 256 per block
// with one wave per SIMD was within 2 % on the classifier and 4-17 % slower on the LSTM products.
#include <type_traits>

#include "pd_internal.h"

typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr int XK = 16;                         // reduction depth of a chunk = of one MFMA
constexpr int X_THREADS = 256;
constexpr int X_TILE = 128;                    // rows and columns of C per block

struct GemmX6Args {
    const float* A;
    const float* B;
    float* C;
    const float* bias;          // [N] or null
    int M, N, K;
    int lda, ldb, ldc;
    float beta;
    int tiles_m, tiles_n, items_per_die;
    int splits, k_per_split;    // work item (tile, z) owns k in [z * k_per_split, ...) and writes C + z * c_split
    int chunks;                 // ... as this many chunks of 16 k (even; those past K are zeros)
    long long c_split;
};

// (the instruction itself: from two conversions the compiler makes an instruction per use of a half)
__device__ __forceinline__ uint32_t x6_pack(float lo, float hi) {
    uint32_t p;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(p) : "v"(lo), "v"(hi));
    return p;
}

// One operand of a block: ROWS rows (of the m or n index) x 16 k per chunk, as `PER` units of 8 k per thread.
// KC: k is contiguous in memory ([rows][k]), else the row index is ([k][rows]).
template <int ROWS, bool KC>
struct X6Operand {
    static constexpr int PER = ROWS * 2 / X_THREADS;
    static constexpr int PLANE = ROWS * 32;            // bytes of one plane of a stage
    static constexpr int STAGE = 3 * PLANE;

    const float* base;          // first element of the next chunk: of the block's first row (KC), of its first k row
    uint32_t voff[PER];         // byte offset of the thread's units from there
    uint32_t lead;              // KC: bytes from the block's first row to its last
    int cols;                   // else: elements of a row behind the block's first
    int k_left;                 // K minus the first k of the next chunk
    float x[PER][8];

    // unit j of a thread: row and half of the 16 k
    __device__ static __forceinline__ int row_of(int j, int tid) { return KC ? (tid + j * X_THREADS) / 2 : (tid + j * X_THREADS) % ROWS; }
    __device__ static __forceinline__ int kh_of(int j, int tid) { return KC ? (tid + j * X_THREADS) % 2 : (tid + j * X_THREADS) / ROWS; }
    // Where it goes in a plane: tiles of 32 rows, the two halves one after the other; the second half swaps
    // neighbouring groups of four rows, so that the eight lanes of a write phase (four rows, both halves when KC) fall
    // into different banks.
    __device__ static __forceinline__ uint32_t dst_of(int j, int tid) {
        const int row = row_of(j, tid), kh = kh_of(j, tid);
        return (uint32_t)((row / 32) * 1024 + kh * 512 + ((row % 32) ^ (kh * 4)) * 16);
    }
    __device__ __forceinline__ void start(const float* m, int ld, int row0, int rows, int K, int k_begin, int tid) {
        k_left = K - k_begin;
        const int here = min(ROWS, rows - row0);
        base = m + (KC ? (size_t)row0 * ld + k_begin : (size_t)k_begin * ld + row0);
        lead = (uint32_t)((here - 1) * ld) * 4;
        cols = rows - row0;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int row = row_of(j, tid), kh = kh_of(j, tid);
            voff[j] = row < here ? (uint32_t)(KC ? row * ld + kh * 8 : kh * 8 * ld + row) * 4 : 0x80000000u;
        }
    }
    // requests unit j of the chunk; rows and k outside the matrix read 0
    __device__ __forceinline__ void load(int j, int ld, int tid) {
        if (KC) {
            // (never past the last row's end, and never 2^31 or more: an offset of 0x80000000 always reads 0)
            const uint32_t bytes = lead + (uint32_t)max(k_left, 0) * 4;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t off = kh_of(j, tid) * 8 + 4 * q < k_left ? voff[j] : 0x80000000u;
                const float4_t v = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * q, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][4 * q + e] = v[e];
            }
        } else {
            const int n = min(XK, k_left);
            const uint32_t ext = n > 0 ? (uint32_t)(((n - 1) * ld + cols) * 4) : 0u;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, ext, 0x00020000);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                x[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, voff[j] + (uint32_t)(e * ld * 4), 0, 0));
        }
    }
    __device__ __forceinline__ void next_chunk(int ld) {
        k_left -= XK;
        base += KC ? XK : (size_t)XK * ld;
    }
};

// Waves 2 x 2, each 2 x 2 MFMA tiles of 32 x 32.
template <bool A_KC, bool B_KC>
__global__ __launch_bounds__(X_THREADS, 2) void pd_gemm_f32x6_kernel(const GemmX6Args a) {
    constexpr int BM = X_TILE, BN = X_TILE, TM = 2, TN = 2, T = TM * TN;
    using OA = X6Operand<BM, A_KC>;
    using OB = X6Operand<BN, B_KC>;
    __shared__ __attribute__((aligned(1024))) char lds_a[2 * OA::STAGE];
    __shared__ __attribute__((aligned(1024))) char lds_b[2 * OB::STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int idx = lane & 31, h = lane >> 5;

    // Persistent blocks.  They go round-robin to the 8 dies: a die takes a contiguous range of the work items
    // (k ranges of one after the other, tiles numbered down columns of 8 tile rows), so that the blocks that share
    // its L2 cover a compact patch of C.
    const int per_die = gridDim.x >> 3, slot = blockIdx.x >> 3;
    const int item0 = (blockIdx.x & 7) * a.items_per_die;
    const int n_items = min(a.items_per_die, a.tiles_m * a.tiles_n * a.splits - item0);
    struct Item { int m0, n0, k0, z; };
    auto item_at = [&](int i) {
        const int tiles = a.tiles_m * a.tiles_n;
        Item it;
        it.z = (item0 + i) / tiles;
        const int t = (item0 + i) - it.z * tiles;
        const int group = t / (8 * a.tiles_n), in_group = t - group * 8 * a.tiles_n;
        const int rows_here = min(8, a.tiles_m - group * 8);
        it.n0 = (in_group / rows_here) * BN;
        it.m0 = (group * 8 + in_group - (in_group / rows_here) * rows_here) * BM;
        it.k0 = it.z * a.k_per_split;
        return it;
    };

    // Two sums: a1 b1, and the five products that are 2^-8 of it and less.  On one accumulator each of the six would
    // round the running sum: 3 times the rounding error (K = 1024: 5e-7 instead of 1.9e-7 of the result).
    float16_t acc[TM][TN], low[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.f;
    };

    OA oa;
    OB ob;
    int l_i = slot, l_kt = 0;                  // what is loaded next: item, chunk
    auto start_item = [&]() {
        const Item it = item_at(l_i);
        oa.start(a.A, a.lda, it.m0, a.M, a.K, it.k0, tid);
        ob.start(a.B, a.ldb, it.n0, a.N, a.K, it.k0, tid);
    };
    auto next_load = [&]() {
        if (++l_kt < a.chunks) {
            oa.next_chunk(a.lda);
            ob.next_chunk(a.ldb);
            return;
        }
        l_kt = 0;
        l_i += per_die;
        if (l_i < n_items) start_item();
        else oa.k_left = ob.k_left = 0;        // past the end: every load reads 0 without touching memory
    };

    // Split of units 0 .. PER_ALL-1 (A's, then B's) of the chunk in registers, in four pieces of two values.
    constexpr int PER_ALL = OA::PER + OB::PER;
    uint32_t pk[3][4];
    auto split_pair = [&](int u, int q) {
        const float x0 = u < OA::PER ? oa.x[u < OA::PER ? u : 0][2 * q] : ob.x[u < OA::PER ? 0 : u - OA::PER][2 * q];
        const float x1 = u < OA::PER ? oa.x[u < OA::PER ? u : 0][2 * q + 1] : ob.x[u < OA::PER ? 0 : u - OA::PER][2 * q + 1];
        const uint32_t p1 = x6_pack(x0, x1);
        const float r0 = x0 - __builtin_bit_cast(float, p1 << 16), r1 = x1 - __builtin_bit_cast(float, p1 & 0xffff0000u);
        const uint32_t p2 = x6_pack(r0, r1);
        const float s0 = r0 - __builtin_bit_cast(float, p2 << 16), s1 = r1 - __builtin_bit_cast(float, p2 & 0xffff0000u);
        pk[0][q] = p1;
        pk[1][q] = p2;
        pk[2][q] = x6_pack(s0, s1);
    };
    auto write_unit = [&](int u, int stage) {
        char* const to = u < OA::PER ? lds_a + stage * OA::STAGE + OA::dst_of(u < OA::PER ? u : 0, tid)
                                     : lds_b + stage * OB::STAGE + OB::dst_of(u < OA::PER ? 0 : u - OA::PER, tid);
        const int plane = u < OA::PER ? OA::PLANE : OB::PLANE;
#pragma unroll
        for (int p = 0; p < 3; ++p)
            *(u32x4_t*)(to + p * plane) = u32x4_t{pk[p][0], pk[p][1], pk[p][2], pk[p][3]};
    };
    auto load_unit = [&](int u) {
        if (u < OA::PER) oa.load(u < OA::PER ? u : 0, a.lda, tid);
        else ob.load(u < OA::PER ? 0 : u - OA::PER, a.ldb, tid);
    };

    const uint32_t fa = (uint32_t)(wm * TM * 1024 + h * 512 + (idx ^ (h * 4)) * 16);
    const uint32_t fb = (uint32_t)(wn * TN * 1024 + h * 512 + (idx ^ (h * 4)) * 16);
    bf16x8_t af[3][TM], bf[2][TN];             // terms of A; the term of B in use and the next one
    auto read_a = [&](int stage, int plane, int i) {
        af[plane][i] = *(const bf16x8_t*)(lds_a + stage * OA::STAGE + plane * OA::PLANE + i * 1024 + fa);
    };
    auto read_b = [&](int buf, int stage, int plane, int j) {
        bf[buf][j] = *(const bf16x8_t*)(lds_b + stage * OB::STAGE + plane * OB::PLANE + j * 1024 + fb);
    };

    // prologue: chunk 0 into LDS stage 0, chunk 1 on its way to the registers
    if (slot >= n_items) return;               // whole block, before any barrier
    start_item();
#pragma unroll
    for (int u = 0; u < PER_ALL; ++u) load_unit(u);
    next_load();
#pragma unroll
    for (int u = 0; u < PER_ALL; ++u) {
#pragma unroll
        for (int q = 0; q < 4; ++q) split_pair(u, q);
        write_unit(u, 0);
        load_unit(u);
    }
    next_load();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i) read_a(0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; ++j) read_b(0, 0, 2, j);

    // One chunk: the products a1 b3, a1 b2, a2 b2, a1 b1, a2 b1, a3 b1, T MFMAs each, every MFMA followed by a small
    // piece of other work that the scheduler may not move: a fragment of a later product from LDS, or a part of the
    // next chunk's split (registers -> other LDS stage, and the request of the chunk after it).  The barrier sits
    // behind the fourth product; the last two cover the first fragment reads of the next chunk.
    auto chunk = [&](auto stage_c, auto buf_c) {
        constexpr int st = decltype(stage_c)::value, b0 = decltype(buf_c)::value, b1 = b0 ^ 1;
        constexpr int PIECES = 6 * PER_ALL;    // per unit: four pairs, the writes, the loads
#pragma unroll
        for (int s = 0; s < 6 * T; ++s) {
            const int prod = s / T, i = (s % T) / TN, j = s % TN;
            const int ap = prod == 2 || prod == 4 ? 1 : prod == 5 ? 2 : 0;
            const int bb = prod == 0 ? b0 : prod <= 2 ? b1 : b0;
            if (prod == 3) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ap][i], bf[bb][j], acc[i][j], 0, 0, 0);
            else low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ap][i], bf[bb][j], low[i][j], 0, 0, 0);
            // fragments: during a1 b3 those of a2, b2; during a1 b2, a2 b2 those of a3, b1
            if (s < TN) read_b(b1, st, 1, s);
            else if (s < TN + TM) read_a(st, 1, s - TN);
            if (s >= T && s < T + TN) read_b(b0, st, 0, s - T);
            else if (s >= T + TN && s < T + TN + TM) read_a(st, 2, s - T - TN);
            // pieces of the split, spread over the first four products
#pragma unroll
            for (int p = 0; p < PIECES; ++p)
                if (p * 4 * T / PIECES == s) {
                    const int u = p / 6, what = p % 6;
                    if (what < 4) split_pair(u, what);
                    else if (what == 4) write_unit(u, st ^ 1);
                    else load_unit(u);
                }
            if (s == 4 * T - 1) __syncthreads();
            if (s >= 4 * T && s < 4 * T + TN) read_b(b1, st ^ 1, 2, s - 4 * T);
            else if (s >= 4 * T + TN && s < 4 * T + TN + TM) read_a(st ^ 1, 0, s - 4 * T - TN);
            __builtin_amdgcn_sched_barrier(0);
        }
        next_load();
    };
    static_assert(TN + TM <= 2 * T && T + TN + TM <= 3 * T + 2, "fragment reads fit their slots");
    using c0 = std::integral_constant<int, 0>;
    using c1 = std::integral_constant<int, 1>;
    for (int i = slot; i < n_items; i += per_die) {
        const Item it = item_at(i);
        clear();
        for (int kt = 0; kt < a.chunks; kt += 2) {         // (an even number of chunks: the LDS stages keep their turn)
            chunk(c0{}, c0{});
            chunk(c1{}, c1{});
        }

        bool bad = false;
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int tj = 0; tj < TN; ++tj) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[ti][tj][e] += low[ti][tj][e];
                    bad |= !(__builtin_fabsf(acc[ti][tj][e]) <= 3.4028235e38f);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        if (__any(bad)) {
            // Infinities and values that round to infinity in bf16 leave NaNs (inf - inf in the split), and the product of
            // two leading terms, both rounded up, may overflow where the product itself does not: a wave that holds a NaN or
            // an infinity computes its part again with fp32 MFMAs straight from memory, which gives what fp32 gives.
            const int k_end = min(a.K, it.k0 + a.k_per_split);
            clear();
            for (int k = it.k0; k < k_end; k += 2) {
                const bool k_ok = k + h < k_end;
                float va[TM], vb[TN];
#pragma unroll
                for (int ti = 0; ti < TM; ++ti) {
                    const int r = it.m0 + (wm * TM + ti) * 32 + idx;
                    va[ti] = k_ok && r < a.M ? a.A[A_KC ? (size_t)r * a.lda + k + h : (size_t)(k + h) * a.lda + r] : 0.f;
                }
#pragma unroll
                for (int tj = 0; tj < TN; ++tj) {
                    const int r = it.n0 + (wn * TN + tj) * 32 + idx;
                    vb[tj] = k_ok && r < a.N ? a.B[B_KC ? (size_t)r * a.ldb + k + h : (size_t)(k + h) * a.ldb + r] : 0.f;
                }
#pragma unroll
                for (int ti = 0; ti < TM; ++ti)
#pragma unroll
                    for (int tj = 0; tj < TN; ++tj)
                        acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[ti], vb[tj], acc[ti][tj], 0, 0, 0);
            }
        }

        // Accumulator element e of lane (idx, h): row 8 (e / 4) + 4 h + e % 4, column idx of its tile.
        float* const C = a.C + it.z * a.c_split;
        const bool inside = it.m0 + BM <= a.M && it.n0 + BN <= a.N;
#pragma unroll
        for (int ti = 0; ti < TM; ++ti)
#pragma unroll
            for (int tj = 0; tj < TN; ++tj) {
                const int col = it.n0 + (wn * TN + tj) * 32 + idx;
                const int row0 = it.m0 + (wm * TM + ti) * 32 + 4 * h;
                const float bv = a.bias && col < a.N ? a.bias[col] : 0.f;
                float* const to = C + (size_t)row0 * a.ldc + col;
                if (inside && a.beta == 0.f) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) to[(size_t)(8 * (e / 4) + e % 4) * a.ldc] = acc[ti][tj][e] + bv;
                } else if (col < a.N) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int r = 8 * (e / 4) + e % 4;
                        if (row0 + r < a.M) {
                            float* const p = to + (size_t)r * a.ldc;
                            float v = acc[ti][tj][e] + bv;
                            if (a.beta != 0.f) v += a.beta * *p;
                            *p = v;
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
    }
}

}  // namespace

extern "C" int pd_gemm_f32x6(int trans_a, int trans_b, int M, int N, int K, const float* A, int lda, const float* B,
                             int ldb, float beta, float* C, int ldc, const float* bias, int splits, float* partials,
                             void* stream) {
    PD_REQUIRE(M > 0 && N > 0 && K > 0 && splits >= 1 && splits <= 64, PD_ESHAPE, "pd_gemm_f32x6: bad dimensions");
    PD_REQUIRE(A && B && C && (splits == 1 || partials), PD_EINVAL, "pd_gemm_f32x6: NULL operand");
    PD_REQUIRE(lda >= (trans_a ? M : K) && ldb >= (trans_b ? K : N) && ldc >= N, PD_ESHAPE,
               "pd_gemm_f32x6: leading dimension smaller than the row length");
    // an operand whose rows hold the reduction index is read 16 bytes at a time
    PD_REQUIRE(trans_a || (pd_aligned(A, 16) && lda % 4 == 0 && K % 4 == 0), PD_EINVAL, "pd_gemm_f32x6: A is not 16-byte aligned");
    PD_REQUIRE(!trans_b || (pd_aligned(B, 16) && ldb % 4 == 0 && K % 4 == 0), PD_EINVAL, "pd_gemm_f32x6: B is not 16-byte aligned");
    PD_REQUIRE(lda < (1 << 20) && ldb < (1 << 20), PD_ESHAPE, "pd_gemm_f32x6: leading dimension too large");
    GemmX6Args g;
    g.A = A; g.B = B;
    g.M = M; g.N = N; g.K = K;
    g.lda = lda; g.ldb = ldb;
    g.k_per_split = ((K + splits - 1) / splits + 2 * XK - 1) / (2 * XK) * (2 * XK);
    g.chunks = g.k_per_split / XK;
    splits = (K + g.k_per_split - 1) / g.k_per_split;       // (no empty range)
    if (splits > 1) {
        PD_REQUIRE(N % 4 == 0 && ldc % 4 == 0 && pd_aligned(partials, 16) && pd_aligned(C, 16) && pd_aligned(bias, 16), PD_EINVAL,
                   "pd_gemm_f32x6: a split reduction needs N and ldc multiples of 4, aligned results and an aligned bias");
        g.C = partials; g.ldc = N; g.bias = nullptr; g.beta = 0.f; g.c_split = (long long)M * N;
    } else {
        g.C = C; g.ldc = ldc; g.bias = bias; g.beta = beta; g.c_split = 0;
    }
    hipStream_t s = (hipStream_t)stream;
    g.tiles_m = (M + X_TILE - 1) / X_TILE;
    g.tiles_n = (N + X_TILE - 1) / X_TILE;
    g.splits = splits;
    const long items = (long)g.tiles_m * g.tiles_n * splits;
    PD_REQUIRE(items < (1l << 30), PD_ESHAPE, "pd_gemm_f32x6: too many tiles");
    g.items_per_die = (int)((items + 7) / 8);
    const dim3 grid(8 * (unsigned)(g.items_per_die < 64 ? g.items_per_die : 64));     // two resident blocks per CU
    if (!trans_a && trans_b) pd_gemm_f32x6_kernel<true, true><<<grid, X_THREADS, 0, s>>>(g);
    else if (!trans_a) pd_gemm_f32x6_kernel<true, false><<<grid, X_THREADS, 0, s>>>(g);
    else if (!trans_b) pd_gemm_f32x6_kernel<false, false><<<grid, X_THREADS, 0, s>>>(g);
    else pd_gemm_f32x6_kernel<false, true><<<grid, X_THREADS, 0, s>>>(g);
    PD_CHECK_LAUNCH("pd_gemm_f32x6");
    if (splits == 1) return PD_OK;
    return pd_splitk_reduce_f32(partials, splits, M, N, bias, 0, beta, C, ldc, stream);
}
