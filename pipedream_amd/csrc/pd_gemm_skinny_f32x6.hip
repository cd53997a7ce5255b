// fp32 products with at most 128 rows (Linear layers of a small batch: the classifiers of VGG16, MLPs) on the bf16 matrix
// pipes: the same calls as pd_gemm_f32 (which see for what they replace in the reference), arithmetic as in
// pd_gemm_f32x6.hip (each operand the exact sum of three bf16 terms, six MFMAs a product).
//
// Such a product reads a large B once.  A block owns 16 RT x 16 CT of C and one range of k; its eight waves take an
// eighth of the range each, with both operands straight from memory into registers in MFMA order: no LDS and no
// barrier in the loop, and each wave's next chunk of 32 k is on its way while it multiplies.  The eight partial sums
// meet in LDS and are added in wave order (and over the ranges by pd_splitk_reduce_f32, unless there is only one).
//   B k-contiguous ([N][K]): lane (n = lane % 16, lane / 16) reads 8 consecutive k of its row.
//   B row-contiguous ([K][N]): it reads CT consecutive columns of 8 rows of B; column CT i + j of the block is column
//   i of MFMA tile j, so that what one lane fetches are the fragments of CT tiles and nothing is transposed.
// Bound: reading B from memory, 5.4 TB/s at 8 rows; from 64 rows on also the conversions (both operands, once per block)
// beside the MFMAs.  us, launches and sums included, before (fp32 MFMA kernel with 64 rows a block whatever M is,
// operands through an LDS ring with a barrier per 16 k) / now: 8 x 4096 x 25088 154 / 76, 64 x 4096 x 25088 176 / 123,
// its input gradient 202 / 126, 64 x 4096 x 4096 30 / 27 and 30 / 24.  Error against 64 bits (2-norm) 2.9e-7 / 1.6e-7 at
// K = 1024, 1.0e-6 / 4.8e-7 at 25088.
#include "pd_f32x6.hpp"

namespace {

constexpr int KX_WAVES = 8;
constexpr int KX_THREADS = 64 * KX_WAVES;

struct SkinnyX6Args {
    const float* A;             // [M][lda]
    const float* B;             // [N][ldb] or [K][ldb]
    float* C;                   // partial sums [splits][M][N], or (one range) the result [M][ldc]
    const float* bias;          // one range: [N] or null
    int M, N, K;
    int lda, ldb, ldc;
    float beta;
    int relu;
    int row_blocks, col_blocks, splits, items_per_die;
};

template <int RT, int CT, bool B_KC>
__global__ __launch_bounds__(KX_THREADS, 2) void pd_gemm_skinny_f32x6_kernel(const SkinnyX6Args a) {
    constexpr int ROWS = 16 * RT, COLS = 16 * CT;
    constexpr int P = RT <= 2 ? 32 : 64;           // floats of a column of a partial tile in LDS: a multiple of 8 units of 16 bytes
    __shared__ __attribute__((aligned(16))) float part[KX_WAVES][COLS * P];

    // a die's blocks share columns of B (its row blocks) and ranges of k
    const int item = (blockIdx.x & 7) * a.items_per_die + (blockIdx.x >> 3);
    if (item >= a.row_blocks * a.col_blocks * a.splits) return;                   // whole block
    const int row0 = item % a.row_blocks * ROWS;
    const int t = item / a.row_blocks;
    const int z = t / a.col_blocks, n0 = t % a.col_blocks * COLS;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int idx = lane & 15, kq = lane >> 4;

    f32x4_t acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int chunks = (a.K + 31) / 32, ways = a.splits * KX_WAVES, way = z * KX_WAVES + wave;
    const int c0 = (int)((long)chunks * way / ways), n = (int)((long)chunks * (way + 1) / ways) - c0;
    if (n > 0) {
        const int k0 = c0 * 32 + 8 * kq;
        const float* ap[RT];                       // (rows past M read the last one, columns past N the last ones: dropped)
#pragma unroll
        for (int i = 0; i < RT; ++i) ap[i] = a.A + (size_t)min(row0 + 16 * i + idx, a.M - 1) * a.lda + k0;
        const float* bp[B_KC ? CT : 1];
        if (B_KC) {
#pragma unroll
            for (int j = 0; j < CT; ++j) bp[B_KC ? j : 0] = a.B + (size_t)min(n0 + 16 * j + idx, a.N - 1) * a.ldb + k0;
        } else {
            bp[0] = a.B + (size_t)k0 * a.ldb + min(n0 + CT * idx, a.N - CT);
        }
        float ar[RT][8], br[CT][8];
        // A lane's eight k are inside the reduction or past its end together (K is a multiple of 8).  Past it the
        // lane reads the last ones again, and its A counts as zero.
        auto load_a = [&](int i, int c) {
            const float* src = ap[i] + c * 32 + min(0, a.K - 8 - (k0 + c * 32));
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4_t v = *(const f32x4_t*)(src + 4 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) ar[i][4 * q + e] = v[e];
            }
            if ((c0 + c) * 32 + 32 > a.K) {        // the last chunk of a K that 32 does not divide
#pragma unroll
                for (int e = 0; e < 8; ++e) ar[i][e] = k0 + c * 32 < a.K ? ar[i][e] : 0.f;
            }
        };
        auto load_b = [&](int c) {
            const int at = c * 32 + min(0, a.K - 8 - (k0 + c * 32));
            if (B_KC) {
#pragma unroll
                for (int j = 0; j < CT; ++j)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const f32x4_t v = *(const f32x4_t*)(bp[B_KC ? j : 0] + at + 4 * q);
#pragma unroll
                        for (int e = 0; e < 4; ++e) br[j][4 * q + e] = v[e];
                    }
            } else {
                typedef float vec_t __attribute__((ext_vector_type(CT)));
                const float* src = bp[0] + (long)at * a.ldb;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const vec_t v = *(const vec_t*)(src + (size_t)e * a.ldb);
#pragma unroll
                    for (int j = 0; j < CT; ++j) br[j][e] = v[j];
                }
            }
        };
        load_b(0);
#pragma unroll
        for (int i = 0; i < RT; ++i) load_a(i, 0);
        const float sign = pd_x6_sign(chunks, ways, way);
        for (int c = 0; c < n; ++c) {
            const int next = min(c + 1, n - 1);    // (past the end the last chunk is fetched again)
            u32x4_t bt[CT][3];
#pragma unroll
            for (int j = 0; j < CT; ++j) pd_x6_split8(br[j], bt[j]);
            load_b(next);
            // a row tile is split just before its MFMAs: one wave's conversions run beside the other's MFMAs
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                u32x4_t at[3];
                pd_x6_split8<true>(ar[i], at, sign);
                load_a(i, next);
#pragma unroll
                for (int s = 0; s < 6; ++s)
#pragma unroll
                    for (int j = 0; j < CT; ++j) acc[i][j] = pd_x6_mfma(at[PD_X6_A[s]], bt[j][PD_X6_B[s]], acc[i][j]);
            }
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] *= sign;

        bool bad = false;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) bad |= !(__builtin_fabsf(acc[i][j][e]) <= 3.4028235e38f);
        if (__any(bad)) {
            // infinities and values that round to infinity in bf16 leave NaNs: once more with fp32 MFMAs, which give
            // what fp32 gives
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            for (int k = c0 * 32 + kq; k < min(a.K, (c0 + n) * 32); k += 4) {     // (K is a multiple of 4)
                float bv[CT];
#pragma unroll
                for (int j = 0; j < CT; ++j)
                    bv[j] = B_KC ? a.B[(size_t)min(n0 + 16 * j + idx, a.N - 1) * a.ldb + k]
                                 : a.B[(size_t)k * a.ldb + min(n0 + CT * idx, a.N - CT) + j];
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const float av = a.A[(size_t)min(row0 + 16 * i + idx, a.M - 1) * a.lda + k];
#pragma unroll
                    for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    }

    // Element e of lane (idx, kq): row 4 kq + e, column idx of its tile.  Columns of a partial tile lie P floats apart,
    // groups of four rows within one at the group's number xor swizzle(column): eight lanes that write neighbouring
    // columns of a tile, or read neighbouring columns of C, meet eight different bank groups for either order of B.
    auto at = [&](int col, int group) { return col * P + 4 * (group ^ ((col ^ ((col >> 3) & 3)) & 7)); };
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
            *(f32x4_t*)&part[wave][at(B_KC ? 16 * j + idx : CT * idx + j, 4 * i + kq)] = acc[i][j];
    __syncthreads();
    float* const C = a.C + (size_t)z * a.M * a.N;
#pragma unroll
    for (int s = 0; s < (4 * RT * COLS + KX_THREADS - 1) / KX_THREADS; ++s) {
        const int id = s * KX_THREADS + threadIdx.x;
        const int col = id % COLS, group = id / COLS;
        if (group >= 4 * RT || n0 + col >= a.N) continue;
        f32x4_t v = *(const f32x4_t*)&part[0][at(col, group)];
#pragma unroll
        for (int w = 1; w < KX_WAVES; ++w) v += *(const f32x4_t*)&part[w][at(col, group)];
        const float bias = a.bias ? a.bias[n0 + col] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = row0 + 4 * group + e;
            if (row >= a.M) continue;
            float* const to = C + (size_t)row * a.ldc + n0 + col;
            float r = v[e] + bias;
            if (a.beta != 0.f) r += a.beta * *to;
            *to = a.relu && !(r > 0.f) ? 0.f : r;
        }
    }
}

template <int RT, int CT>
void launch_skinny(const SkinnyX6Args& g, int trans_b, hipStream_t s) {
    const dim3 grid(8 * g.items_per_die);
    if (trans_b) pd_gemm_skinny_f32x6_kernel<RT, CT, true><<<grid, KX_THREADS, 0, s>>>(g);
    else pd_gemm_skinny_f32x6_kernel<RT, CT, false><<<grid, KX_THREADS, 0, s>>>(g);
}

}  // namespace

// Columns of C per block, 64 or 32.
static int skinny_cols(int M, int N) { return (N + 63) / 64 * ((M + 63) / 64) <= 16 ? 32 : 64; }

// Ranges of k: one block per CU and a chunk of k per wave.  Up to 32 chunks (24 from 17 rows on, whose conversions spread
// over the CUs as well) stay in one piece, since the launch that adds up the ranges costs what they save: us, one piece /
// two ranges, 8 x 8192 x 768 11.3 / 11.4 and, B as [K][N], 8.1 / 10.1, x 1024 13.4 / 12.6 and 9.8 / 11.3,
// 32 x 5120 x 1024 16.5 / 14.0 and 11.2 / 10.9, x 8192 x 1024 17.0 / 14.7 and 11.6 / 12.1, x 768 13.7 / 13.5 and 9.3 / 11.5,
// 64 x 8192 x 768 18.4 / 19.2 and 15.3 / 18.3, x 1024 22.4 / 19.6 and 18.2 / 18.4.
extern "C" int pd_gemm_skinny_f32x6_splits(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= (M > 16 ? 768 : 1024)) return 1;
    const int cols = skinny_cols(M, N);
    const long blocks = (long)((N + cols - 1) / cols) * ((M + 63) / 64);
    const long most = (K + 31) / 32 / KX_WAVES, want = 256 / blocks;
    const long splits = want < most ? want : most;
    return splits < 1 ? 1 : (int)splits;
}

extern "C" int pd_gemm_skinny_f32x6(int trans_b, int M, int N, int K, const float* A, int lda, const float* B, int ldb,
                                    float beta, float* C, int ldc, const float* bias, int relu, int splits,
                                    float* partials, void* stream) {
    PD_REQUIRE(M > 0 && M <= 128 && N > 0 && K > 0 && splits >= 1 && splits <= 1024, PD_ESHAPE, "pd_gemm_skinny_f32x6: bad dimensions");
    PD_REQUIRE(A && B && C && (splits == 1 || partials), PD_EINVAL, "pd_gemm_skinny_f32x6: NULL operand");
    PD_REQUIRE(lda >= K && ldb >= (trans_b ? K : N) && ldc >= N, PD_ESHAPE,
               "pd_gemm_skinny_f32x6: leading dimension smaller than the row length");
    PD_REQUIRE(K % 8 == 0 && lda % 4 == 0 && ldb % 4 == 0 && (trans_b || N % 4 == 0) && pd_aligned(A, 16) && pd_aligned(B, 16),
               PD_EINVAL, "pd_gemm_skinny_f32x6: needs K a multiple of 8, lda, ldb (and N of a plain B) multiples of 4 and "
               "16-byte aligned operands");
    SkinnyX6Args g;
    g.A = A; g.B = B;
    g.M = M; g.N = N; g.K = K;
    g.lda = lda; g.ldb = ldb;
    g.splits = splits;
    if (splits > 1) {
        PD_REQUIRE(N % 4 == 0 && ldc % 4 == 0 && pd_aligned(partials, 16) && pd_aligned(C, 16) && pd_aligned(bias, 16), PD_EINVAL,
                   "pd_gemm_skinny_f32x6: a split reduction needs N and ldc multiples of 4, aligned results and an aligned bias");
        g.C = partials; g.ldc = N; g.bias = nullptr; g.beta = 0.f; g.relu = 0;
    } else {
        g.C = C; g.ldc = ldc; g.bias = bias; g.beta = beta; g.relu = relu != 0;
    }
    g.row_blocks = (M + 63) / 64;
    const int rt = ((M + g.row_blocks - 1) / g.row_blocks + 15) / 16;
    const int cols = skinny_cols(M, N);
    g.col_blocks = (N + cols - 1) / cols;
    const long items = (long)g.row_blocks * g.col_blocks * splits;
    PD_REQUIRE(items < (1l << 30), PD_ESHAPE, "pd_gemm_skinny_f32x6: too many blocks");
    g.items_per_die = (int)((items + 7) / 8);
    hipStream_t s = (hipStream_t)stream;
    if (cols == 64) {
        if (rt == 1) launch_skinny<1, 4>(g, trans_b, s);
        else if (rt == 2) launch_skinny<2, 4>(g, trans_b, s);
        else if (rt == 3) launch_skinny<3, 4>(g, trans_b, s);
        else launch_skinny<4, 4>(g, trans_b, s);
    } else {
        if (rt == 1) launch_skinny<1, 2>(g, trans_b, s);
        else if (rt == 2) launch_skinny<2, 2>(g, trans_b, s);
        else if (rt == 3) launch_skinny<3, 2>(g, trans_b, s);
        else launch_skinny<4, 2>(g, trans_b, s);
    }
    PD_CHECK_LAUNCH("pd_gemm_skinny_f32x6");
    if (splits == 1) return PD_OK;
    return pd_splitk_reduce_f32(partials, splits, M, N, bias, relu, beta, C, ldc, stream);
}
