// The Winograd F(2x2, 3x3) convolution of pd_conv3x3_winograd.hip (which see for the algorithm and what it replaces in
// the reference) on the f16 matrix pipes, with fp32 operands, fp32 accumulation and fp32 accuracy.  For input channel
// counts that are multiples of 16.
//
// An fp32 value, scaled by a power of two into f16's range, is the sum of two f16 values (x1 = f16(x), x2 = f16(x - x1))
// up to 2^-23 of it, or 2^-25 of f16's unit where that is more; products of f16 values are exact in fp32, so
// u v = u1 v1 + u1 v2 + u2 v1  up to 2^-21 u v (4 million products: 2^-21.1 at most, 2^-23.6 rms; the rounding of the
// running sum, eight times a chunk in the fp32 kernel and three times here, is what decides the error), three sixteenths
// of the time of the fp32 MFMA (v_mfma_f32_32x32x16_f16 runs at sixteen times its rate), and unlike an fp32 MFMA it runs
// beside vector instructions.  Splitting two values takes four instructions (v_cvt_pk_f16_f32, two v_fma_mix_f32 for the
// remainders, v_cvt_pk_f16_f32).
//
// f16 ends at 2^-24 below its unit, so a value far below the largest of its scale loses bits.  The scales are powers of two:
//   * filter, per output channel k and per input channel c: with e(k, c) the exponent of the largest tap, R(k) = max over c
//     of e and s(c) = max over k of e - R, w 2^-(R + s) is at most 1 to 2 everywhere and reaches it in every row and column;
//     it is split at 2^13 times that (|U| is at most 2.25 times |w|).  R comes out of the sums, s goes into the input: a
//     channel that is small and has large weights counts as much as one that is large and has small ones;
//   * input: x 2^s, one scale per 2x2-output tile, from the largest value of its patch in the first chunk of 16 channels;
//     that becomes 2^11 to 2^12 (|V| at most four times it).  The tile keeps its scale while later chunks stay below twice
//     that, else the scale follows and the waves that hold the tile's sums multiply them accordingly (a test per chunk,
//     hardly ever more).
// A value is then held to 2^-37.8 (rms) of the largest of its patch over all channels, and what that costs is bounded by what
// the largest contributes, provided that the channel it lies in has weights to speak of and that the pixel is one that the
// output sees.  Hence two tests, and fp32 MFMAs for the work items that fail one:
//   * a block of 64 output channels that holds a kernel w(k, c) which is zero, or below 2^-P of what its row and column
//     have, with 2^P sqrt(C) = 2^13 (the error is then 2^-24.8 even where all of an output comes through that kernel; random
//     filters of 512 x 512 channels reach 2^-4 of it);
//   * a tile whose four inner pixels, which all four outputs see, are below 2^-8 of its patch in all channels.
// Infinities, and values of 2^64 and more, cannot be split either.  A block that met one of those or such a tile stays on
// the fp32 MFMAs for one item, then for two, four, ... if it goes on.
//
// Bound: f16 MFMAs, vector instructions and LDS traffic side by side.  Per chunk of 16 channels a SIMD's two waves issue
// 48 MFMAs (1700 cycles) and 2 x 165 vector instructions, the block moves 290 KB through LDS (2300 cycles): 4100 cycles,
// where the fp32 kernel takes 9580 for the same chunk.  64 images, C = K = 128 at 112 x 112: 595 us (398 TFLOP/s of a
// direct convolution; 564 with one scale for all channels and no tests), C = K = 512 at 28 x 28: 530 us (446); 8 images
// 86 us.  With the weight gradient's kernel VGG16's front stage 7.7 -> 5.1 ms a step, all of VGG16 26.3 -> 17.2 ms, a
// validation pass over 2 x 8 images 3.68 -> 2.53 ms.  An item of 64 channels takes 28 000
// cycles, 9000 of them behind its last product; before its divisions went to the ring of decoded items 35 000.
// A block (512 threads, one per CU) owns 16 x 16 output pixels x 64 channels:
// wave (j, kh) holds column j of the 4 x 4 transformed positions for 64 tiles x 32 channels (128 accumulators a lane);
// filters are the A operand, so that a lane has four consecutive channels of a tile, and the wave folds its four rows to
// two before anything goes through LDS.  The chunks of a block's items form one sequence of steps of half a chunk
// (transformed rows 0, 1 and 2, 3, one LDS buffer each), software-pipelined as in the fp32 kernel.
#include <type_traits>

#include "pd_winograd.hpp"

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int H3_CC = 16;                              // input channels per chunk = depth of one MFMA
constexpr int H3_FRAG = 1024;                          // bytes of a fragment: 64 lanes x 8 f16
constexpr int H3_U_CHUNK = 16 * 2 * 2 * H3_FRAG;       // transformed filter: [position][k half][term][lane][8]
constexpr int H3_SLOT = 8 * 2 * 2 * H3_FRAG;           // V of half a chunk: [position][term][tile half][c half][tile][8]
constexpr int H3_RAW_MAX = 2 * WG_HALO * 2 * 12 * 32;  // halo tile: [c half][row][column parity][column / 2][8] floats
constexpr int H3_PITCH = 68;                           // floats between two tiles of the staged sums
constexpr int H3_STAGE = 4 * 2 * 32 * H3_PITCH * 4;    // [position column][row][tile][channel], 32 tiles at a time
// LDS map (bytes)
constexpr int H3_RAW_OFF = H3_SLOT;
constexpr int H3_SLOT1_OFF = H3_RAW_OFF + H3_RAW_MAX;  // (the staged sums begin here too: slot 1 is free by then)
constexpr int H3_ZERO_OFF = H3_SLOT1_OFF + (H3_STAGE > H3_SLOT ? H3_STAGE : H3_SLOT);
constexpr int H3_EXP_OFF = H3_ZERO_OFF + 512;          // [parity of the chunk][tile]
constexpr int H3_FLAG_OFF = H3_EXP_OFF + 2 * 64 * 4;
constexpr int H3_ITEM_OFF = H3_FLAG_OFF + 16;          // the next work items, decoded
constexpr int H3_ITEMS = 16;
constexpr int H3_WIDE_OFF = H3_ITEM_OFF + H3_ITEMS * 48;   // a bit per block of 64 output channels: not for f16
constexpr int H3_MAX_K_BLOCKS = 1024;
constexpr int H3_LDS = H3_WIDE_OFF + H3_MAX_K_BLOCKS / 8;
static_assert(H3_LDS <= 160 * 1024, "LDS budget of one CU");

// Scales as biased exponents: a field e (of the largest value) stands for the factor 2^(H3_X_BASE - e) on the input and
// 2^(H3_W_BASE - e) on the filter, so that the largest value becomes 2^11 to 2^12 and 2^13 to 2^14.
constexpr int H3_X_BASE = 138, H3_W_BASE = 140;
constexpr int H3_MIN_FIELD = 11;                       // (the factor must stay finite; denormals are still held exactly)
constexpr int H3_MAX_FIELD = 190;                      // (below what an infinity has in any channel)
constexpr int H3_SLACK = 1;                            // how far a tile's values may exceed its scale
constexpr int H3_INNER = 8;                            // how far its inner pixels may stay below it
constexpr int H3_MIN_SHIFT = -60;                      // range of s(c); a channel without weights has this too
static_assert(255 + H3_MIN_SHIFT > H3_MAX_FIELD && H3_X_BASE - H3_MAX_FIELD + H3_MIN_SHIFT > -127, "fields");
__device__ __forceinline__ float h3_scale(int field, int base) {
    return __builtin_bit_cast(float, (uint32_t)(base + 127 - field) << 23);
}

// What the filter's buffer holds behind the fragments (byte offsets from its start).
struct H3Layout {
    size_t fields;      // [k_pad] int: R(k)
    size_t shifts;      // [C] int: s(c)
    size_t exps;        // [k_pad][C] bytes: e(k, c)
    size_t part;        // [C / 16][k_pad] int: max of e over a slice of c (one slice where c is the innermost index of w)
    size_t wide;        // [k_blocks][2 C / 16] int: not 0 where 32 output x 16 input channels lie as fp32, see below
    size_t bytes;
    __host__ __device__ H3Layout(int K, int C) {
        const size_t k_blocks = (K + WG_BN - 1) / WG_BN, k_pad = k_blocks * WG_BN, chunks = C / H3_CC;
        fields = k_blocks * chunks * H3_U_CHUNK;
        shifts = fields + k_pad * 4;
        exps = shifts + (size_t)C * 4;
        part = exps + k_pad * C;
        wide = part + chunks * k_pad * 4;
        bytes = wide + k_blocks * chunks * 8;
    }
};

// e(k, c) and its maxima over c.  0: all nine taps are zero (or NaN); denormals count as the smallest normal numbers.
// (lanes: threads per output channel where the input channels are the innermost index of w, 64, 128 or 256: as many as
// there are input channels to read, so that a thread waits for memory once.  A wave for all 512 took 7 us, 256 threads 4)
__global__ __launch_bounds__(256) void winograd_exps_kernel(const float* __restrict__ w, char* __restrict__ u, int K, int C,
                                                            int k_pad, int rot180, int lanes) {
    __shared__ int red[256];
    const H3Layout at(K, C);
    uint8_t* const exps = (uint8_t*)(u + at.exps);
    int* const part = (int*)(u + at.part);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto exponent = [](float m) { return m > 0.f ? max((int)(__builtin_bit_cast(uint32_t, m) >> 23), 1) : 0; };
    if (!rot180) {
        const int k = blockIdx.x * (256 / lanes) + threadIdx.x / lanes;
        int top = 0;
        if (k < K) {
            const float* row = w + (size_t)k * 9 * C;
#pragma unroll 2
            for (int c = threadIdx.x % lanes; c < C; c += lanes) {
                float m = 0.f;
#pragma unroll
                for (int t = 0; t < 9; ++t) m = fmaxf(m, fabsf(row[(size_t)t * C + c]));
                const int e = exponent(m);
                exps[(size_t)k * C + c] = (uint8_t)e;
                top = max(top, e);
            }
        }
#pragma unroll
        for (int d = 32; d; d >>= 1) top = max(top, __shfl_xor(top, d));
        if (lane == 0) red[wave] = top;
        __syncthreads();
        if (threadIdx.x % lanes == 0 && k < k_pad) {
            for (int i = 1; i < lanes / 64; ++i) top = max(top, red[wave + i]);
            part[k] = top;
        }
        return;
    }
    // lanes along the output channels, 16 input channels per block
    const int k = blockIdx.x * 64 + lane, slice = blockIdx.y;
    int top = 0;
    if (k < K) {
        uint32_t packed = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float m = 0.f;
#pragma unroll
            for (int t = 0; t < 9; ++t) m = fmaxf(m, fabsf(w[((size_t)(slice * H3_CC + wave * 4 + i) * 9 + t) * K + k]));
            const int e = exponent(m);
            packed |= (uint32_t)e << (8 * i);
            top = max(top, e);
        }
        *(uint32_t*)(exps + (size_t)k * C + slice * H3_CC + wave * 4) = packed;
    }
    red[threadIdx.x] = top;
    __syncthreads();
    if (wave == 0 && k < k_pad)
        part[(size_t)slice * k_pad + k] = max(max(red[lane], red[64 + lane]), max(red[128 + lane], red[192 + lane]));
}

// U = G g G^T, scaled and split, in the order in which a wave consumes it:
// [k / 64][c / 16][position][(k % 64) / 32][term][(c % 16) / 8][k % 32][c % 8].  Rows k >= K are zero.  A block makes
// 32 output x 16 input channels; a thread transforms one output channel and two consecutive input channels, four
// neighbouring threads share a lane's 16 bytes.  If the block holds a kernel that two terms do not hold (head of this
// file; P is `range`), its U goes out in fp32, unscaled: the first four of a lane's eight channels in place of the first
// terms, the others in place of the second ones.
__global__ __launch_bounds__(256) void winograd_filter_f16x3_kernel(const float* __restrict__ w, char* __restrict__ u,
                                                                    int slices, int K, int C, int k_pad, int rot180,
                                                                    int range) {
    __shared__ uint32_t s_part[4][H3_CC / 2];
    const H3Layout at(K, C);
    const uint8_t* const exps = (const uint8_t*)(u + at.exps);
    const int* const part = (const int*)(u + at.part);
    const int n_chunks = C / H3_CC;
    const int kb = blockIdx.y, chunk = blockIdx.x >> 1, kh = blockIdx.x & 1;
    const int tid = threadIdx.x;
    // the fast thread index runs along the contiguous index of w: input channels, or (rot180) output channels
    const int cp = rot180 ? tid >> 5 : tid & 7, k32 = rot180 ? tid & 31 : tid >> 3;
    const int k = kb * WG_BN + kh * 32 + k32, c0 = chunk * H3_CC + cp * 2;

    // (everything is requested before anything is waited for: taps, exponents and maxima of up to 512 output channels)
    float g[3][3][2];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int s = 0; s < 3; ++s)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                g[r][s][e] = k >= K ? 0.f : rot180 ? w[((size_t)(c0 + e) * 9 + (2 - r) * 3 + (2 - s)) * K + k]
                                                   : w[((size_t)k * 9 + r * 3 + s) * C + c0 + e];
    const uint32_t own2 = k < K ? *(const uint16_t*)(exps + (size_t)k * C + c0) : 0;
    // s(c) of the block's 16 channels over all k: a thread takes whole rows of them, 255 + e - R as 16 bits, 0 for no weights
    typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
    u16x2_t best[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) best[i] = u16x2_t{0, 0};
    int top = 0;
    for (int sl = 0; sl < slices; sl += 8) {
        int v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = part[(size_t)min(sl + q, slices - 1) * k_pad + k];
#pragma unroll
        for (int q = 0; q < 8; ++q) top = max(top, v[q]);
    }
    for (int k0 = 0; k0 < K; k0 += 512) {
        u32x4_t e[2];
        int row_top[2] = {0, 0};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int kk = k0 + 256 * h + tid;
            e[h] = kk < K ? *(const u32x4_t*)(exps + (size_t)kk * C + chunk * H3_CC) : u32x4_t{0, 0, 0, 0};
        }
        // (rows past the filter read the last one's maximum beside exponents of zero)
        const int* const p0 = part + min(k0 + tid, k_pad - 1);
        const int* const p1 = part + min(k0 + 256 + tid, k_pad - 1);
        for (int sl = 0; sl < slices; sl += 8) {
            int v[8][2];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const size_t at_slice = (size_t)min(sl + q, slices - 1) * k_pad;
                v[q][0] = p0[at_slice];
                v[q][1] = p1[at_slice];
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                row_top[0] = max(row_top[0], v[q][0]);
                row_top[1] = max(row_top[1], v[q][1]);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t pair = e[h][i / 2] >> (16 * (i % 2));
                const int lo = pair & 255, hi = pair >> 8 & 255;
                const u16x2_t v = {(uint16_t)(lo ? 255 + lo - row_top[h] : 0), (uint16_t)(hi ? 255 + hi - row_top[h] : 0)};
                best[i] = __builtin_elementwise_max(best[i], v);
            }
    }
#pragma unroll
    for (int d = 32; d; d >>= 1)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            best[i] = __builtin_elementwise_max(
                best[i], __builtin_bit_cast(u16x2_t, __shfl_xor(__builtin_bit_cast(int, best[i]), d)));
    if ((tid & 63) == 0)
#pragma unroll
        for (int i = 0; i < 8; ++i) s_part[tid >> 6][i] = __builtin_bit_cast(uint32_t, best[i]);
    __syncthreads();
    constexpr int NONE = -1000;
    int shift[2];
    bool wide = top == 255;                                        // infinities
    const int field = top ? top : 127;                             // (a row of zeros)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const auto of = [&](int i) { return (int)(s_part[i][cp] >> (16 * e) & 0xffffu); };
        const int v = max(max(of(0), of(1)), max(of(2), of(3))), s = v ? v - 255 : NONE;
        wide |= s != NONE && s < H3_MIN_SHIFT;
        shift[e] = max(s, H3_MIN_SHIFT);
        wide |= field + shift[e] < 13;                             // (the factor must stay finite)
        if (top && s != NONE) {
            const int own = own2 >> (8 * e) & 255;
            wide |= own == 0 || own - top - s < -range;
        }
    }
    if (chunk == 0 && cp == 0) ((int*)(u + at.fields))[k] = field;
    if (kb == 0 && kh == 0 && k32 == 0) {
        ((int*)(u + at.shifts))[c0] = shift[0];
        ((int*)(u + at.shifts))[c0 + 1] = shift[1];
    }
    wide = __syncthreads_or(wide);
    if (tid == 0) ((int*)(u + at.wide))[(kb * n_chunks + chunk) * 2 + kh] = wide;
    const float scale[2] = {wide ? 1.f : h3_scale(field + shift[0], H3_W_BASE),
                            wide ? 1.f : h3_scale(field + shift[1], H3_W_BASE)};
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int s = 0; s < 3; ++s)
#pragma unroll
            for (int e = 0; e < 2; ++e) g[r][s][e] *= scale[e];
    float t[4][3][2];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            t[0][s][e] = g[0][s][e];
            t[1][s][e] = 0.5f * (g[0][s][e] + g[1][s][e] + g[2][s][e]);
            t[2][s][e] = 0.5f * (g[0][s][e] - g[1][s][e] + g[2][s][e]);
            t[3][s][e] = g[2][s][e];
        }
    char* dst = u + (size_t)(kb * n_chunks + chunk) * H3_U_CHUNK + kh * (2 * H3_FRAG) + (cp >> 2) * 512 + k32 * 16 +
                (cp & 3) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
                o[e] = j == 0 ? t[i][0][e] : j == 3 ? t[i][2][e]
                              : 0.5f * (j == 1 ? t[i][0][e] + t[i][1][e] + t[i][2][e] : t[i][0][e] - t[i][1][e] + t[i][2][e]);
            if (wide) {
                char* to = u + (size_t)(kb * n_chunks + chunk) * H3_U_CHUNK + kh * (2 * H3_FRAG) + (cp >> 2) * 512 + k32 * 16 +
                           (size_t)(i * 4 + j) * (4 * H3_FRAG) + ((cp >> 1) & 1) * H3_FRAG + (cp & 1) * 8;
                *(float2_t*)to = float2_t{o[0], o[1]};
                continue;
            }
            const uint32_t p = wino_f16_pack(o[0], o[1]);
            float r0 = wino_f16_rest_lo(p, o[0]), r1 = wino_f16_rest_hi(p, o[1]);
            if ((p & 0x7c00u) == 0x7c00u) r0 = 0.f;                // infinities and NaNs stand in the first term alone
            if ((p & 0x7c000000u) == 0x7c000000u) r1 = 0.f;
            char* to = dst + (size_t)(i * 4 + j) * (4 * H3_FRAG);
            *(uint32_t*)to = p;
            *(uint32_t*)(to + H3_FRAG) = wino_f16_pack(r0, r1);
        }
}

// POOL, UNPOOL, STACKED, SEG: as in the fp32 kernel (a.u is the split filter, a.n_chunks counts chunks of 16).
// MASK: the input is taken as 0 where a.mask <= 0.  SPLIT: an item reduces over one of 2^split_log2 ranges of the input
// channels and stores its sums alone (no bias, ReLU, mask); winograd_split_sum_kernel does the rest.
template <bool POOL, bool UNPOOL, bool STACKED, int SEG, bool MASK = false, bool SPLIT = false>
__global__ __launch_bounds__(WG_THREADS, 1) void winograd_fwd_f16x3_kernel(const WinoArgs a) {
    static_assert((SEG == 1 || STACKED) && !(MASK && (STACKED || POOL || UNPOOL)) && !(SPLIT && (MASK || POOL || UNPOOL)),
                  "variants that exist");
    const auto block_of = [&](int kb) { return SPLIT ? kb >> a.split_log2 : kb; };            // of output channels
    const auto range_of = [&](int kb) { return SPLIT ? kb & ((1 << a.split_log2) - 1) : 0; };  // of input channels
    constexpr int SEGW = WG_PIX / SEG;
    constexpr int HALO_W = WG_PIX + 2 * SEG;
    constexpr int P = HALO_W / 2;                                  // columns of one parity
    constexpr int PIECES = WG_HALO * HALO_W * 4;                   // 16-byte pieces of a chunk's halo tile
    constexpr int NP = (PIECES + WG_THREADS - 1) / WG_THREADS;
    constexpr int RAW_HALF = WG_HALO * 2 * P * 32;                 // bytes of one channel half
    __shared__ __attribute__((aligned(1024))) char lds[H3_LDS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gx8 = gridDim.x / WG_XCD;
    const int xcd = blockIdx.x % WG_XCD, first = blockIdx.x / WG_XCD;
    const int item0 = xcd * a.items_per_xcd + first;
    int lim = a.n_items - xcd * a.items_per_xcd;
    lim = lim < a.items_per_xcd ? lim : a.items_per_xcd;
    const int n_my = first < lim ? (lim - first + gx8 - 1) / gx8 : 0;
    if (n_my == 0) return;                                         // whole block, before any barrier

    int* const exps = (int*)(lds + H3_EXP_OFF);
    int* const flag = (int*)(lds + H3_FLAG_OFF);
    uint32_t* const wide = (uint32_t*)(lds + H3_WIDE_OFF);
    const H3Layout at(a.K, a.C);
    const char* const u = (const char*)a.u;

    // ---- the block's items i .. i + H3_ITEMS - 1 lie decoded in a ring in LDS: the divisions are done by eight lanes for
    //      eight items at a time, instead of by everybody wherever an item begins.  Image, channel block, and first
    //      output row and column of every piece (no row where there is no piece).
    struct Item { int n, kb, pos[4][2], pad[2]; };
    static_assert(sizeof(Item) == 48, "ring of items");
    Item* const items = (Item*)(lds + H3_ITEM_OFF);
    auto decode_item = [&](int i) {
        Item it;
        const WinoItem w = wino_decode(a, item0 + i * gx8);
        it.n = w.n;
        it.kb = w.kb;
#pragma unroll
        for (int p = 0; p < SEG; ++p) {
            const SegPos sp = seg_pos<SEG>(a, item0 + i * gx8, p);
            it.pos[p][0] = sp.ok ? sp.y0 : 0x40000000;
            it.pos[p][1] = sp.x0;
        }
        items[i % H3_ITEMS] = it;
    };

    // ---- halo tile, global -> registers -> LDS: piece = (halo pixel, quarter of the 16 channels)
    const float* ximg = a.x;
    const float* mimg = MASK ? a.mask : a.x;
    const uint32_t img_bytes = (uint32_t)a.H * a.W * a.C * 4;
    uint32_t loff[NP], raw_dst[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        const int p = tid + WG_THREADS * j, pix = p >> 2, quarter = p & 3;
        const int row = pix / HALO_W, col = pix - row * HALO_W;
        raw_dst[j] = H3_RAW_OFF + (quarter >> 1) * RAW_HALF + ((row * 2 + (col & 1)) * P + (col >> 1)) * 32 + (quarter & 1) * 16;
    }
    auto set_load_item = [&](int i) {
        const Item* it = items + i % H3_ITEMS;
        if (i < n_my && SEG == 1) {
            const size_t img = (size_t)__builtin_amdgcn_readfirstlane(it->n) * a.H * a.W * a.C;
            ximg = a.x + img;
            if (MASK) mimg = a.mask + img;
        }
        const uint32_t range = SPLIT && i < n_my ? (uint32_t)(range_of(it->kb) * a.n_chunks) * (H3_CC * 4) : 0u;
        int t = tid;
        asm volatile("" : "+v"(t));            // (rows and columns are formed anew: kept, they would be spilled)
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int p = t + WG_THREADS * j, pix = p >> 2, quarter = p & 3;
            const int row = pix / HALO_W, col = pix - row * HALO_W;
            const int sg = SEG == 1 ? 0 : min(col / (SEGW + 2), SEG - 1);
            const int gy = it->pos[sg][0] - 1 + row, gx = it->pos[sg][1] - 1 + col - sg * (SEGW + 2);
            // out of the buffer: reads 0
            const bool in = i < n_my && gy >= 0 && gy < a.H && gx >= 0 && gx < a.W && p < PIECES;
            loff[j] = in ? (uint32_t)((gy * a.W + gx) * a.C) * 4 + quarter * 16 + range : 0x80000000u;
        }
    };
    float4_t rawr[NP], rawm[MASK ? NP : 1];
    auto load_raw = [&](int chunk) {
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)ximg, 0, img_bytes, 0x00020000);
#pragma unroll
        for (int j = 0; j < NP; ++j)
            rawr[j] = __builtin_bit_cast(float4_t,
                                         __builtin_amdgcn_raw_buffer_load_b128(xr, loff[j], chunk * (H3_CC * 4), 0));
        if (MASK) {
            const __amdgpu_buffer_rsrc_t mr = __builtin_amdgcn_make_buffer_rsrc((void*)mimg, 0, img_bytes, 0x00020000);
#pragma unroll
            for (int j = 0; j < NP; ++j)
                rawm[MASK ? j : 0] = __builtin_bit_cast(
                    float4_t, __builtin_amdgcn_raw_buffer_load_b128(mr, loff[j], chunk * (H3_CC * 4), 0));
        }
    };
    auto store_raw = [&]() {
        if (MASK) {
#pragma unroll
            for (int j = 0; j < NP; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) rawr[j][c] = rawm[MASK ? j : 0][c] > 0.f ? rawr[j][c] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < NP; ++j)
            if ((j + 1) * WG_THREADS <= PIECES || tid + WG_THREADS * j < PIECES) *(float4_t*)(lds + raw_dst[j]) = rawr[j];
    };
    int l_i = 0, l_cc = 0;
    auto advance_l = [&]() {
        if (++l_cc == a.n_chunks) { l_cc = 0; set_load_item(++l_i); }
    };

    // ---- input transform: tile tt (row `wave` of the 8 x 8 tiles, column (lane / 4) % 8), channels 8 (lane / 32) +
    //      2 (lane % 4) + 0, 1.  The eight lanes of a tile are neighbours or 32 apart.
    const int ch8 = lane >> 5, tx = (lane >> 2) & 7, tt = wave * 8 + tx;
    const int tseg = SEG == 1 ? 0 : tx / (8 / SEG);
    const int src_tile = H3_RAW_OFF + ch8 * RAW_HALF + (2 * wave * 2 * P + tx + tseg) * 32 + (lane & 3) * 8;
    const int zeros = H3_ZERO_OFF + (lane & 3) * 8;
    const int v_dst = (wave >> 2) * H3_FRAG + ch8 * 512 + ((wave & 3) * 8 + tx) * 16 + (lane & 3) * 4;
    const char* row0 = lds + src_tile;                             // patch rows 0 and 3: zeros at an image's edge
    const char* row3 = lds + src_tile + 3 * (2 * P * 32);
    auto set_patch_rows = [&](int i) {
        if (!STACKED || i >= n_my) return;
        const int r0 = items[i % H3_ITEMS].pos[tseg][0] + 2 * wave;
        row0 = lds + (r0 % a.img_h == 0 ? zeros : src_tile);
        row3 = lds + ((r0 + 2) % a.img_h == 0 ? zeros : src_tile + 3 * (2 * P * 32));
    };
    int p_i = 0, p_cc = 0;                                         // item and chunk of the next patch
    int p_range = 0;                                               // SPLIT: first chunk of its range
    auto set_patch_range = [&](int i) {
        if (SPLIT && i < n_my) p_range = __builtin_amdgcn_readfirstlane(range_of(items[i % H3_ITEMS].kb)) * a.n_chunks;
    };
    int field = H3_MIN_FIELD;                                      // scale of the tile
    int inner = 0;                                                 // field of its inner pixels, all chunks of the item
    int shift[2];                                                  // s(c) of the thread's two channels of the next patch
    auto load_shift = [&]() {
        typedef int int2_t __attribute__((ext_vector_type(2)));
        const int2_t v = *(const int2_t*)(u + at.shifts + (size_t)((p_range + p_cc) * H3_CC + ch8 * 8 + (lane & 3) * 2) * 4);
        shift[0] = v[0];
        shift[1] = v[1];
    };
    float2_t d[4][4];                                              // patch, then B^T d
    auto read_patch_row = [&](int r) {
        const char* src = r == 0 ? row0 : r == 3 ? row3 : lds + src_tile + r * (2 * P * 32);
#pragma unroll
        for (int s = 0; s < 4; ++s) d[r][s] = *(const float2_t*)(src + (s & 1) * (P * 32) + (s >> 1) * 32);
    };
    float pmax[2], imax[2];                                        // per channel: all of the patch, its inner pixels
    auto patch_max = [&](int e) {
        auto abs = [&](int r, int s) { return fabsf(d[r][s][e]); };
        float m;                                                   // (fmaxf of two would first quiet both)
        asm("v_max_f32 %0, |%1|, |%2|" : "=v"(m) : "v"(d[1][1][e]), "v"(d[1][2][e]));
        imax[e] = m = fmaxf(fmaxf(m, abs(2, 1)), abs(2, 2));
        m = fmaxf(fmaxf(m, abs(0, 0)), abs(0, 1));
        m = fmaxf(fmaxf(m, abs(0, 2)), abs(0, 3));
        m = fmaxf(fmaxf(m, abs(1, 0)), abs(1, 3));
        m = fmaxf(fmaxf(m, abs(2, 0)), abs(2, 3));
        m = fmaxf(fmaxf(m, abs(3, 0)), abs(3, 1));
        pmax[e] = fmaxf(fmaxf(m, abs(3, 2)), abs(3, 3));
    };
    auto tile_max = [&](int m) {                                   // over the tile's lanes
        m = max(m, __builtin_amdgcn_mov_dpp(m, 0xB1, 0xf, 0xf, true));
        m = max(m, __builtin_amdgcn_mov_dpp(m, 0x4E, 0xf, 0xf, true));
        // (the copy is made opaque: of a swap of one value with itself the compiler takes both results for the same)
        int copy = m;
        asm("" : "+v"(copy));
        const auto sw = __builtin_amdgcn_permlane32_swap((uint32_t)m, (uint32_t)copy, false, false);
        return max((int)sw[0], (int)sw[1]);
    };
    auto set_scale = [&](int parity) {
        auto exponent = [](float m) { return (int)(__builtin_bit_cast(uint32_t, m) >> 23); };
        const int f = tile_max(max(exponent(pmax[0]) + shift[0], exponent(pmax[1]) + shift[1]));
        const int here = max(exponent(imax[0]) + shift[0], exponent(imax[1]) + shift[1]);
        // (a new work item starts anew: p_cc is uniform, these are scalars)
        const int forget = p_cc ? 0 : 1000, slack = p_cc ? H3_SLACK : 0;
        inner = max(inner - forget, here);
        const int before = max(field - forget, H3_MIN_FIELD);
        field = f > before + slack ? f : before;
        int to = v_dst;                                            // (tt formed anew: kept, it would be spilled)
        asm volatile("" : "+v"(to));
        if ((lane & 35) == 0) *(int*)(lds + H3_EXP_OFF + parity * 256 + (to >> 2) - (wave >> 2) * 128) = field;
    };
    auto look_inside = [&]() {                                     // the tile's inner pixels, all chunks of the item seen
        if (tile_max(inner) + H3_INNER < field && field > H3_MIN_FIELD) {
            const Item* it = items + (p_i - 1) % H3_ITEMS;         // (tiles beyond the image have none)
            if (it->pos[tseg][0] + 2 * wave < a.H && it->pos[tseg][1] + 2 * (tx - tseg * (8 / SEG)) < a.W) *flag = 1;
        }
    };
    auto transform_col = [&](int s) {                              // column s of the patch -> column s of B^T d, scaled
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float sc = h3_scale(field - shift[e], H3_X_BASE);
            const float s1 = d[1][s][e] * sc, s2 = d[2][s][e] * sc;
            const float t0 = fmaf(d[0][s][e], sc, -s2), t3 = fmaf(d[3][s][e], -sc, s1);
            d[0][s][e] = t0;
            d[1][s][e] = s1 + s2;
            d[2][s][e] = s2 - s1;
            d[3][s][e] = t3;
        }
    };
    auto write_v = [&](int row, int m) {                           // position (row, m), split, into the slot of its row
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
            v[e] = m == 0 ? d[row][0][e] - d[row][2][e] : m == 1 ? d[row][1][e] + d[row][2][e]
                 : m == 2 ? d[row][2][e] - d[row][1][e] : d[row][1][e] - d[row][3][e];
        const uint32_t p = wino_f16_pack(v[0], v[1]);
        const uint32_t q = wino_f16_pack(wino_f16_rest_lo(p, v[0]), wino_f16_rest_hi(p, v[1]));
        char* to = lds + (row < 2 ? 0 : H3_SLOT1_OFF) + ((row & 1) * 4 + m) * (4 * H3_FRAG) + v_dst;
        *(uint32_t*)to = p;
        *(uint32_t*)(to + 2 * H3_FRAG) = q;
    };

    // ---- MFMAs: position column j, channel half kh; 4 position rows x 2 tile halves
    const int j = wave & 3, kh = wave >> 2;
    const __amdgpu_buffer_rsrc_t ur =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.u, 0, (uint32_t)a.k_blocks * a.n_chunks * H3_U_CHUNK, 0x00020000);
    const uint32_t u_lane = (uint32_t)(j * (4 * H3_FRAG) + kh * (2 * H3_FRAG) + lane * 16);
    half8_t uf[2][2];                                              // [row of the step][term]
    int u_i = 0, u_cc = 0, u_kb = item0 % a.k_blocks;
    auto load_u = [&](int row) {
        const int base = (u_kb * a.n_chunks + u_cc) * H3_U_CHUNK + row * (16 * H3_FRAG);
#pragma unroll
        for (int t = 0; t < 2; ++t)
            uf[row & 1][t] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(ur, u_lane + t * H3_FRAG, base, 0));
    };
    auto advance_u = [&]() {                                       // stays on the last chunk once the sequence ends
        if (u_cc + 1 < a.n_chunks) ++u_cc;
        else if (u_i + 1 < n_my) { u_cc = 0; u_kb = __builtin_amdgcn_readfirstlane(items[++u_i % H3_ITEMS].kb); }
    };
    half8_t vf[2][2];                                              // fragments of two sections, [section & 1][term]
    auto read_v = [&](int slot, int section) {                     // section = (row of the step, tile half)
        const char* src = lds + (slot ? H3_SLOT1_OFF : 0) + ((section >> 1) * 4 + j) * (4 * H3_FRAG) +
                          (section & 1) * H3_FRAG + lane * 16;
        vf[section & 1][0] = *(const half8_t*)src;
        vf[section & 1][1] = *(const half8_t*)(src + 2 * H3_FRAG);
    };
    float16_t acc[4][2];
    int cur[2];                                                    // fields of the scales the sums are held at

    // ---- output: a thread's tile of an item, channels k .. k + 3
    struct Out {
        int y, x;                              // first pixel
        bool ok;                               // the tile's piece and the channels exist
        int n;                                 // image
        size_t img;                            // its first element [.., K]
        uint32_t off;                          // element offset of the first pixel in it
        uint32_t mbits;                        // output mask, four bits a pixel
        uint32_t iw[UNPOOL ? 4 : 1];
    };
    typedef int int4_t __attribute__((ext_vector_type(4)));
    const int* const k_fields = (const int*)(u + at.fields);
    const uint32_t out_elems = (uint32_t)a.H * a.W * a.K;
    float4_t b4;                               // of the channels: bias (past K, or without one, 0), scales
    int4_t kf;
    auto load_channels = [&](int k) {
        const __amdgpu_buffer_rsrc_t br =
            __builtin_amdgcn_make_buffer_rsrc((void*)a.bias, 0, a.bias ? (uint32_t)a.K * 4 : 0u, 0x00020000);
        b4 = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(br, (uint32_t)k * 4, 0, 0));
        kf = *(const int4_t*)(k_fields + k);
    };
    // requests what else the stores need besides the sums: output mask or index bytes
    auto prepare_out = [&](Out& o, int i, int k, int tile) {
        const int col = tile & 7, sg = SEG == 1 ? 0 : col / (8 / SEG);
        const Item* it = items + i % H3_ITEMS;
        o.y = it->pos[sg][0] + 2 * (tile >> 3);
        o.x = it->pos[sg][1] + 2 * (col - sg * (8 / SEG));
        o.ok = o.y < a.H && o.x < a.W && k < a.K;
        o.n = SEG == 1 ? __builtin_amdgcn_readfirstlane(it->n) : 0;
        o.img = (size_t)o.n * a.H * a.W * a.K;
        if (SPLIT) o.img += __builtin_amdgcn_readfirstlane(range_of(it->kb)) * a.part_elems;
        o.off = (uint32_t)((o.y * a.W + o.x) * a.K + k);
        if (UNPOOL) {
            const __amdgpu_buffer_rsrc_t ir =
                __builtin_amdgcn_make_buffer_rsrc((void*)(a.unpool_idx + o.img), 0, out_elems, 0x00020000);
#pragma unroll
            for (int px = 0; px < 4; ++px) {
                const bool in = o.ok && o.y + (px >> 1) < a.H && o.x + (px & 1) < a.W;
                o.iw[UNPOOL ? px : 0] = __builtin_amdgcn_raw_buffer_load_b32(
                    ir, in ? o.off + ((px >> 1) * a.W + (px & 1)) * a.K : 0x80000000u, 0, 2);
            }
        } else if (!POOL && a.out_mask) {
            const __amdgpu_buffer_rsrc_t mr =
                __builtin_amdgcn_make_buffer_rsrc((void*)(a.out_mask + o.img), 0, out_elems * 4, 0x00020000);
            float4_t mk[4];
#pragma unroll
            for (int px = 0; px < 4; ++px) {
                const bool in = o.ok && o.y + (px >> 1) < a.H && o.x + (px & 1) < a.W;
                mk[px] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                    mr, in ? (o.off + ((px >> 1) * a.W + (px & 1)) * a.K) * 4 : 0x80000000u, 0, 2));
            }
            o.mbits = 0;
#pragma unroll
            for (int px = 0; px < 4; ++px)
#pragma unroll
                for (int c = 0; c < 4; ++c) o.mbits |= (mk[px][c] > 0.f ? 1u : 0u) << (4 * px + c);
        }
    };
    // bias, ReLU, mask / pooling / unpooling of the tile's pixels (row-major) and the stores; what lies outside the
    // image gets an offset beyond the buffer's size, with which a store is dropped
    auto finish = [&](const Out& o, int k, float4_t (&v)[4]) {
#pragma unroll
        for (int px = 0; px < 4; ++px) v[px] += b4;
        if (a.relu) {
#pragma unroll
            for (int px = 0; px < 4; ++px)
#pragma unroll
                for (int c = 0; c < 4; ++c) v[px][c] = v[px][c] > 0.f ? v[px][c] : 0.f;
        }
        if constexpr (POOL) {
            // index byte: bits 0-1 = position of the first maximum (row-major), bit 2 = "maximum > 0"
            const int Hp = a.H >> 1, Wp = a.W >> 1;
            const size_t pimg = o.n * (size_t)Hp * Wp * a.K;
            const uint32_t elems = (uint32_t)Hp * Wp * a.K;
            const bool in = o.ok && (o.y >> 1) < Hp && (o.x >> 1) < Wp;
            const uint32_t off = (uint32_t)(((o.y >> 1) * Wp + (o.x >> 1)) * a.K + k);
            float4_t best;
            uint32_t packed = 0;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float b = v[0][c];
                uint32_t arg = 0;
#pragma unroll
                for (int px = 1; px < 4; ++px) {
                    const bool take = v[px][c] > b || v[px][c] != v[px][c];
                    b = take ? v[px][c] : b;
                    arg = take ? (uint32_t)px : arg;
                }
                best[c] = b;
                packed |= (arg | (b > 0.f ? 4u : 0u)) << (8 * c);
            }
            const __amdgpu_buffer_rsrc_t pyr =
                __builtin_amdgcn_make_buffer_rsrc((void*)(a.pool_y + pimg), 0, elems * 4, 0x00020000);
            const __amdgpu_buffer_rsrc_t pir =
                __builtin_amdgcn_make_buffer_rsrc((void*)(a.pool_idx + pimg), 0, elems, 0x00020000);
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, best), pyr, in ? off * 4 : 0x80000000u, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(packed, pir, in ? off : 0x80000000u, 0, 0);
        } else {
            const __amdgpu_buffer_rsrc_t yr =
                __builtin_amdgcn_make_buffer_rsrc((void*)(a.y + o.img), 0, out_elems * 4, 0x00020000);
            const __amdgpu_buffer_rsrc_t fr = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(a.unpool_y + (UNPOOL ? 4 * o.img : 0)), 0, UNPOOL ? out_elems * 16 : 0, 0x00020000);
#pragma unroll
            for (int px = 0; px < 4; ++px) {
                const bool in = o.ok && o.y + (px >> 1) < a.H && o.x + (px & 1) < a.W;
                const uint32_t at = o.off + ((px >> 1) * a.W + (px & 1)) * a.K;
                float4_t w = v[px];
                if constexpr (UNPOOL) {
                    // y with the mask of bit 2, and the four positions of the window in front of the pooling: the
                    // value where the byte says 4 | position
                    const uint32_t fat = (uint32_t)((2 * (o.y + (px >> 1)) * 2 * a.W + 2 * (o.x + (px & 1))) * a.K + k);
                    uint32_t code[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) code[c] = (o.iw[UNPOOL ? px : 0] >> (8 * c)) & 7u;
#pragma unroll
                    for (int pos = 0; pos < 4; ++pos) {
                        float4_t f;
#pragma unroll
                        for (int c = 0; c < 4; ++c) f[c] = code[c] == (4u | pos) ? w[c] : 0.f;
                        __builtin_amdgcn_raw_buffer_store_b128(
                            __builtin_bit_cast(u32x4_t, f), fr,
                            in ? (fat + ((pos >> 1) * 2 * a.W + (pos & 1)) * a.K) * 4 : 0x80000000u, 0, 2);
                    }
#pragma unroll
                    for (int c = 0; c < 4; ++c) w[c] = (code[c] & 4u) ? w[c] : 0.f;
                } else if (a.out_mask) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) w[c] = (o.mbits >> (4 * px + c)) & 1u ? w[c] : 0.f;
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, w), yr, in ? at * 4 : 0x80000000u, 0, 2);
            }
        }
    };

    // (marks of filters that are not for f16: requested here, looked at behind the first item's loads)
    const int n_marks = a.k_blocks * a.n_chunks * 2;
    const int* const marks = (const int*)(u + at.wide);
    const int mark = tid < n_marks ? marks[tid] : 0;
    if (tid < H3_ITEMS && tid < n_my) decode_item(tid);
    if (tid < H3_MAX_K_BLOCKS / 32) wide[tid] = 0;
    if (tid < 128) ((float*)(lds + H3_ZERO_OFF))[tid] = 0.f;
    __syncthreads();
    auto advance_p = [&]() {
        if (++p_cc == a.n_chunks) {
            p_cc = 0;
            set_patch_rows(++p_i);
            set_patch_range(p_i);
        }
    };
    int q = 0;                                                     // chunk of the whole sequence
    // ---- start of the sequence, at item i: chunk 0 transformed (rows 0, 1 in slot 0, rows 2, 3 in registers), chunk 1 in
    //      LDS, chunk 2 requested
    auto prime = [&](int i) {
        l_i = i;
        l_cc = 0;
        set_load_item(i);
        load_raw(0);
        advance_l();
        u_i = i;
        u_cc = 0;
        u_kb = __builtin_amdgcn_readfirstlane(items[i % H3_ITEMS].kb);
        load_u(0);
        load_u(1);
        p_i = i;
        p_cc = 0;
        set_patch_range(i);
        load_shift();
        if (tid == 0) *flag = 0;
        store_raw();
        load_raw(l_cc);
        advance_l();
        set_patch_rows(i);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) read_patch_row(r);
        patch_max(0);
        patch_max(1);
        set_scale(q & 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) transform_col(s);
        __syncthreads();                                           // every patch is read
        store_raw();
        load_raw(l_cc);
        advance_l();
#pragma unroll
        for (int m = 0; m < 8; ++m) write_v(m >> 2, m & 3);
        advance_p();
        __syncthreads();
        read_v(0, 0);
    };

    auto clear = [&]() {                                           // (by MFMAs: eight instructions instead of 64)
        const half8_t none = {};
        const float16_t zero = {};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[r][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(none, none, zero, 0, 0, 0);
    };
    bool primed = false;
    int penalty = 1, wait = 0;                                     // items that stay on the fp32 MFMAs after one that had to
    auto note = [&](int i) {
        const int kb = i / (a.n_chunks * 2);
        atomicOr(&wide[kb >> 5], 1u << (kb & 31));
    };
    for (int m_i = 0; m_i < n_my; ++m_i) {
        const int kb = __builtin_amdgcn_readfirstlane(items[m_i % H3_ITEMS].kb);
        bool plain = wait > 0 || (m_i > 0 && __builtin_amdgcn_readfirstlane(wide[kb >> 5]) >> (kb & 31) & 1);
        if (wait > 0) --wait;
        if (!plain && !primed) {
            prime(m_i);
            primed = true;
            if (m_i == 0) {
                if (mark) note(tid);
                for (int i = tid + WG_THREADS; i < n_marks; i += WG_THREADS)
                    if (marks[i]) note(i);
                __syncthreads();
                plain = __builtin_amdgcn_readfirstlane(wide[kb >> 5]) >> (kb & 31) & 1;
            }
        }
        if (!plain) {
        clear();
#pragma unroll
        for (int t = 0; t < 2; ++t) cur[t] = exps[(q & 1) * 64 + t * 32 + (lane & 31)];
        plain = __any(max(cur[0], cur[1]) > H3_MAX_FIELD);         // (all 64 tiles: the same in every wave)
        for (int m_cc = 0; m_cc < a.n_chunks; ++m_cc, ++q) {
            // the tiles' scales of this chunk: sums held at another scale are brought to it
            {
                int now[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) now[t] = exps[(q & 1) * 64 + t * 32 + (lane & 31)];
                if (__any(now[0] != cur[0] || now[1] != cur[1])) {
                    plain |= __any(max(now[0], now[1]) > H3_MAX_FIELD) != 0;
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const float f = h3_scale(max(min(now[t] - cur[t] + 127, 254), 0) , 127);   // 2^(cur - now)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int e = 0; e < 16; ++e) acc[r][t][e] *= f;
                        cur[t] = now[t];
                    }
                }
            }
            if (p_cc == 0) look_inside();
            // Two steps of four sections (position row, tile half) of three MFMAs.  Every MFMA is followed by a piece of
            // the other work, which the scheduler may not move across.  The barrier of a step sits before its last
            // section: by then what the next step reads is in LDS, and that section's operands are in registers.
            //   step 0: rows 2, 3 of this chunk's V -> slot 1; the next chunk's patch -> registers
            //   step 1: its scale, B^T d, rows 0, 1 of its V -> slot 0; the chunk after it -> LDS, one more requested
            auto step = [&](auto step_c) {
                constexpr int S = decltype(step_c)::value;
#pragma unroll
                for (int k = 0; k < 12; ++k) {
                    const int section = k / 3, rr = section >> 1, t = section & 1, row = 2 * S + rr, cb = section & 1;
                    const int prod = k % 3;
                    acc[row][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(uf[rr][prod == 0], vf[cb][prod == 1], acc[row][t], 0, 0, 0);
                    if (prod == 0 && section < 3) read_v(S, section + 1);
                    if (S == 0) {
                        if (k < 8) write_v(2 + (k >> 2), k & 3);
                        if (k < 2) read_patch_row(k);                   // (into rows of B^T d that are used up)
                        if (k == 2) load_shift();
                        if (k == 4) read_patch_row(2);
                        if (k == 7) read_patch_row(3);
                    } else {
                        if (k == 0) { set_scale((q + 1) & 1); store_raw(); transform_col(0); }
                        if (k == 1) { transform_col(1); transform_col(2); load_raw(l_cc); }
                        if (k == 2) { transform_col(3); write_v(0, 0); }
                        if (k > 2 && k < 8) write_v((k - 2) >> 2, (k - 2) & 3);
                        if (k == 8) { write_v(1, 2); write_v(1, 3); }
                    }
                    if (k == 8) {
                        __syncthreads();
                        read_v(S ^ 1, 0);
                    }
                    if (S == 0 && k >= 10) patch_max(k - 10);
                    if (k == 5) {                                  // (the first row's filter fragments: their last use was here)
                        if (S == 0) load_u(2);
                        else { advance_u(); load_u(0); }
                    }
                    if (k == 11) load_u(S == 0 ? 3 : 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            advance_l();
            advance_p();
        }
        plain |= __builtin_amdgcn_readfirstlane(*flag) != 0;       // (written before the last two barriers of the item)
        wait = plain ? penalty : 0;
        penalty = plain ? min(2 * penalty, 1 << 20) : 1;
        }
        if (plain) {
            // The item on the fp32 MFMAs, one chunk after the other: halo tile -> LDS, all of V in fp32 -> LDS
            // ([position][tile half][c half][tile][8]), products with the filter put together from its two terms or, where
            // these do not hold it, as it is.  128 -> 128 channels at 112 x 112, 64 images, every filter of that kind: 1.09 ms,
            // the fp32 kernel 0.88, the f16 MFMAs 0.55
            primed = false;
            clear();
            set_load_item(m_i);
            set_patch_rows(m_i);
            const int kfield = k_fields[block_of(kb) * WG_BN + kh * 32 + (lane & 31)];
            char* const v32 = lds + H3_SLOT1_OFF;
            u_kb = kb;
            u_cc = 0;
            load_raw(0);
            load_u(0);
            load_u(1);
#pragma unroll 1
            for (int cc = 0; cc < a.n_chunks; ++cc) {
                store_raw();
                __syncthreads();
                const bool as_is = marks[(kb * a.n_chunks + cc) * 2 + kh] != 0;
                const int4_t* const s8 = (const int4_t*)(u + at.shifts) + (range_of(kb) * a.n_chunks + cc) * 4 + (lane >> 5) * 2;
                const int4_t s_lo = s8[0], s_hi = s8[1];
                if (cc + 1 < a.n_chunks) load_raw(cc + 1);
#pragma unroll
                for (int r = 0; r < 4; ++r) read_patch_row(r);
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float d1 = d[1][s][e], d2 = d[2][s][e];
                        d[0][s][e] -= d2;
                        d[1][s][e] = d1 + d2;
                        d[2][s][e] = d2 - d1;
                        d[3][s][e] = d1 - d[3][s][e];
                    }
                char* to = v32 + (wave >> 2) * 2048 + ch8 * 1024 + ((wave & 3) * 8 + tx) * 32 + (lane & 3) * 8;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    *(float2_t*)(to + (4 * r) * 4096) = d[r][0] - d[r][2];
                    *(float2_t*)(to + (4 * r + 1) * 4096) = d[r][1] + d[r][2];
                    *(float2_t*)(to + (4 * r + 2) * 4096) = d[r][2] - d[r][1];
                    *(float2_t*)(to + (4 * r + 3) * 4096) = d[r][1] - d[r][3];
                }
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float w[8];
                    if (as_is) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) w[e] = __builtin_bit_cast(float4_t, uf[r & 1][e >> 2])[e & 3];
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            w[e] = __builtin_ldexpf((float)uf[r & 1][0][e] + (float)uf[r & 1][1][e],
                                                    kfield + (e < 4 ? s_lo[e & 3] : s_hi[e & 3]) - H3_W_BASE);
                    }
                    if (r >= 2 && cc + 1 < a.n_chunks) u_cc = cc + 1;
                    load_u(r ^ 2);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const float* src = (const float*)(v32 + (r * 4 + j) * 4096 + t * 2048 + (lane >> 5) * 1024 + (lane & 31) * 32);
                        const float4_t v0 = *(const float4_t*)src, v1 = *(const float4_t*)(src + 4);
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            acc[r][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[e], e < 4 ? v0[e & 3] : v1[e & 3], acc[r][t], 0, 0, 0);
                    }
                }
                // (the next chunk's halo tile is written behind this one's patch reads: the barrier above; its V behind
                // the next barrier, which every wave reaches after these fragment reads)
            }
            __syncthreads();
        }

        // ---- epilogue of item m_i, 32 tiles at a time: a lane folds its four rows of M to two (A^T M), the staged
        //      sums are [column of positions][row][tile][channel]; then a thread has a tile and four channels, adds up the
        //      columns and stores the tile's 2 x 2 pixels.
        const int k4 = block_of(kb) * WG_BN + (tid & 15) * 4;
        load_channels(k4);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float* st = (float*)(lds + H3_SLOT1_OFF) + ((j * 2) * 32 + (lane & 31)) * H3_PITCH + kh * 32 + 4 * (lane >> 5);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float4_t z0, z1;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float m[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) m[r] = acc[r][t][4 * g + e];
                    z0[e] = m[0] + m[1] + m[2];
                    z1[e] = m[1] - m[2] - m[3];
                }
                *(float4_t*)(st + 8 * g) = z0;
                *(float4_t*)(st + 32 * H3_PITCH + 8 * g) = z1;
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
            // (the output mask is kept as bits: its 16 values and what else is live here would spill 53 registers)
            Out o;
            prepare_out(o, m_i, k4, t * 32 + (tid >> 4));
            const int tf = exps[((q - 1) & 1) * 64 + t * 32 + (tid >> 4)];
            __syncthreads();
            const float* src = (const float*)(lds + H3_SLOT1_OFF) + (tid >> 4) * H3_PITCH + (tid & 15) * 4;
            float4_t y[4];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                float4_t z[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) z[c] = *(const float4_t*)(src + (c * 2 + s) * 32 * H3_PITCH);
                y[2 * s] = z[0] + z[1] + z[2];
                y[2 * s + 1] = z[1] - z[2] - z[3];
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int exponent = plain ? 0 : tf + kf[c] - (H3_X_BASE + H3_W_BASE);
#pragma unroll
                for (int px = 0; px < 4; ++px) y[px][c] = __builtin_ldexpf(y[px][c], exponent);
            }
            finish(o, k4, y);
            __syncthreads();
        }
        if (m_i % 8 == 7 && tid < 8 && m_i + 9 + tid < n_my) decode_item(m_i + 9 + tid);     // (in place of m_i - 7 + tid)
    }
}

// y = the sum of the ranges' results + bias, ReLU, output mask; or its 2 x 2 maxima and index bytes (as the epilogue above
// forms them).  A thread has four channels of a pixel or of a window.
struct SplitSumArgs {
    const float* part;
    const float* bias;
    const float* out_mask;
    float* y;
    float* pool_y;
    uint8_t* pool_idx;
    size_t part_elems;
    int N, H, W, K, splits, relu;
};
template <bool POOL>
__global__ __launch_bounds__(256) void winograd_split_sum_kernel(const SplitSumArgs a) {
    const int K4 = a.K / 4, Ho = POOL ? a.H / 2 : a.H, Wo = POOL ? a.W / 2 : a.W;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long)a.N * Ho * Wo * K4) return;
    const int k = (int)(id % K4) * 4;
    const long pix = id / K4;
    const int x = (int)(pix % Wo), y = (int)(pix / Wo % Ho);
    const long n = pix / ((long)Wo * Ho);
    constexpr int PX = POOL ? 4 : 1;
    size_t at[PX];
    float4_t v[PX];
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        at[p] = POOL ? ((size_t)(n * a.H + 2 * y + (p >> 1)) * a.W + 2 * x + (p & 1)) * a.K + k : (size_t)pix * a.K + k;
        v[p] = *(const float4_t*)(a.part + at[p]);
    }
    for (int s = 1; s < a.splits; s += 3) {            // (2^n - 1 more of them, three in flight)
        float4_t q[3][PX];
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
            for (int p = 0; p < PX; ++p) q[u][p] = *(const float4_t*)(a.part + min(s + u, a.splits - 1) * a.part_elems + at[p]);
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (s + u < a.splits)
#pragma unroll
                for (int p = 0; p < PX; ++p) v[p] += q[u][p];
    }
    if (a.bias) {
#pragma unroll
        for (int p = 0; p < PX; ++p)
#pragma unroll
            for (int c = 0; c < 4; ++c) v[p][c] += a.bias[k + c];
    }
    if (a.relu) {
#pragma unroll
        for (int p = 0; p < PX; ++p)
#pragma unroll
            for (int c = 0; c < 4; ++c) v[p][c] = v[p][c] > 0.f ? v[p][c] : 0.f;
    }
    if constexpr (POOL) {
        float4_t best;
        uint32_t packed = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float b = v[0][c];
            uint32_t arg = 0;
#pragma unroll
            for (int p = 1; p < 4; ++p) {
                const bool take = v[p][c] > b || v[p][c] != v[p][c];
                b = take ? v[p][c] : b;
                arg = take ? (uint32_t)p : arg;
            }
            best[c] = b;
            packed |= (arg | (b > 0.f ? 4u : 0u)) << (8 * c);
        }
        *(float4_t*)(a.pool_y + (size_t)pix * a.K + k) = best;
        *(uint32_t*)(a.pool_idx + (size_t)pix * a.K + k) = packed;
    } else {
        if (a.out_mask) {
            const float4_t m = *(const float4_t*)(a.out_mask + at[0]);
#pragma unroll
            for (int c = 0; c < 4; ++c) v[0][c] = m[c] > 0.f ? v[0][c] : 0.f;
        }
        *(float4_t*)(a.y + at[0]) = v[0];
    }
}

}  // namespace

namespace {

int h3_shape(const char* who, int C, int K) {
    PD_REQUIRE(C > 0 && K > 0 && C % H3_CC == 0 && K % 4 == 0, PD_ESHAPE, "%s: needs C %% 16 == 0 and K %% 4 == 0 (C=%d K=%d)",
               who, C, K);
    PD_REQUIRE(pd_conv3x3_winograd_f16x3_supported(C, K), PD_ESHAPE, "%s: too many channels (C=%d K=%d)", who, C, K);
    return PD_OK;
}

// P of the head of this file
int h3_range(int C) {
    int bits = 0;
    while (1 << bits < C) ++bits;
    return 13 - (bits + 1) / 2;
}

// Into how many ranges of the input channels a launch's reduction is cut (1: it is not).  An item of 64 channels is
// 28 000 cycles and every 16 more 4100, so a launch of few items with many channels leaves most CUs idle for long.  A cut
// writes and reads the result once per range and costs a launch: from four chunks a range on, and while every item still
// finds a CU.  us for 512 -> 512 channels with the filter's launches, uncut / cut: 8 images of 14 x 14 78 / 49 (4 ranges),
// 1 image 77 / 35 (8), 4 images of 28 x 28 78 / 62 (2); 256 -> 256, 1 image of 56 x 56 50 / 35 (4).  With 128 input
// channels there is nothing left to gain (1 image of 112 x 112 33 / 34).
int h3_splits(const WinoArgs& a) {
    int splits = 1;
    if (a.n_chunks < 16) return 1;
    while (2 * splits * (long)a.n_items <= 256 && a.n_chunks % (2 * splits) == 0 && a.n_chunks / (2 * splits) >= 4 &&
           2 * splits * a.k_blocks <= H3_MAX_K_BLOCKS)
        splits *= 2;
    return splits;
}

template <bool STACKED, int SEG>
void h3_launch(const WinoArgs& a, dim3 grid, hipStream_t s) {
    if (a.unpool_y) winograd_fwd_f16x3_kernel<false, true, STACKED, SEG><<<grid, WG_THREADS, 0, s>>>(a);
    else if (a.pool_y) winograd_fwd_f16x3_kernel<true, false, STACKED, SEG><<<grid, WG_THREADS, 0, s>>>(a);
    else winograd_fwd_f16x3_kernel<false, false, STACKED, SEG><<<grid, WG_THREADS, 0, s>>>(a);
}

}  // namespace

extern "C" int pd_conv3x3_winograd_f16x3_supported(int C, int K) {
    return C > 0 && K > 0 && C % H3_CC == 0 && K % 4 == 0 &&
           (long)((K + WG_BN - 1) / WG_BN) * (C / H3_CC) * H3_U_CHUNK < (1L << 31) &&
           (K + WG_BN - 1) / WG_BN <= H3_MAX_K_BLOCKS;
}

extern "C" int pd_conv3x3_winograd_f16x3_filter_bytes(int C, int K, uint64_t* bytes) {
    const char* who = "pd_conv3x3_winograd_f16x3_filter_bytes";
    PD_REQUIRE(bytes != nullptr, PD_EINVAL, "%s: NULL pointer", who);
    if (int rc = h3_shape(who, C, K)) return rc;
    *bytes = H3Layout(K, C).bytes;
    return PD_OK;
}

extern "C" int pd_conv3x3_winograd_f16x3_filter_f32(const float* w, void* u, int C, int K, int rot180, void* stream) {
    const char* who = "pd_conv3x3_winograd_f16x3_filter_f32";
    PD_REQUIRE(w && u && (const void*)w != u, PD_EINVAL, "%s: NULL or aliased pointer", who);
    if (int rc = h3_shape(who, C, K)) return rc;
    PD_REQUIRE(pd_aligned(u, 16), PD_EINVAL, "%s: u must be 16-byte aligned", who);
    const int k_blocks = (K + WG_BN - 1) / WG_BN, k_pad = k_blocks * WG_BN, n_chunks = C / H3_CC;
    const int slices = rot180 ? n_chunks : 1;
    hipStream_t s = (hipStream_t)stream;
    const int lanes = C >= 256 ? 256 : C >= 128 ? 128 : 64;
    const dim3 grid = rot180 ? dim3(k_blocks, n_chunks) : dim3(k_pad / (256 / lanes));
    winograd_exps_kernel<<<grid, 256, 0, s>>>(w, (char*)u, K, C, k_pad, rot180, lanes);
    PD_CHECK_LAUNCH(who);
    winograd_filter_f16x3_kernel<<<dim3(n_chunks * 2, k_blocks), 256, 0, s>>>(w, (char*)u, slices, K, C, k_pad, rot180,
                                                                              h3_range(C));
    PD_CHECK_LAUNCH(who);
    return PD_OK;
}

extern "C" int pd_conv3x3_winograd_f16x3_fwd_nhwc_f32(const float* x, const void* u, const float* bias,
                                                      const float* in_mask, const float* out_mask, float* y, float* y_pool, uint8_t* pool_idx,
                                                      const uint8_t* unpool_idx, float* y_full, int N, int H, int W,
                                                      int C, int K, int relu, void* stream) {
    const char* who = "pd_conv3x3_winograd_f16x3_fwd_nhwc_f32";
    PD_REQUIRE(N > 0 && H > 0 && W > 0, PD_ESHAPE, "%s: dimensions must be positive", who);
    if (int rc = h3_shape(who, C, K)) return rc;
    PD_REQUIRE((long)H * W * (C > K ? C : K) < (1L << 29), PD_ESHAPE, "%s: image too large", who);
    PD_REQUIRE(x && u, PD_EINVAL, "%s: NULL pointer", who);
    if (y_pool) {
        PD_REQUIRE(pool_idx && !y && !y_full && !in_mask && !out_mask && !unpool_idx, PD_EINVAL,
                   "%s: a pooled output goes with its index bytes and nothing else", who);
        PD_REQUIRE(H >= 2 && W >= 2, PD_ESHAPE, "%s: the image must hold at least one 2x2 window", who);
    } else {
        PD_REQUIRE(y && !pool_idx, PD_EINVAL, "%s: NULL pointer", who);
        PD_REQUIRE(!y_full == !unpool_idx && !(y_full && (in_mask || out_mask || bias || relu)), PD_EINVAL,
                   "%s: a full-resolution output goes with the pooling's index bytes and no bias, ReLU or mask", who);
        PD_REQUIRE(!y_full || (long)H * W * K < (1L << 27), PD_ESHAPE, "%s: image too large for the full-resolution output", who);
    }
    PD_REQUIRE(pd_aligned(x, 16) && pd_aligned(u, 16) && pd_aligned(y, 16) && pd_aligned(in_mask, 16) &&
                   pd_aligned(out_mask, 16) && pd_aligned(y_pool, 16) && pd_aligned(y_full, 16) && pd_aligned(pool_idx, 4) && pd_aligned(unpool_idx, 4),
               PD_EINVAL, "%s: tensors must be 16-byte aligned, index bytes 4-byte aligned", who);
    WinoArgs a;
    a.x = x; a.u = (const float*)u; a.bias = bias; a.mask = in_mask; a.out_mask = out_mask; a.y = y;
    a.pool_y = y_pool; a.pool_idx = pool_idx; a.unpool_idx = unpool_idx; a.unpool_y = y_full;
    a.relu = relu != 0;
    WinoPlan plan;
    if (int rc = pd_wino_plan(who, a, N, H, W, C, K, H3_CC, !in_mask, &plan)) return rc;
    const dim3 grid(plan.blocks);
    hipStream_t s = (hipStream_t)stream;
    if (in_mask) winograd_fwd_f16x3_kernel<false, false, false, 1, true><<<grid, WG_THREADS, 0, s>>>(a);
    else if (plan.seg == 2) h3_launch<true, 2>(a, grid, s);
    else if (plan.seg == 4) h3_launch<true, 4>(a, grid, s);
    else if (plan.stacked) h3_launch<true, 1>(a, grid, s);
    else h3_launch<false, 1>(a, grid, s);
    PD_CHECK_LAUNCH(who);
    return PD_OK;
}

extern "C" int pd_conv3x3_winograd_f16x3_split_bytes(int N, int H, int W, int C, int K, uint64_t* bytes) {
    const char* who = "pd_conv3x3_winograd_f16x3_split_bytes";
    PD_REQUIRE(bytes && N > 0 && H > 0 && W > 0, PD_EINVAL, "%s: NULL pointer or empty tensor", who);
    if (int rc = h3_shape(who, C, K)) return rc;
    PD_REQUIRE((long)H * W * (C > K ? C : K) < (1L << 29), PD_ESHAPE, "%s: image too large", who);
    WinoArgs a;
    a.unpool_y = nullptr;
    WinoPlan plan;
    if (int rc = pd_wino_plan(who, a, N, H, W, C, K, H3_CC, true, &plan)) return rc;
    const int splits = h3_splits(a);
    *bytes = splits > 1 ? (uint64_t)splits * N * H * W * K * sizeof(float) : 0;
    return PD_OK;
}

extern "C" int pd_conv3x3_winograd_f16x3_fwd_split_nhwc_f32(const float* x, const void* u, const float* bias,
                                                            const float* out_mask, float* y, float* y_pool, uint8_t* pool_idx,
                                                            void* partials, uint64_t partials_bytes, int N, int H, int W,
                                                            int C, int K, int relu, void* stream) {
    const char* who = "pd_conv3x3_winograd_f16x3_fwd_split_nhwc_f32";
    uint64_t need = 0;
    if (int rc = pd_conv3x3_winograd_f16x3_split_bytes(N, H, W, C, K, &need)) return rc;
    PD_REQUIRE(need > 0, PD_ESHAPE, "%s: the reduction of this shape is not split", who);
    PD_REQUIRE(x && u && partials && partials_bytes >= need, PD_EINVAL, "%s: NULL pointer or too few bytes", who);
    PD_REQUIRE(y_pool ? pool_idx && !y && !out_mask && H >= 2 && W >= 2 : y && !pool_idx, PD_EINVAL,
               "%s: y, or a pooled output with its index bytes", who);
    PD_REQUIRE(pd_aligned(x, 16) && pd_aligned(u, 16) && pd_aligned(y, 16) && pd_aligned(out_mask, 16) && pd_aligned(y_pool, 16) &&
                   pd_aligned(partials, 16) && pd_aligned(pool_idx, 4), PD_EINVAL,
               "%s: tensors must be 16-byte aligned, index bytes 4-byte aligned", who);
    WinoArgs a;
    a.x = x; a.u = (const float*)u; a.bias = nullptr; a.mask = nullptr; a.out_mask = nullptr; a.y = (float*)partials;
    a.pool_y = nullptr; a.pool_idx = nullptr; a.unpool_idx = nullptr; a.unpool_y = nullptr;
    a.relu = 0;
    WinoPlan plan;
    if (int rc = pd_wino_plan(who, a, N, H, W, C, K, H3_CC, true, &plan)) return rc;
    SplitSumArgs f;
    f.splits = h3_splits(a);
    a.split_log2 = __builtin_ctz((unsigned)f.splits);
    a.part_elems = (size_t)N * H * W * K;
    a.k_blocks *= f.splits;
    a.n_chunks /= f.splits;
    a.n_items *= f.splits;                             // (at most 256: a block each)
    a.items_per_xcd = (a.n_items + WG_XCD - 1) / WG_XCD;
    const dim3 grid((unsigned)a.items_per_xcd * WG_XCD);
    hipStream_t s = (hipStream_t)stream;
    if (plan.seg == 2) winograd_fwd_f16x3_kernel<false, false, true, 2, false, true><<<grid, WG_THREADS, 0, s>>>(a);
    else if (plan.seg == 4) winograd_fwd_f16x3_kernel<false, false, true, 4, false, true><<<grid, WG_THREADS, 0, s>>>(a);
    else if (plan.stacked) winograd_fwd_f16x3_kernel<false, false, true, 1, false, true><<<grid, WG_THREADS, 0, s>>>(a);
    else winograd_fwd_f16x3_kernel<false, false, false, 1, false, true><<<grid, WG_THREADS, 0, s>>>(a);
    PD_CHECK_LAUNCH(who);
    f.part = (const float*)partials;
    f.bias = bias; f.out_mask = out_mask; f.y = y; f.pool_y = y_pool; f.pool_idx = pool_idx;
    f.part_elems = a.part_elems;
    f.N = N; f.H = H; f.W = W; f.K = K; f.relu = relu != 0;
    const long threads = y_pool ? (long)N * (H / 2) * (W / 2) * (K / 4) : (long)N * H * W * (K / 4);
    const dim3 sum_grid((unsigned)((threads + 255) / 256));
    if (y_pool) winograd_split_sum_kernel<true><<<sum_grid, 256, 0, s>>>(f);
    else winograd_split_sum_kernel<false><<<sum_grid, 256, 0, s>>>(f);
    PD_CHECK_LAUNCH(who);
    return PD_OK;
}
