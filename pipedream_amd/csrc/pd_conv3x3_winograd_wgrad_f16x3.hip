// Weight gradient of the Winograd F(2x2, 3x3) convolution on the f16 matrix pipes: the sums
//   dU[g][k][c] = sum over tiles of  dM[g][tile][k] V[g][tile][c],   dM = A dY A^T,  V = B^T d B
// of pd_conv3x3_winograd.hip's weight gradient (which see, also for the kernels that add up the blocks' partial sums and
// apply G^T . G), with fp32 operands, fp32 accumulation and fp32 accuracy: both operands scaled by powers of two and
// split into two f16 terms, three products each, as in pd_conv3x3_winograd_f16x3.hip.
//
// The reduction runs over tiles, so a scale must hold for all tiles of a sum, but not for all channels: every channel of x
// and every channel of dY has its own, a power of two, put one binary order above the largest value of a step of 16 tiles,
// which becomes 2^10 to 2^11 (|V|, |dM| at most four times a value; f16 ends at 2^16).  It moves with a step whose largest
// value lies above it or below 2^-13 of it, and the sums of that channel are multiplied accordingly, so that a value is
// held to 2^-24.8 (rms) of the largest of its channel within a step.  What is far below that in the same step would lose
// bits: where, in any channel, a dY value is below 2^-23 of the scale or all nine x values under an output pixel are below
// 2^-19 of it, the step runs on fp32 MFMAs, and so does a step with infinities or with values 2^64 times those before.  A
// sum thus comes from values held to the rounding of fp32 against the largest of their channel in their own 16 tiles,
// whatever the other channels, images and pixels are like.  (Over 500 random shapes, masks and ranges an element's error
// stays below 1.9e-6 of the sum of its products' sizes, the fp32 kernel's below 0.5e-6: elements whose few products lie
// beside dY values 2^20 times as large in the same tiles, where x is zero.)
// (A step of VGG16: 12 to 28 % of the steps of a block look at their scales anew, 0.1 to 0.3 % run on fp32 MFMAs.)
//
// Bound: f16 MFMAs beside vector instructions and LDS traffic: a step takes 7500 cycles, of which 1700 are MFMAs and
// about 1500 the issue of its loads; the fp32 kernel takes 12000 for the same tiles.  64 images, C = K = 128 at 112 x 112:
// 975 -> 612 us with the two kernels behind it (387 TFLOP/s of a direct weight gradient; 572 with one scale per block).  A step of a block covers 16 tiles (eight units of two
// tiles side by side) x 64 k x 64 c x 16 positions: 24 MFMAs a wave; every operand value is formed once per block, from
// x and dY read straight from memory into the registers of the thread that transforms it (a unit and a channel: 24 values
// of x, 8 of dY, coalesced over 16 channels), a step ahead.  Two tiles of a channel make one 32-bit LDS write per term,
// in the order of the MFMA fragments (8 tiles of a channel are 16 bytes); a wave owns one position in each half of a
// step and reads its 64 k and 64 c, so that nothing is read from LDS twice.  Units are numbered along the
// rows of the batch, with no padding where 4 divides the width.
#include "pd_winograd.hpp"

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

constexpr int W3_POS = 8 * 1024;                       // bytes of a position: [V, dM][term][channel half][tile half][32][8]
constexpr int W3_SLOT = 8 * W3_POS;                    // half a step: 8 positions
constexpr int W3_FIELD_OFF = 2 * W3_SLOT;              // [2][128] scales of the channels of x and of dY
constexpr int W3_KEPT_OFF = W3_FIELD_OFF + 2 * 128 * 4;    // [128] ... while a step for fp32 has none
constexpr int W3_TOP_OFF = W3_KEPT_OFF + 128 * 4;      // [128] largest fields of a step
constexpr int W3_FLAG_OFF = W3_TOP_OFF + 128 * 4;      // a scale may not fit a step; the step is for fp32; a scale moves
constexpr int W3_DB_OFF = W3_FLAG_OFF + 16;            // [512] the threads' sums of dY
constexpr int W3_LDS = W3_DB_OFF + WW_THREADS * 4;
static_assert(W3_LDS <= 160 * 1024, "LDS budget of one CU");
constexpr int W3_BASE = 138;                           // field e scales by 2^(138 - e)
constexpr int W3_MIN_FIELD = 17;
constexpr int W3_HEADROOM = 1;                         // where a scale that moves is put above the step's largest value
constexpr int W3_JUMP = 64;                            // how far a scale may rise at once (the sums must not vanish)
constexpr int W3_SLACK = 1;                            // how far values may exceed their scale ..
constexpr int W3_FAINT = 13;                           // .. all values of a step may stay below it ..
constexpr int W3_X_RANGE = 19, W3_Y_RANGE = 23;        // .. the values under one output pixel, one dY value

__device__ __forceinline__ float w3_scale(int field) {
    return __builtin_bit_cast(float, (uint32_t)(W3_BASE + 127 - field) << 23);
}
__global__ __launch_bounds__(WW_THREADS, 1) void winograd_wgrad_f16x3_kernel(const WinoWgradArgs a) {
    __shared__ __attribute__((aligned(1024))) char lds[W3_LDS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int pair, rank;
    wino_wgrad_pair_rank(a, pair, rank);
    const int k0 = pair / a.c_blocks * 64, c0 = pair % a.c_blocks * 64;

    // units: (image, tile row, pair of tile columns), the last fastest
    const int tile_rows = (a.H + 1) / 2, pair_cols = (a.W + 3) / 4;
    const int per_img = tile_rows * pair_cols, units = a.N * per_img;
    const int all_steps = (units + 7) / 8, per_rank = (all_steps + a.ranks - 1) / a.ranks;
    const int q_begin = rank * per_rank, n_steps = max(0, min(per_rank, all_steps - q_begin));

    // ---- the thread's share of a step: unit 4 (wave / 4) + lane / 16, channel c0 / k0 + 16 (wave % 4) +
    //      lane % 16 (neighbouring lanes read neighbouring channels: with the units in neighbouring lanes the loads of a
    //      step took 6000 cycles to issue)
    const int ch = (wave & 3) * 16 + (lane & 15);
    int u_n, u_y, u_x;                                 // the unit that is loaded next: image, first pixel
    {
        const int u = q_begin * 8 + (wave >> 2) * 4 + (lane >> 4);
        u_n = u / per_img;
        const int rem = u - u_n * per_img, ty = rem / pair_cols;
        u_y = 2 * ty;
        u_x = 4 * (rem - ty * pair_cols);
    }
    int l_q = 0;                                       // its step
    const uint32_t xn = (uint32_t)((long)a.N * a.H * a.W * a.C * 4), dyn = (uint32_t)((long)a.N * a.H * a.W * a.K * 4);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, 0, xn, 0x00020000);
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc((void*)a.dy, 0, dyn, 0x00020000);
    float lx[4][6], ly[2][4];                          // patch and gradients, as loaded
    uint32_t xrow[4], yrow[2];                         // byte offsets of pixel (row, u_x)
    // Requested in eight parts.  What lies outside the image gets an offset of at least 2^30, beyond the tensors' size:
    // it reads 0.
    constexpr uint32_t ROW_OUT = 0x80000000u, COL_OUT = 0x40000000u;
    auto load_rows = [&]() {
        const bool live = l_q < n_steps && u_n < a.N;
        const int pix = (u_n * a.H + u_y) * a.W + u_x;
        const uint32_t x_pitch = (uint32_t)a.W * a.C * 4, y_pitch = (uint32_t)a.W * a.K * 4;
        int l;                                         // (the lane, formed anew: kept, it would be spilled)
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
        const int at = (wave & 3) * 16 + (l & 15);
        const uint32_t x0 = (uint32_t)(pix * a.C + c0 + at) * 4 - x_pitch, y0 = (uint32_t)(pix * a.K + k0 + at) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gy = u_y - 1 + r;
            xrow[r] = live && gy >= 0 && gy < a.H ? x0 + r * x_pitch : ROW_OUT;
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) yrow[r] = live && u_y + r < a.H ? y0 + r * y_pitch : ROW_OUT;
    };
    auto load_part = [&](int part) {
        if (part < 6) {
            const int s = part;
            const uint32_t col = u_x - 1 + s >= 0 && u_x - 1 + s < a.W ? (uint32_t)((s - 1) * a.C * 4) : COL_OUT;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                lx[r][s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, xrow[r] + col, 0, 0));
        } else {
#pragma unroll
            for (int s = 2 * (part - 6); s < 2 * (part - 6) + 2; ++s) {
                const uint32_t col = u_x + s < a.W ? (uint32_t)(s * a.K * 4) : COL_OUT;
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    ly[r][s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(yr, yrow[r] + col, 0, 0));
            }
        }
    };
    auto next_unit = [&]() {
        ++l_q;
        u_x += 32;
        while (u_x >= 4 * pair_cols) {
            u_x -= 4 * pair_cols;
            u_y += 2;
            if (u_y >= a.H) { u_y = 0; ++u_n; }
        }
    };
    auto load = [&]() {
        load_rows();
#pragma unroll
        for (int part = 0; part < 8; ++part) load_part(part);
        next_unit();
    };

    // ---- scales of the thread's two channels; what does not fit them is noted in LDS, a barrier before it matters.
    //      (They lie in LDS, and so do the sums of dY: in registers the loop would spill, and wait for its own requests.)
    int* const fields = (int*)(lds + W3_FIELD_OFF);
    int* const top = (int*)(lds + W3_TOP_OFF);
    int* const flags = (int*)(lds + W3_FLAG_OFF);
    int* const kept = (int*)(lds + W3_KEPT_OFF);
    int next = 0;                                      // which fields the step in the registers goes by
    bool moved = false, plain = false;                 // the sums are held at the other ones; the step is for fp32
    struct Range { int x, x_low, y, y_seen, y_low; };  // fields: largest; smallest but zero (255: all zero)
    auto range = [&]() {
        auto seen = [](float m) { return (__builtin_bit_cast(uint32_t, m) << 1) - 1; };   // (zeros become the largest)
        float a[2][6];                                 // largest of three rows, then of 3 x 3 pixels
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int s = 0; s < 6; ++s) a[r][s] = fmaxf(fmaxf(fabsf(lx[r][s]), fabsf(lx[r + 1][s])), fabsf(lx[r + 2][s]));
        float mx = 0.f, my = 0.f;
        uint32_t low_x = ~0u, low_y = ~0u;
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const float m = fmaxf(fmaxf(a[r][s], a[r][s + 1]), a[r][s + 2]);
                mx = fmaxf(mx, m);
                low_x = min(low_x, seen(m));
                my = fmaxf(my, fabsf(ly[r][s]));
                low_y = min(low_y, seen(ly[r][s]));
            }
        const uint32_t seen_y = seen(my);
        return Range{(int)(__builtin_bit_cast(uint32_t, mx) >> 23), (int)(low_x >> 24),
                     (int)(__builtin_bit_cast(uint32_t, my) >> 23), (int)(seen_y >> 24), (int)(low_y >> 24)};
    };
    auto check = [&]() {
        const Range r = range();
        const int fx = fields[next * 128 + ch], fy = fields[next * 128 + 64 + ch];
        if (r.x > fx + W3_SLACK || r.y > fy + W3_SLACK || r.x_low < fx - W3_FAINT || r.y_seen < fy - W3_FAINT ||
            r.y_low < fy - W3_Y_RANGE)
            flags[0] = 1;
    };
    // The step in the registers gets scales anew (`top` and the flags are zero before and after).
    auto new_scales = [&]() {
        const Range r = range();
        atomicMax(&top[ch], r.x);
        atomicMax(&top[64 + ch], r.y);
        __syncthreads();
        const int tx = top[ch], ty = top[64 + ch], fx0 = kept[ch], fy0 = kept[64 + ch];
        auto moved_to = [](int f, int t) {
            if (t == 255 || (t <= f + W3_SLACK && (t == 0 || t >= f - W3_FAINT))) return f;
            const int to = max(t + W3_HEADROOM, W3_MIN_FIELD);
            return f == W3_MIN_FIELD ? to : min(to, f + W3_JUMP);
        };
        const int fx = moved_to(fx0, tx), fy = moved_to(fy0, ty);
        if (r.x > fx + W3_SLACK || r.y > fy + W3_SLACK || r.x_low < fx - W3_X_RANGE || r.y_low < fy - W3_Y_RANGE) flags[1] = 1;
        if (fx != fx0 || fy != fy0) flags[2] = 1;
        __syncthreads();
        const bool was = plain;
        plain = __builtin_amdgcn_readfirstlane(flags[1]) != 0;
        moved = plain != was || (!plain && __builtin_amdgcn_readfirstlane(flags[2]) != 0);
        if (moved) next ^= 1;
        if (wave < 4 && lane < 16) {                   // (without a move these are the fields already there)
            fields[next * 128 + ch] = plain ? W3_BASE : fx;
            fields[next * 128 + 64 + ch] = plain ? W3_BASE : fy;
            kept[ch] = fx;
            kept[64 + ch] = fy;
        }
        if (tid < 128) top[tid] = 0;
        __syncthreads();
        if (tid < 3) flags[tid] = 0;                   // (next written behind another barrier)
    };
    auto set_scales = [&]() {
        if (plain || __builtin_amdgcn_readfirstlane(flags[0]) != 0) new_scales();
    };

    // Odd ranks sum up -dU.  The f16 MFMA rounds its sums towards minus infinity, and half an ulp of the same sign in each
    // of 600 additions and 256 blocks adds up where G^T . G only adds (tap 0, 0: an error of 6.9e-6 of the gradient over
    // 64 images of 224 x 224, against 2.0e-6 of the fp32 kernel).  A rank that is alone changes the sign every 32 steps
    // (1024 -> 1024 channels, 64 images of 14 x 14: mean error of tap 0, 0 4.4e-7 of the gradient's size without it).
    constexpr int TURN = 32;
    float sign = rank & 1 ? -1.f : 1.f;
    bool turned = false;                               // the step in the registers has the other sign than the sums

    // ---- transforms.  v: rows of B^T d of the two tiles (six columns); m: the columns of A dY (rows d0, d0 + d1,
    //      d0 - d1, d1; the signs of A's last row and column are left to the kernel behind this one)
    float v[4][6], m[2][4];
    float* const db = (float*)(lds + W3_DB_OFF) + tid;
    auto take = [&]() {                                // the loaded values, scaled: rows 0 .. 3 of B^T d
        const float sx = w3_scale(fields[next * 128 + ch]), sy = sign * w3_scale(fields[next * 128 + 64 + ch]);
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            const float s1 = lx[1][s] * sx, s2 = lx[2][s] * sx;
            v[0][s] = fmaf(lx[0][s], sx, -s2);
            v[1][s] = s1 + s2;
            v[2][s] = s2 - s1;
            v[3][s] = fmaf(lx[3][s], -sx, s1);
        }
        *db += ((ly[0][0] + ly[1][0]) + (ly[0][1] + ly[1][1])) + ((ly[0][2] + ly[1][2]) + (ly[0][3] + ly[1][3]));
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            m[0][s] = ly[0][s] * sy;
            m[1][s] = ly[1][s] * sy;
        }
    };
    const int dst = (wave & 2) * 512 + (wave >> 2) * 512 + ((wave & 1) * 16 + (lane & 15)) * 16 + (lane >> 4) * 4;
    // (an LDS instruction's offset ends at 2^16: a base of its own for each slot, opaque, else the compiler forms the
    // addresses anew, 45 additions a step)
    int dsts[2] = {dst, dst + W3_SLOT}, srcs[2] = {wave * W3_POS + lane * 16, W3_SLOT + wave * W3_POS + lane * 16};
#pragma unroll
    for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(dsts[i]), "+v"(srcs[i]));
    auto put = [&](int row, int pos, int op, float v0, float v1) {
        char* const to = lds + dsts[row >> 1] + ((row & 1) * 4 + pos) * W3_POS + op * 4096;
        const uint32_t p = wino_f16_pack(v0, v1);
        *(uint32_t*)to = p;
        *(uint32_t*)(to + 2048) = wino_f16_pack(wino_f16_rest_lo(p, v0), wino_f16_rest_hi(p, v1));
    };
    auto v_of = [&](int row, int pos, int t) {         // position (row, pos) of tile t
        const float* w = &v[row][2 * t];
        return pos == 0 ? w[0] - w[2] : pos == 1 ? w[1] + w[2] : pos == 2 ? w[2] - w[1] : w[1] - w[3];
    };
    auto m_of = [&](int row, int pos, int t) {
        float e[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float d0 = m[0][2 * t + s], d1 = m[1][2 * t + s];
            e[s] = row == 0 ? d0 : row == 1 ? d0 + d1 : row == 2 ? d0 - d1 : d1;
        }
        return pos == 0 ? e[0] : pos == 1 ? e[0] + e[1] : pos == 2 ? e[0] - e[1] : e[1];
    };
    auto write_v = [&](int row, int pos) {             // of both tiles
        put(row, pos, 0, v_of(row, pos, 0), v_of(row, pos, 1));
    };
    auto write_m = [&](int row, int pos) {
        put(row, pos, 1, m_of(row, pos, 0), m_of(row, pos, 1));
    };

    // ---- MFMAs: position `wave` of each half of a step, 64 k x 64 c
    half8_t fa[2][2], fb[2][2];                        // [channel half][term]
    auto read_a = [&](int half, int h) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
            fa[h][t] = *(const half8_t*)(lds + srcs[half] + 4096 + t * 2048 + h * 1024);
    };
    auto read_b = [&](int half, int h) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
            fb[h][t] = *(const half8_t*)(lds + srcs[half] + t * 2048 + h * 1024);
    };
    float16_t acc[2][2][2];                            // [half][k half][c half]
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[s][i][j][e] = 0.f;

    // ---- prologue: step 0 scaled, its first half in slot 0; step 1 requested
    if (tid < 128) top[tid] = 0;
    if (tid < 3) flags[tid] = 0;
    if (tid < 256) fields[tid] = W3_MIN_FIELD;
    if (tid < 128) kept[tid] = W3_MIN_FIELD;
    *db = 0.f;
    load();
    __syncthreads();
    new_scales();
    take();
    load();
#pragma unroll
    for (int p = 0; p < 8; ++p) { write_v(p >> 2, p & 3); write_m(p >> 2, p & 3); }
    __syncthreads();
    read_a(0, 0);
    read_b(0, 0);

    const int idx = lane & 31, h = lane >> 5;
    // the fields of the sums' channels k, four at a time, and c
    typedef int int4_t __attribute__((ext_vector_type(4)));
    auto k_field = [&](int which, int i, int g) { return *(const int4_t*)(fields + which * 128 + 64 + i * 32 + 8 * g + 4 * h); };
    auto c_field = [&](int which, int j) { return fields[which * 128 + j * 32 + idx]; };
    for (int q = 0; q < n_steps; ++q) {
        if (moved) {
            const int dc[2] = {c_field(next ^ 1, 0) - c_field(next, 0), c_field(next ^ 1, 1) - c_field(next, 1)};
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int4_t dk = k_field(next ^ 1, i, g) - k_field(next, i, g);
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                acc[s][i][j][4 * g + e] = __builtin_ldexpf(acc[s][i][j][4 * g + e], dk[e] + dc[j]);
                }
            moved = false;
        }
        if (turned) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[s][i][j][e] = -acc[s][i][j][e];
        }
        if (plain) {
            // fp32 MFMAs on the operands as they are, [position][V, dM][tile][channel] over both slots; the f16 MFMAs below
            // then have zeros to add (1.8 ms instead of 0.6 if every step is of this kind, the fp32
            // kernel 0.97)
            int at = ((wave >> 2) * 4 + (lane >> 4)) * 128 + ch, from = wave * 2048 + h * 64 + idx;
            asm volatile("" : "+v"(at), "+v"(from));   // (formed here: kept over the loop, their sums would be spilled)
            float* const f32 = (float*)lds;
#pragma unroll
            for (int row = 0; row < 4; ++row)
#pragma unroll
                for (int pos = 0; pos < 4; ++pos)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        f32[(row * 4 + pos) * 2048 + at + t * 64] = v_of(row, pos, t);
                        f32[(row * 4 + pos) * 2048 + 1024 + at + t * 64] = m_of(row, pos, t);
                    }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll 1
                for (int t = 0; t < 16; t += 2) {
                    const float* src = f32 + from + s * 16384 + t * 64;
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[s][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(src[1024 + i * 32], src[j * 32], acc[s][i][j], 0, 0, 0);
                }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < W3_SLOT / 16 / WW_THREADS; ++i)
                *(float4_t*)(lds + (i * WW_THREADS + tid) * 16) = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 6; ++s) v[2][s] = v[3][s] = 0.f;
#pragma unroll
            for (int s = 0; s < 4; ++s) m[0][s] = m[1][s] = 0.f;
            __syncthreads();
            read_a(0, 0);
            read_b(0, 0);
        }
        // Two halves (transformed rows 0, 1 and 2, 3) of four sections (k half, c half) of three MFMAs, every MFMA
        // followed by a piece of the other work, which the scheduler may not move across:
        //   half 0: rows 2, 3 of this step's operands -> slot 1; the next step's values (in registers by now) are looked over
        //   half 1: they are scaled and transformed, rows 0, 1 -> slot 0; the step after it is requested
        // The barrier of a half sits before its last section, whose operands are in registers by then.
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int k = 0; k < 12; ++k) {
                const int section = k / 3, i = section >> 1, j = section & 1, prod = k % 3;
                acc[half][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i][prod == 0], fb[j][prod == 1], acc[half][i][j], 0, 0, 0);
                if (k == 0) read_b(half, 1);
                if (k == 1) read_a(half, 1);
                if (half == 0) {
                    if (k < 8) { write_v(2 + (k >> 2), k & 3); write_m(2 + (k >> 2), k & 3); }
                    if (k == 8) check();
                } else {
                    if (k == 0) {
                        set_scales();
                        turned = a.ranks == 1 && (q + 1) % TURN == 0 && q + 1 < n_steps;
                        if (turned) sign = -sign;
                        take();
                    }
                    if (k == 1) load_rows();
                    if (k >= 1 && k < 9) load_part(k - 1);
                    if (k == 9) next_unit();
                    if (k >= 1 && k < 9) { write_v((k - 1) >> 2, (k - 1) & 3); write_m((k - 1) >> 2, (k - 1) & 3); }
                }
                if (k == 8) {
                    __syncthreads();
                    read_a(half ^ 1, 0);
                    // (fb[0] is free too: the last section takes fb[1])
                    read_b(half ^ 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    // ---- the block's sums, unscaled: partial dU in [g][k][c] order and partial dbias per (half of the units, k), laid out
    //      as the kernel that adds them up reads them (see the fp32 kernel)
    const int held = moved ? next ^ 1 : next;
    float* part = a.part + (size_t)pair * a.ranks * WW_PART_STRIDE + (size_t)rank * 256;
    const size_t chunk_pitch = (size_t)a.ranks * 256;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int k = i * 32 + 8 * (e / 4) + 4 * h + e % 4;
                    const int el = ((s * 8 + wave) * 64 + k) * 64 + j * 32 + idx;
                    const int shift = k_field(held, i, e / 4)[e % 4] + c_field(held, j) - 2 * W3_BASE;
                    part[(size_t)(el >> 8) * chunk_pitch + (el & 255)] = __builtin_ldexpf(sign * acc[s][i][j][e], shift);
                }
    float sum = *db;
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (lane < 16) a.part_db[((size_t)(pair * a.ranks + rank) * 2 + (wave >> 2)) * 64 + ch] = sum;
}

}  // namespace

void pd_wino_wgrad_f16x3(const WinoWgradArgs& a, hipStream_t s) {
    winograd_wgrad_f16x3_kernel<<<WW_BLOCKS, WW_THREADS, 0, s>>>(a);
}
