// Weight gradient of the Winograd F(2x2, 3x3) convolution on the f16 matrix pipes: the sums
//   dU[g][k][c] = sum over tiles of  dM[g][tile][k] V[g][tile][c],   dM = A dY A^T,  V = B^T d B
// of pd_conv3x3_winograd.hip's weight gradient (which see, also for the kernels that add up the blocks' partial sums and
// apply G^T . G), with fp32 operands, fp32 accumulation and fp32 accuracy: both operands scaled by powers of two and
// split into two f16 terms, three products each, as in pd_conv3x3_winograd_f16x3.hip.
//
// The reduction runs over tiles, so a scale must hold for all tiles of a block's range: one for x, one for dY, from the
// largest value met so far, which becomes 2^10 to 2^11 (|V|, |dM| at most four times that; f16 ends at 2^16).  A larger
// value raises the scale when it is more than four times the last one that did, and all sums are multiplied accordingly;
// what lies below 2^-24 of f16's unit is less than 2^-34 of that largest value.  Infinities are reported in a.failed, and the
// fp32 kernel does the launch again.
//
// Bound: f16 MFMAs beside vector instructions and LDS traffic: a step takes 7000 cycles, of which 1700 are MFMAs and
// about 1500 the issue of its loads; the fp32 kernel takes 12000 for the same tiles.  64 images, C = K = 128 at 112 x 112:
// 975 -> 620 us with the two kernels behind it (382 TFLOP/s of a direct weight gradient).  A step of a block covers 16 tiles (eight units of two
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
constexpr int W3_MAX_OFF = 2 * W3_SLOT;                // largest exponent fields met, of x and dY
constexpr int W3_LDS = W3_MAX_OFF + 16;
static_assert(W3_LDS <= 160 * 1024, "LDS budget of one CU");
constexpr int W3_BASE = 137;                           // field e scales by 2^(137 - e)
constexpr int W3_MIN_FIELD = 16;
constexpr int W3_SLACK = 2;

__device__ __forceinline__ float w3_scale(int field) {
    return __builtin_bit_cast(float, (uint32_t)(W3_BASE + 127 - field) << 23);
}
__device__ __forceinline__ uint32_t w3_pack(float lo, float hi) {
    uint32_t p;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(p) : "v"(lo), "v"(hi));
    return p;
}
// x - (the lower / upper half of p), exactly
__device__ __forceinline__ float w3_rest_lo(uint32_t p, float x) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(p), "v"(x));
    return r;
}
__device__ __forceinline__ float w3_rest_hi(uint32_t p, float x) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(p), "v"(x));
    return r;
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
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int gy = u_y - 1 + r;
            xrow[r] = live && gy >= 0 && gy < a.H ? (uint32_t)((pix + (r - 1) * a.W) * a.C + c0 + ch) * 4 : ROW_OUT;
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
            yrow[r] = live && u_y + r < a.H ? (uint32_t)((pix + r * a.W) * a.K + k0 + ch) * 4 : ROW_OUT;
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

    // ---- scales: what exceeds the present one is noted in LDS, a barrier before it is used
    int* const top = (int*)(lds + W3_MAX_OFF);
    int fx = W3_MIN_FIELD, fy = W3_MIN_FIELD;
    auto check = [&]() {
        float mx = 0.f, my = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int s = 0; s < 6; s += 2) mx = fmaxf(fmaxf(mx, fabsf(lx[r][s])), fabsf(lx[r][s + 1]));
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int s = 0; s < 4; s += 2) my = fmaxf(fmaxf(my, fabsf(ly[r][s])), fabsf(ly[r][s + 1]));
        const int ex = (int)(__builtin_bit_cast(uint32_t, mx) >> 23), ey = (int)(__builtin_bit_cast(uint32_t, my) >> 23);
        if (__any(ex > fx + W3_SLACK || ey > fy + W3_SLACK)) {
            atomicMax(&top[0], ex);
            atomicMax(&top[1], ey);
        }
    };
    auto set_scales = [&]() {
        const int tx = __builtin_amdgcn_readfirstlane(top[0]), ty = __builtin_amdgcn_readfirstlane(top[1]);
        if (tx > fx + W3_SLACK) fx = tx;
        if (ty > fy + W3_SLACK) fy = ty;
    };

    // Odd ranks sum up -dU.  The f16 MFMA rounds its sums towards minus infinity, and half an ulp of the same sign in each
    // of 600 additions and 256 blocks adds up where G^T . G only adds (tap 0, 0: an error of 6.9e-6 of the gradient over
    // 64 images of 224 x 224, against 2.0e-6 of the fp32 kernel).
    const float sign = rank & 1 ? -1.f : 1.f;

    // ---- transforms.  v: rows of B^T d of the two tiles (six columns); m: the columns of A dY (rows d0, d0 + d1,
    //      d0 - d1, d1; the signs of A's last row and column are left to the kernel behind this one)
    float v[4][6], m[2][4];
    float db = 0.f;
    auto take = [&]() {                                // the loaded values, scaled: rows 0 .. 3 of B^T d
        const float sx = w3_scale(fx), sy = sign * w3_scale(fy);
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            const float s1 = lx[1][s] * sx, s2 = lx[2][s] * sx;
            v[0][s] = fmaf(lx[0][s], sx, -s2);
            v[1][s] = s1 + s2;
            v[2][s] = s2 - s1;
            v[3][s] = fmaf(lx[3][s], -sx, s1);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            db += ly[0][s] + ly[1][s];
            m[0][s] = ly[0][s] * sy;
            m[1][s] = ly[1][s] * sy;
        }
    };
    const int dst = (wave & 2) * 512 + (wave >> 2) * 512 + ((wave & 1) * 16 + (lane & 15)) * 16 + (lane >> 4) * 4;
    auto put = [&](char* to, float v0, float v1) {
        const uint32_t p = w3_pack(v0, v1);
        *(uint32_t*)to = p;
        *(uint32_t*)(to + 2048) = w3_pack(w3_rest_lo(p, v0), w3_rest_hi(p, v1));
    };
    auto write_v = [&](int row, int pos) {             // position (row, pos) of both tiles
        float o[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const float* w = &v[row][2 * t];
            o[t] = pos == 0 ? w[0] - w[2] : pos == 1 ? w[1] + w[2] : pos == 2 ? w[2] - w[1] : w[1] - w[3];
        }
        put(lds + (row >> 1) * W3_SLOT + ((row & 1) * 4 + pos) * W3_POS + dst, o[0], o[1]);
    };
    auto write_m = [&](int row, int pos) {
        float o[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float e[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const float d0 = m[0][2 * t + s], d1 = m[1][2 * t + s];
                e[s] = row == 0 ? d0 : row == 1 ? d0 + d1 : row == 2 ? d0 - d1 : d1;
            }
            o[t] = pos == 0 ? e[0] : pos == 1 ? e[0] + e[1] : pos == 2 ? e[0] - e[1] : e[1];
        }
        put(lds + (row >> 1) * W3_SLOT + ((row & 1) * 4 + pos) * W3_POS + 4096 + dst, o[0], o[1]);
    };

    // ---- MFMAs: position `wave` of each half of a step, 64 k x 64 c
    half8_t fa[2][2], fb[2][2];                        // [channel half][term]
    auto read_a = [&](int half, int h) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
            fa[h][t] = *(const half8_t*)(lds + half * W3_SLOT + wave * W3_POS + 4096 + t * 2048 + h * 1024 + lane * 16);
    };
    auto read_b = [&](int half, int h) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
            fb[h][t] = *(const half8_t*)(lds + half * W3_SLOT + wave * W3_POS + t * 2048 + h * 1024 + lane * 16);
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
    if (tid < 2) top[tid] = 0;
    load();
    __syncthreads();
    check();
    __syncthreads();
    set_scales();
    take();
    load();
    __syncthreads();                                   // (the noted maxima are read)
#pragma unroll
    for (int p = 0; p < 8; ++p) { write_v(p >> 2, p & 3); write_m(p >> 2, p & 3); }
    __syncthreads();
    read_a(0, 0);
    read_b(0, 0);

    int held = fx + fy;                                // the scale the sums are held at
    for (int q = 0; q < n_steps; ++q) {
        if (fx + fy != held) {
            const float f = __builtin_bit_cast(float, (uint32_t)max(127 - (fx + fy - held), 0) << 23);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[s][i][j][e] *= f;
            held = fx + fy;
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
                    if (k == 0) { set_scales(); take(); }
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
    const int idx = lane & 31, h = lane >> 5, shift = held - 2 * W3_BASE;
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
                    part[(size_t)(el >> 8) * chunk_pitch + (el & 255)] = __builtin_ldexpf(sign * acc[s][i][j][e], shift);
                }
    db += __shfl_xor(db, 16);
    db += __shfl_xor(db, 32);
    if (lane < 16) a.part_db[((size_t)(pair * a.ranks + rank) * 2 + (wave >> 2)) * 64 + ch] = db;
    if (tid == 0) a.failed[blockIdx.x] = fx == 255 || fy == 255;
}

}  // namespace

void pd_wino_wgrad_f16x3(const WinoWgradArgs& a, hipStream_t s) {
    winograd_wgrad_f16x3_kernel<<<WW_BLOCKS, WW_THREADS, 0, s>>>(a);
}
