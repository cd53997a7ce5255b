// The time loop of an LSTM layer with its recurrent products on the bf16 matrix pipes at fp32 accuracy (pd_f32x6.hpp).
//
// Stands in for torch.nn.LSTM of the reference's translation stages
// (runtime/translation/models/gnmt_large/gpus=4/stage0.py:14-19) like pd_lstm.hip, whose fp32 MFMA products and cells
// remain for the shapes this file does not take.
//
// Forward: one launch per step.  A block owns 16 RT batch rows x 4 CT hidden units, i.e. all four gates of its units,
// over the whole reduction: the gate sums never leave the CU.  Its eight waves take an eighth of k each, with operands
// from L2 straight into registers (no LDS, no barrier in the loop); the eight partial sums meet in LDS, where one
// thread per (row, unit) adds them in wave order and applies the cell.  (The product split over k across blocks and a
// cell launch that adds the parts write and read 8 MB of partial sums a step.)
// Backward: dgates W_hh reduces over 4H, so a block per output tile would read four times as much: the product is
// split over k into partial sums (4 MB a step), which the next step's cell adds.
//
// Everything the products read lies in memory in the order in which lanes read it.  W_hh is laid out, and split into its
// terms, once per layer and direction (24 H^2 bytes; 7 us at H = 1024); a cell writes h (dgates) a second time in
// "tiles": 16 rows x 32 k, as two halves of four k per lane.  Rows of 4H floats fetched 16 at a time start in the same
// L2 channel: with h read row by row a forward step took 15.6 us where tiles gave 12.4.  A row tile is split just before
// its MFMAs (all of a chunk at once: 12.4, so 11.2 before the sums took turns in sign: the two waves of a SIMD then overlap
// one's conversions with the other's MFMAs).  fp32 weights split in the loop instead of the three terms: 11.5 us; sixteen
// waves a block: 11.6-12.8.
//
// Bound: reads from L2, 448 KB per CU and forward step at 128 x 1024, 26 bytes a cycle; MFMAs 2.6 us of it.
// us per time step in a chain of 20, before (fp32 MFMA product and cell) / now: forward at H = 1024 18.5 / 12.0 (batch 128),
// 14.3 / 8.1 (40), 12.8 / 5.8 (16), at H = 512 and batch 128 12.1 / 7.2; backward 18.9 / 15.0, 14.8 / 10.0, 12.8 / 7.5 and
// 12.1 / 8.6.  2-norm errors against 64 bits after 50 steps of 128 x 1024: h 1.1e-7 / 9.9e-8, bias gradient 1.6e-7 / 1.5e-7.
#include <type_traits>

#include "pd_f32x6.hpp"

namespace {

constexpr int LX_WAVES = 8;
constexpr int LX_THREADS = 64 * LX_WAVES;

using std::integral_constant;

// Offset in floats of (row, k) in an operand of `chunks` x 32 k laid out as tiles.
__device__ __forceinline__ size_t tile_offset(int row, int k, int chunks) {
    return ((size_t)(row / 16 * chunks + k / 32) * 2 + k % 8 / 4) * 256 + (k % 32 / 8 * 16 + row % 16) * 4 + k % 4;
}

// One wave's product: rows of `x` (tiles; 16 RT of them, from its first chunk on) with the split weights `w` (16 CT
// columns), n chunks of 32 k, summed up with `sign`.
template <int RT, int CT>
__device__ __forceinline__ void wave_product(f32x4_t (&acc)[RT][CT], const float* x, const u32x4_t* w, int chunks, int n,
                                             int lane, float sign) {
    f32x4_t raw[RT][2];
    u32x4_t wt[2][CT][3];
    auto load_x = [&](int i, int c) {
        raw[i][0] = *(const f32x4_t*)(x + ((size_t)i * chunks + c) * 512 + lane * 4);
        raw[i][1] = *(const f32x4_t*)(x + ((size_t)i * chunks + c) * 512 + 256 + lane * 4);
    };
    auto load_w = [&](auto buf, int c) {
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int p = 0; p < 3; ++p) wt[decltype(buf)::value][j][p] = w[((size_t)j * chunks + c) * 192 + p * 64 + lane];
    };
    auto step = [&](auto buf, int c) {
        constexpr int b = decltype(buf)::value;
        const int next = min(c + 1, n - 1);        // (past the end the last chunk is fetched again)
        load_w(integral_constant<int, b ^ 1>{}, next);
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const float v[8] = {raw[i][0][0], raw[i][0][1], raw[i][0][2], raw[i][0][3],
                                raw[i][1][0], raw[i][1][1], raw[i][1][2], raw[i][1][3]};
            u32x4_t xt[3];
            pd_x6_split8<true>(v, xt, sign);
            load_x(i, next);
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = pd_x6_mfma(xt[PD_X6_A[s]], wt[b][j][PD_X6_B[s]], acc[i][j]);
        }
    };
    load_w(integral_constant<int, 0>{}, 0);
#pragma unroll
    for (int i = 0; i < RT; ++i) load_x(i, 0);
    for (int c = 0; c < n; c += 2) {
        step(integral_constant<int, 0>{}, c);
        if (c + 1 < n) step(integral_constant<int, 1>{}, c + 1);
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] *= sign;
}

// Whether a sum is NaN or infinite.  Infinities and values that round to infinity in bf16 leave NaNs: the wave then
// repeats its product with fp32 MFMAs from the plain operands, which gives what fp32 gives.
template <int RT, int CT>
__device__ __forceinline__ bool not_finite(const f32x4_t (&acc)[RT][CT]) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) bad |= !(__builtin_fabsf(acc[i][j][e]) <= 3.4028235e38f);
    return __any(bad);
}

template <int RT, int CT>
__device__ __forceinline__ void clear(f32x4_t (&acc)[RT][CT]) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}

// W_hh [4H][H] -> [unit / 4][k / 32][term][lane][8 bf16]: lane (n = lane % 16, lane / 16) holds gate n / 4 of unit
// 4 (unit / 4) + n % 4 at k = 8 (lane / 16) .. + 7 of the chunk.
__global__ __launch_bounds__(256) void lstm_split_weights_kernel(const float* __restrict__ w, u32x4_t* __restrict__ out,
                                                                 int H) {
    const int chunks = H / 32;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long)(H / 4) * chunks * 64) return;
    const int lane = (int)(id % 64);
    const long tile = id / 64;                       // unit group * chunks + chunk
    const int group = (int)(tile / chunks), chunk = (int)(tile % chunks);
    const int n = lane % 16;
    const float* src = w + ((size_t)(n / 4) * H + 4 * group + n % 4) * H + chunk * 32 + 8 * (lane / 16);
    const f32x4_t lo = *(const f32x4_t*)src, hi = *(const f32x4_t*)(src + 4);
    const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    u32x4_t t[3];
    pd_x6_split8(x, t);
#pragma unroll
    for (int p = 0; p < 3; ++p) out[(tile * 3 + p) * 64 + lane] = t[p];
}

// The same of W_hh^T for the backward product: -> [unit / 16][k / 32][term][lane][8 bf16], k over the 4H gate rows: lane
// holds unit 16 (unit / 16) + lane % 16.
__global__ __launch_bounds__(256) void lstm_split_weights_t_kernel(const float* __restrict__ w, u32x4_t* __restrict__ out,
                                                                   int H) {
    const int chunks = 4 * H / 32;
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long)(H / 16) * chunks * 64) return;
    const int lane = (int)(id % 64);
    // (the chunk's row block of W first: the waves that run together read neighbouring columns of the same rows)
    const int units = H / 16, chunk = (int)(id / 64 / units), group = (int)(id / 64 % units);
    const float* src = w + (size_t)(chunk * 32 + 8 * (lane / 16)) * H + 16 * group + lane % 16;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = src[(size_t)e * H];
    u32x4_t t[3];
    pd_x6_split8(x, t);
#pragma unroll
    for (int p = 0; p < 3; ++p) out[(((size_t)group * chunks + chunk) * 3 + p) * 64 + lane] = t[p];
}

struct LstmStepArgs {
    float* gates;               // [B][4H]: x W_ih^T, becomes the activated gates
    const float* h_prev;        // [B][H], null at the first step (zero state)
    const float* h_in;          // the same in the order of the MFMA operands; read
    float* h_next;              // ... and written, for the next step
    const u32x4_t* w_split;
    const float* w;             // [4H][H]
    const float* b_ih;          // [4H] or null, both
    const float* b_hh;
    const float* c_prev;        // [B][H]
    float* c_out;
    float* h_out;
    int B, H;
    int row_blocks, items, items_per_die;
};

__device__ __forceinline__ float lx_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

template <int RT, int CT>
__global__ __launch_bounds__(LX_THREADS, 2) void lstm_step_f32x6_kernel(const LstmStepArgs a) {
    constexpr int ROWS = 16 * RT, UNITS = 4 * CT, COLS = 16 * CT, P = ROWS + 4;
    __shared__ __attribute__((aligned(16))) float part[LX_WAVES][COLS * P];

    // neighbouring units on one die: its L2 then holds an eighth of W_hh over the whole sequence, and the 32 bytes of
    // a row that a block writes complete lines there
    const int item = (blockIdx.x & 7) * a.items_per_die + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= a.items_per_die || item >= a.items) return;      // whole block
    const int group0 = item / a.row_blocks * CT, row0 = item % a.row_blocks * ROWS;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H;

    // the cell's operands are requested first and arrive beside the product
    const int u = tid % UNITS, row = tid / UNITS;
    const bool live = row < ROWS && row0 + row < a.B;
    const int unit = group0 * 4 + u;
    const size_t at = (size_t)(live ? row0 + row : 0) * H + unit;
    float* const g = a.gates + (size_t)(live ? row0 + row : 0) * 4 * H + unit;
    float pre[4], cp = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) pre[q] = 0.f;
    if (live) {
#pragma unroll
        for (int q = 0; q < 4; ++q) pre[q] = g[(size_t)q * H];
        if (a.h_prev) cp = a.c_prev[at];
    }

    f32x4_t acc[RT][CT];
    clear(acc);
    const int chunks = H / 32;
    const int c0 = chunks * wave / LX_WAVES, n = a.h_prev ? chunks * (wave + 1) / LX_WAVES - c0 : 0;
    if (n > 0) {
        wave_product(acc, a.h_in + ((size_t)row0 / 16 * chunks + c0) * 512, a.w_split + ((size_t)group0 * chunks + c0) * 192,
                     chunks, n, lane, pd_x6_sign(chunks, LX_WAVES, wave));
        if (not_finite(acc)) {
            clear(acc);
            const int idx = lane & 15;
            for (int k = c0 * 32 + (lane >> 4); k < (c0 + n) * 32; k += 4) {
                float wv[CT];
#pragma unroll
                for (int j = 0; j < CT; ++j) wv[j] = a.w[((size_t)(idx / 4) * H + 4 * (group0 + j) + idx % 4) * H + k];
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const float hv = a.h_prev[(size_t)min(row0 + 16 * i + idx, a.B - 1) * H + k];
#pragma unroll
                    for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(hv, wv[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    }

    // element e of lane l: row 4 (l / 16) + e, column l % 16 of its tile
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
            *(f32x4_t*)&part[wave][(16 * j + (lane & 15)) * P + 16 * i + 4 * (lane >> 4)] = acc[i][j];
    __syncthreads();
    if (row >= ROWS) return;
    float* const h_to = a.h_next + tile_offset(row0 + row, unit, chunks);
    if (!live) {                                   // rows of the last tile past the batch
        *h_to = 0.f;
        return;
    }
    const int col = (u / 4) * 16 + u % 4;          // column of gate 0; gate q lies 4 q further
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < LX_WAVES; ++w) s += part[w][(col + 4 * q) * P + row];
        // (four terms, rounded once)
        double z = (double)pre[q] + (double)s;
        if (a.b_ih) z += (double)a.b_ih[(size_t)q * H + unit] + (double)a.b_hh[(size_t)q * H + unit];
        pre[q] = (float)z;
    }
    const float gi = lx_sigmoid(pre[0]), gf = lx_sigmoid(pre[1]), gg = tanhf(pre[2]), go = lx_sigmoid(pre[3]);
    const float c = gf * cp + gi * gg;
    g[0] = gi;
    g[(size_t)H] = gf;
    g[2 * (size_t)H] = gg;
    g[3 * (size_t)H] = go;
    a.c_out[at] = c;
    const float h = go * tanhf(c);
    a.h_out[at] = h;
    *h_to = h;
}

// Backward of one step's cell (the arithmetic of lstm_cell_bwd_kernel in pd_lstm.hip): dgates as rows, which the weight
// gradients read, and as tiles.  A block takes 8 rows x 32 units: whole lines of the rows, and of the tiles.
__global__ __launch_bounds__(256) void lstm_cell_bwd_tiles_kernel(const float* __restrict__ gates,
                                                                  const float* __restrict__ c_prev,
                                                                  const float* __restrict__ c,
                                                                  const float* __restrict__ dy,
                                                                  const float* __restrict__ dh_rec, int n_rec,
                                                                  float* __restrict__ dc_io, float* __restrict__ dgates,
                                                                  float* __restrict__ tiles, int B, int H, int first_step) {
    const int b = blockIdx.y * 8 + threadIdx.x / 32, j = blockIdx.x * 32 + threadIdx.x % 32;
    const int chunks = 4 * H / 32;
    if (b >= B) {
#pragma unroll
        for (int q = 0; q < 4; ++q) tiles[tile_offset(b, q * H + j, chunks)] = 0.f;
        return;
    }
    const float* g = gates + (size_t)b * 4 * H + j;
    const float gi = g[0], gf = g[(size_t)H], gg = g[2 * (size_t)H], go = g[3 * (size_t)H];
    const size_t o = (size_t)b * H + j;
    const float cp = c_prev ? c_prev[o] : 0.f, ct = c[o];
    float dh = dy[o];
    const float dc_next = first_step ? 0.f : dc_io[o];
    if (!first_step) {
        for (int s0 = 0; s0 < n_rec; s0 += 8) {
            float p[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const bool live = s0 + u < n_rec;
                p[u] = dh_rec[(size_t)(live ? s0 + u : s0) * B * H + o];
                if (!live) p[u] = 0.f;
            }
            dh += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        }
    }
    const float tc = tanhf(ct);
    const float dck = dc_next + dh * go * (1.0f - tc * tc);
    const float d[4] = {dck * gg * gi * (1.0f - gi), dck * cp * gf * (1.0f - gf), dck * gi * (1.0f - gg * gg),
                        dh * tc * go * (1.0f - go)};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        dgates[(size_t)b * 4 * H + q * (size_t)H + j] = d[q];
        tiles[tile_offset(b, q * H + j, chunks)] = d[q];
    }
    dc_io[o] = dck * gf;
}

struct LstmDhArgs {
    const float* tiles;         // dgates as tiles
    const float* dgates;        // [B][4H]
    const u32x4_t* w_split;     // of W_hh^T
    const float* w;             // [4H][H]
    float* out;                 // [splits][B][H]
    int B, H;
    int row_blocks, col_blocks, splits, items_per_die;
};

// out[z] = dgates[:, range z] W_hh[range z, :]: 16 RT rows x 16 CT units and one range of k per block, an eighth of it per
// wave.
template <int RT, int CT>
__global__ __launch_bounds__(LX_THREADS, 2) void lstm_dh_f32x6_kernel(const LstmDhArgs a) {
    constexpr int ROWS = 16 * RT, COLS = 16 * CT, P = ROWS + 4;
    __shared__ __attribute__((aligned(16))) float part[LX_WAVES][COLS * P];
    // one die: neighbouring columns and ranges of W
    const int item = (blockIdx.x & 7) * a.items_per_die + (blockIdx.x >> 3);
    if (item >= a.row_blocks * a.col_blocks * a.splits) return;                    // whole block
    const int row0 = item % a.row_blocks * ROWS;
    const int t = item / a.row_blocks;
    const int z = t / a.col_blocks, j0 = t % a.col_blocks * COLS;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = a.H;

    f32x4_t acc[RT][CT];
    clear(acc);
    const int chunks = 4 * H / 32, ways = a.splits * LX_WAVES, way = z * LX_WAVES + wave;
    const int c0 = chunks * way / ways, n = chunks * (way + 1) / ways - c0;
    if (n > 0) {
        wave_product(acc, a.tiles + ((size_t)row0 / 16 * chunks + c0) * 512, a.w_split + ((size_t)j0 / 16 * chunks + c0) * 192,
                     chunks, n, lane, pd_x6_sign(chunks, ways, way));
        if (not_finite(acc)) {
            clear(acc);
            const int idx = lane & 15;
            for (int k = c0 * 32 + (lane >> 4); k < (c0 + n) * 32; k += 4) {
                float wv[CT];
#pragma unroll
                for (int j = 0; j < CT; ++j) wv[j] = a.w[(size_t)k * H + j0 + 16 * j + idx];
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const float gv = a.dgates[(size_t)min(row0 + 16 * i + idx, a.B - 1) * 4 * H + k];
#pragma unroll
                    for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(gv, wv[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
            *(f32x4_t*)&part[wave][(16 * j + (lane & 15)) * P + 16 * i + 4 * (lane >> 4)] = acc[i][j];
    __syncthreads();
    // one column and four rows per thread and turn
    float* const out = a.out + (size_t)z * a.B * H + j0;
#pragma unroll
    for (int s = 0; s < (4 * RT * COLS + LX_THREADS - 1) / LX_THREADS; ++s) {
        const int id = s * LX_THREADS + threadIdx.x;
        const int col = id % COLS, r = id / COLS * 4;
        if (r >= ROWS) continue;
        f32x4_t v = *(const f32x4_t*)&part[0][col * P + r];
#pragma unroll
        for (int w = 1; w < LX_WAVES; ++w) v += *(const f32x4_t*)&part[w][col * P + r];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (row0 + r + e < a.B) out[(size_t)(row0 + r + e) * H + col] = v[e];
    }
}

template <int RT>
void launch_dh(const LstmDhArgs& g, int cols, hipStream_t stream) {
    const dim3 grid(8 * g.items_per_die);
    if (cols == 64) lstm_dh_f32x6_kernel<RT, 4><<<grid, LX_THREADS, 0, stream>>>(g);
    else lstm_dh_f32x6_kernel<RT, 2><<<grid, LX_THREADS, 0, stream>>>(g);
}

// How the backward product of B rows is cut: row blocks of at most 64, 64 or 32 columns, and ranges of k so that about
// one block per CU runs, each wave with a chunk at least.  32 columns where 64 would leave CUs idle.
struct DhPlan { int row_blocks, rt, cols, splits; };
DhPlan dh_plan(int B, int H) {
    DhPlan p;
    p.row_blocks = (B + 63) / 64;
    p.rt = ((B + p.row_blocks - 1) / p.row_blocks + 15) / 16;
    const int most = 4 * H / 32 / LX_WAVES > 1 ? 4 * H / 32 / LX_WAVES : 1;
    p.cols = H % 64 == 0 && H / 64 * p.row_blocks * most >= 256 ? 64 : 32;
    const int want = 256 / (H / p.cols * p.row_blocks);
    p.splits = want < 1 ? 1 : want < most ? want : most;
    return p;
}

template <int RT>
void launch_step(const LstmStepArgs& s, int ct, dim3 grid, hipStream_t stream) {
    if (ct == 2) lstm_step_f32x6_kernel<RT, 2><<<grid, LX_THREADS, 0, stream>>>(s);
    else lstm_step_f32x6_kernel<RT, 1><<<grid, LX_THREADS, 0, stream>>>(s);
}

}  // namespace

extern "C" int pd_lstm_f32x6_supported(int B, int H) { return B > 0 && B <= 128 && H > 0 && H % 32 == 0 && H <= 8192; }

// Bytes of the scratch a layer's time loop needs: the split weights, then the tiles.
extern "C" int pd_lstm_f32x6_workspace_bytes(int backward, int B, int H, uint64_t* weights, uint64_t* tiles) {
    PD_REQUIRE(pd_lstm_f32x6_supported(B, H) && weights && tiles, PD_ESHAPE, "pd_lstm_f32x6_workspace_bytes: shape is not supported");
    const uint64_t row_blocks = (B + 63) / 64, rt = ((B + row_blocks - 1) / row_blocks + 15) / 16;
    const uint64_t rows = row_blocks * rt * 16;
    *weights = 24ull * H * H;
    *tiles = rows * H * 4 * (backward ? 4 : 2);    // dgates; h of this step and of the next
    return PD_OK;
}

extern "C" int pd_lstm_split_weights_f32x6(int backward, const float* w_hh, void* out, int H, void* stream) {
    PD_REQUIRE(H > 0 && H % 32 == 0 && H <= 8192, PD_ESHAPE, "pd_lstm_split_weights_f32x6: H must be a multiple of 32 up to 8192");
    PD_REQUIRE(w_hh && out && pd_aligned(w_hh, 16) && pd_aligned(out, 16), PD_EINVAL,
               "pd_lstm_split_weights_f32x6: NULL or unaligned pointer");
    const long threads = (long)(H / 4) * (H / 32) * 64;
    const dim3 grid((unsigned)((threads + 255) / 256));
    if (backward) lstm_split_weights_t_kernel<<<grid, dim3(256), 0, (hipStream_t)stream>>>(w_hh, (u32x4_t*)out, H);
    else lstm_split_weights_kernel<<<grid, dim3(256), 0, (hipStream_t)stream>>>(w_hh, (u32x4_t*)out, H);
    PD_CHECK_LAUNCH("pd_lstm_split_weights_f32x6");
    return PD_OK;
}

extern "C" int pd_lstm_recurrence_fwd_f32x6(float* gates, const float* w_hh, const void* w_split, const float* b_ih,
                                            const float* b_hh, float* h_tiles, float* c, float* y, int t_begin, int t_end, int B, int H,
                                            void* stream) {
    PD_REQUIRE(pd_lstm_f32x6_supported(B, H), PD_ESHAPE, "pd_lstm_recurrence_fwd_f32x6: shape is not supported");
    PD_REQUIRE(0 <= t_begin && t_begin <= t_end, PD_ESHAPE, "pd_lstm_recurrence_fwd_f32x6: bad range of steps");
    PD_REQUIRE(gates && w_hh && h_tiles && c && y && (t_end <= 1 || w_split), PD_EINVAL, "pd_lstm_recurrence_fwd_f32x6: NULL pointer");
    PD_REQUIRE((b_ih == nullptr) == (b_hh == nullptr), PD_EINVAL, "pd_lstm_recurrence_fwd_f32x6: pass both biases or neither");
    PD_REQUIRE(pd_aligned(gates, 16) && pd_aligned(w_split, 16) && pd_aligned(h_tiles, 16) && pd_aligned(c, 16) && pd_aligned(y, 16) &&
                   (!b_ih || (pd_aligned(b_ih, 16) && pd_aligned(b_hh, 16))), PD_EINVAL,
               "pd_lstm_recurrence_fwd_f32x6: pointers must be 16-byte aligned");
    const size_t bh = (size_t)B * H;
    LstmStepArgs s;
    s.w_split = (const u32x4_t*)w_split;
    s.w = w_hh;
    s.b_ih = b_ih;
    s.b_hh = b_hh;
    s.B = B;
    s.H = H;
    s.row_blocks = (B + 63) / 64;
    const int rt = ((B + s.row_blocks - 1) / s.row_blocks + 15) / 16;
    // eight units a block (less of h read per product), four where that leaves no more blocks than CUs
    const int ct = (H / 4) * s.row_blocks <= 256 ? 1 : 2;
    s.items = H / (4 * ct) * s.row_blocks;
    s.items_per_die = (s.items + 7) / 8;
    const size_t tiles = (size_t)s.row_blocks * rt * 16 * H;
    const dim3 grid(8 * s.items_per_die);
    for (int t = t_begin; t < t_end; ++t) {
        s.gates = gates + t * 4 * bh;
        s.h_prev = t > 0 ? y + (t - 1) * bh : nullptr;
        s.c_prev = t > 0 ? c + (t - 1) * bh : nullptr;
        s.h_in = h_tiles + (t & 1) * tiles;
        s.h_next = h_tiles + ((t & 1) ^ 1) * tiles;
        s.c_out = c + t * bh;
        s.h_out = y + t * bh;
        if (rt == 1) launch_step<1>(s, ct, grid, (hipStream_t)stream);
        else if (rt == 2) launch_step<2>(s, ct, grid, (hipStream_t)stream);
        else if (rt == 3) launch_step<3>(s, ct, grid, (hipStream_t)stream);
        else launch_step<4>(s, ct, grid, (hipStream_t)stream);
        PD_CHECK_LAUNCH("pd_lstm_recurrence_fwd_f32x6");
    }
    return PD_OK;
}

extern "C" int pd_lstm_dh_f32x6_splits(int B, int H) { return pd_lstm_f32x6_supported(B, H) ? dh_plan(B, H).splits : 0; }

extern "C" int pd_lstm_cell_bwd_f32x6(const float* gates, const float* c_prev, const float* c, const float* dy,
                                      const float* dh_rec, int n_rec, float* dc_io, float* dgates, float* tiles, int B,
                                      int H, int first_step, void* stream) {
    PD_REQUIRE(pd_lstm_f32x6_supported(B, H), PD_ESHAPE, "pd_lstm_cell_bwd_f32x6: shape is not supported");
    PD_REQUIRE(gates && c && dy && dc_io && dgates && tiles && (first_step || (dh_rec && n_rec >= 1)), PD_EINVAL,
               "pd_lstm_cell_bwd_f32x6: NULL pointer");
    const int tile_rows = (B + 63) / 64 * dh_plan(B, H).rt;
    lstm_cell_bwd_tiles_kernel<<<dim3(H / 32, 2 * tile_rows), dim3(256), 0, (hipStream_t)stream>>>(
        gates, c_prev, c, dy, dh_rec, n_rec, dc_io, dgates, tiles, B, H, first_step);
    PD_CHECK_LAUNCH("pd_lstm_cell_bwd_f32x6");
    return PD_OK;
}

extern "C" int pd_lstm_dh_f32x6(const float* tiles, const float* dgates, const float* w_hh, const void* w_split,
                                float* dh_rec, int B, int H, void* stream) {
    PD_REQUIRE(pd_lstm_f32x6_supported(B, H), PD_ESHAPE, "pd_lstm_dh_f32x6: shape is not supported");
    PD_REQUIRE(tiles && dgates && w_hh && w_split && dh_rec && pd_aligned(tiles, 16) && pd_aligned(w_split, 16), PD_EINVAL,
               "pd_lstm_dh_f32x6: NULL or unaligned pointer");
    const DhPlan p = dh_plan(B, H);
    LstmDhArgs g;
    g.tiles = tiles; g.dgates = dgates;
    g.w_split = (const u32x4_t*)w_split; g.w = w_hh;
    g.out = dh_rec;
    g.B = B; g.H = H;
    g.row_blocks = p.row_blocks;
    g.col_blocks = H / p.cols;
    g.splits = p.splits;
    g.items_per_die = (g.row_blocks * g.col_blocks * g.splits + 7) / 8;
    hipStream_t s = (hipStream_t)stream;
    if (p.rt == 1) launch_dh<1>(g, p.cols, s);
    else if (p.rt == 2) launch_dh<2>(g, p.cols, s);
    else if (p.rt == 3) launch_dh<3>(g, p.cols, s);
    else launch_dh<4>(g, p.cols, s);
    PD_CHECK_LAUNCH("pd_lstm_dh_f32x6");
    return PD_OK;
}

extern "C" int pd_lstm_recurrence_bwd_f32x6(const float* gates, const float* c, const float* dy, const float* w_hh,
                                            const void* w_split, float* tiles, float* dh_rec, float* dc, float* dgates,
                                            int T, int B, int H, void* stream) {
    PD_REQUIRE(T > 0 && pd_lstm_f32x6_supported(B, H), PD_ESHAPE, "pd_lstm_recurrence_bwd_f32x6: shape is not supported");
    PD_REQUIRE(gates && c && dy && w_hh && dc && dgates && tiles && (T == 1 || (w_split && dh_rec)), PD_EINVAL,
               "pd_lstm_recurrence_bwd_f32x6: NULL pointer");
    const size_t bh = (size_t)B * H;
    const int splits = dh_plan(B, H).splits;
    for (int t = T - 1; t >= 0; --t) {
        int rc = pd_lstm_cell_bwd_f32x6(gates + t * 4 * bh, t > 0 ? c + (t - 1) * bh : nullptr, c + t * bh, dy + t * bh,
                                        dh_rec, splits, dc, dgates + t * 4 * bh, tiles, B, H, t == T - 1, stream);
        if (rc != PD_OK) return rc;
        if (t > 0) {
            rc = pd_lstm_dh_f32x6(tiles, dgates + t * 4 * bh, w_hh, w_split, dh_rec, B, H, stream);
            if (rc != PD_OK) return rc;
        }
    }
    return PD_OK;
}
