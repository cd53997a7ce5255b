// What the Winograd F(2x2, 3x3) forward / input-gradient kernels share: the description of a launch and the division of
// the output into work items of 16 x 16 pixels (64 tiles of 2 x 2) x 64 output channels.
#pragma once
#include "pd_internal.h"

namespace {

typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int WG_THREADS = 512;
constexpr int WG_PIX = 16;                       // a block covers WG_PIX x WG_PIX output pixels
constexpr int WG_BN = 64;                        // output channels per block
constexpr int WG_XCD = 8;
constexpr int WG_HALO = WG_PIX + 2;              // input halo tile: 18 rows x (16 + 2 per segment) pixels

// weight gradient
constexpr int WW_THREADS = 512;
constexpr int WW_BLOCKS = 256;                       // persistent blocks: 8 dies x 32
constexpr int WW_PART_FLOATS = 16 * 64 * 64;         // one block's partial dU
constexpr int WW_PART_STRIDE = WW_PART_FLOATS;       // floats between two blocks' partials

// Two fp32 values as two f16 terms each: the first terms, packed; what a first term leaves of its value, exactly.
__device__ __forceinline__ uint32_t wino_f16_pack(float lo, float hi) {
    uint32_t p;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(p) : "v"(lo), "v"(hi));
    return p;
}
__device__ __forceinline__ float wino_f16_rest_lo(uint32_t p, float x) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(p), "v"(x));
    return r;
}
__device__ __forceinline__ float wino_f16_rest_hi(uint32_t p, float x) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(p), "v"(x));
    return r;
}

}  // namespace

struct WinoArgs {
    const float* x;         // [N,H,W,C]
    const float* u;         // transformed filter, see winograd_filter_kernel
    const float* bias;      // [K] or null
    const float* mask;      // [N,H,W,C] or null: x is taken as 0 where mask <= 0
    const float* out_mask;  // [N,H,W,K] or null: y is written as 0 where out_mask <= 0
    float* y;               // [N,H,W,K]
    float* pool_y;          // pooling variant: [N,H/2,W/2,K], written instead of y
    uint8_t* pool_idx;      // pooling variant: [N,H/2,W/2,K] window position (bits 0-1) and sign (bit 2)
    const uint8_t* unpool_idx;   // unpooling variant: [N,H,W,K] index bytes of the 2x2 pooling that produced this
                                 // convolution's input (the convolution is an input gradient)
    float* unpool_y;        // unpooling variant: [N,2H,2W,K], the gradient in front of that pooling
    int N, H, W, C, K;
    int img_h;              // stacked variant: rows of one image (N is then 1 and H the rows of the whole batch)
    int relu;
    int tiles_x, tiles_y, k_blocks, n_chunks;
    int segs_per_row, n_segs;     // segmented variant: pieces per 16 rows of the stacked batch, pieces in all
    int n_items, items_per_xcd;   // work items (pixel tile x channel block) in all / per die
    int split_log2;         // f16 kernel, split reduction: k_blocks counts (channel block, range of input channels) pairs,
    size_t part_elems;      // n_chunks the chunks of a range, y holds a result per range, part_elems apart
};

// How a launch divides its work (a's sizes, tiles, segments and items are filled in): persistent blocks, segments
// per work item, whether the batch is taken as one tall image.  chunk: input channels per reduction step.
struct WinoPlan { unsigned blocks; int seg; bool stacked; };
int pd_wino_plan(const char* who, WinoArgs& a, int N, int H, int W, int C, int K, int chunk, bool may_stack,
                 WinoPlan* plan);

// Decoded work item: one 16 x 16 pixel tile of one image x one block of 64 output channels.
struct WinoItem { int n, y0, x0, kb; };

__device__ __forceinline__ WinoItem wino_decode(const WinoArgs& a, int item) {
    WinoItem w;
    w.kb = item % a.k_blocks;
    const int tile = item / a.k_blocks;
    const int per_img = a.tiles_x * a.tiles_y;
    w.n = tile / per_img;
    const int rem = tile - w.n * per_img;
    const int ty = rem / a.tiles_x;
    w.y0 = ty * WG_PIX;
    w.x0 = (rem - ty * a.tiles_x) * WG_PIX;
    return w;
}

// Piece s of a work item: first output row and column, and whether it exists (the last item may have fewer).
// SEG = 1: the item's square.
struct SegPos { int y0, x0; bool ok; };
template <int SEG>
__device__ __forceinline__ SegPos seg_pos(const WinoArgs& a, int item, int s) {
    SegPos p;
    if (SEG == 1) {
        const WinoItem w = wino_decode(a, item);
        p.y0 = w.y0; p.x0 = w.x0; p.ok = true;
    } else {
        const int sg = (item / a.k_blocks) * SEG + s;
        const int rb = sg / a.segs_per_row;
        p.y0 = rb * WG_PIX;
        p.x0 = (sg - rb * a.segs_per_row) * (WG_PIX / SEG);
        p.ok = sg < a.n_segs;
    }
    return p;
}

// Weight gradient: a launch of either kernel.
struct WinoWgradArgs {
    const float* x;      // [N,H,W,C]
    const float* dy;     // [N,H,W,K]
    float* part;         // [pair][rank][16][64][64]
    float* part_db;      // [pair][rank][2][64]
    int N, H, W, C, K;
    int sx, sy;          // strips per row pair, row pairs per image (upright strips: strips side by side, unused)
    int n_strips, strips_per_rank;
    int rows_all;        // upright strips: N * H, the rows of the batch taken as one tall image
    int c_blocks, n_pairs, ranks;
};
// block -> (pair, rank): the 32 blocks of a die cover all pairs of a contiguous range of ranks, so that the pairs that
// read the same x and dY run side by side on one L2
__device__ __forceinline__ void wino_wgrad_pair_rank(const WinoWgradArgs& a, int& pair, int& rank) {
    if (a.n_pairs <= 32) {
        const int xcd = blockIdx.x % WG_XCD, slot = blockIdx.x / WG_XCD;
        pair = slot % a.n_pairs;
        rank = xcd * (32 / a.n_pairs) + slot / a.n_pairs;
    } else {                                   // more pairs than a die has blocks: plain round robin
        pair = blockIdx.x % a.n_pairs;
        rank = blockIdx.x / a.n_pairs;
    }
}
// The f16 kernel: writes a.part and a.part_db.
void pd_wino_wgrad_f16x3(const WinoWgradArgs& a, hipStream_t s);
