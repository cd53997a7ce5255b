// A pre-LayerNorm transformer layer's forward and backward pass as one call each: the launches that
// layers._TransformerLayerFn otherwise issues one by one, in the same order with the same arguments (host code only; the
// kernels are the library's).  The reference's checked-out branch has no such stage (README.md:7-8); the layer plays the
// part of torch.nn modules in the reference's stages (runtime/runtime.py:529-530 forward, :606-608 backward).
//
// Why: seven launches forward and some twenty backward through Python and ctypes are about 11 us of host time each, more
// than the kernels take below a few hundred tokens.  Six layers' validation pass over 128 tokens 504 -> 349 us, four
// layers' training step of 4 x 600 tokens 6.9 -> 3.8 ms (with the fused attention for its 200 positions; 5.5 without).
#include "pd_internal.h"

namespace {

constexpr int COLSUM_SPLITS = 64;              // row ranges of the batched column sums

// Regions of a buffer, each on a 256-byte boundary.
struct Regions {
    char* base;
    uint64_t at = 0;
    uint64_t* starts;                          // of the regions so far, where somebody asks for them
    explicit Regions(void* p, uint64_t* starts = nullptr) : base((char*)p), starts(starts) {}
    template <typename T>
    T* take(uint64_t count) {
        T* p = base ? (T*)(base + at) : nullptr;
        if (starts) *starts++ = at;
        at += (count * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

struct Dims {
    int batch, seq, heads, H, F;
    uint64_t T;                                // tokens
    bool fused;                                // attention without score matrices
    uint64_t scores;                           // [batch][heads][seq][seq] or [batch][heads][seq]
};

int make_dims(const char* who, int batch, int seq, int heads, int hidden, int ffn, Dims* d) {
    PD_REQUIRE(batch > 0 && seq > 0 && heads > 0 && hidden > 0 && ffn > 0 && hidden % heads == 0, PD_ESHAPE, "%s: bad dimensions", who);
    PD_REQUIRE((long long)batch * seq < (1ll << 31) && (long long)batch * heads <= 65535, PD_ESHAPE, "%s: too large", who);
    d->batch = batch; d->seq = seq; d->heads = heads; d->H = hidden; d->F = ffn;
    d->T = (uint64_t)batch * seq;
    d->fused = pd_attention_fwd_supported(seq, hidden / heads) != 0;
    d->scores = (uint64_t)batch * heads * seq * (d->fused ? 1 : seq);
    return PD_OK;
}

// What the forward pass leaves for the backward pass.
struct Saved {
    uint16_t *h1, *qkv, *att, *x2, *h2, *f, *g;
    float *mean1, *rstd1, *mean2, *rstd2;
    float* lse2;
    uint16_t* probs;
    uint64_t bytes;
    Saved(const Dims& d, void* p, uint64_t* starts = nullptr) {
        Regions r(p, starts);
        h1 = r.take<uint16_t>(d.T * d.H);
        mean1 = r.take<float>(d.T);
        rstd1 = r.take<float>(d.T);
        qkv = r.take<uint16_t>(d.T * 3 * d.H);
        lse2 = d.fused ? r.take<float>(d.scores) : nullptr;      // (either of the two)
        probs = d.fused ? nullptr : r.take<uint16_t>(d.scores);
        att = r.take<uint16_t>(d.T * d.H);
        x2 = r.take<uint16_t>(d.T * d.H);
        h2 = r.take<uint16_t>(d.T * d.H);
        mean2 = r.take<float>(d.T);
        rstd2 = r.take<float>(d.T);
        f = r.take<uint16_t>(d.T * d.F);
        g = r.take<uint16_t>(d.T * d.F);
        bytes = r.at;
    }
};

// Temporaries of the backward pass.
struct Work {
    uint16_t *df, *dh2, *dx2, *datt, *dqkv, *dh1, *dscores;
    float *delta, *ln[4], *partials, *sums;
    uint64_t sums_floats, bytes;
    int ln_rows;
    Work(const Dims& d, void* p) {
        Regions r(p);
        df = r.take<uint16_t>(d.T * d.F);
        dh2 = r.take<uint16_t>(d.T * d.H);
        dx2 = r.take<uint16_t>(d.T * d.H);
        datt = r.take<uint16_t>(d.T * d.H);
        dqkv = r.take<uint16_t>(d.T * 3 * d.H);
        dh1 = r.take<uint16_t>(d.T * d.H);
        delta = d.fused ? r.take<float>(d.scores) : nullptr;
        dscores = d.fused ? nullptr : r.take<uint16_t>(d.scores);
        ln_rows = pd_layernorm_bwd_partials((int)d.T);
        for (float*& q : ln) q = r.take<float>((uint64_t)ln_rows * d.H);
        const int shapes[4][2] = {{d.H, d.F}, {d.F, d.H}, {d.H, d.H}, {3 * d.H, d.H}};
        uint64_t most = 0;
        for (const auto& s : shapes) {
            const int splits = pd_gemm_bf16_wgrad_splits(d.T, s[0], s[1]);
            const uint64_t n = splits > 1 ? (uint64_t)splits * s[0] * s[1] : 0;
            if (n > most) most = n;
        }
        partials = r.take<float>(most);
        const int kinds[8] = {1, 1, 0, 0, 1, 1, 0, 0}, cols[8] = {d.H, d.F, d.H, d.H, d.H, 3 * d.H, d.H, d.H};
        sums_floats = 0;
        pd_colsum_batch_workspace_floats(8, kinds, cols, COLSUM_SPLITS, &sums_floats);
        sums = r.take<float>(sums_floats);
        bytes = r.at;
    }
};

// rc of a step, or go on
#define PD_STEP(call)                 \
    do {                              \
        const int rc__ = (call);      \
        if (rc__ != PD_OK) return rc__; \
    } while (0)

int batched(int ta, int tb, int M, int N, int K, const uint16_t* a, int lda, const uint16_t* b, int ldb, uint16_t* c, int ldc,
            float alpha, const Dims& d, const int64_t (&strides)[6], void* stream) {
    return pd_gemm_bf16(ta, tb, M, N, K, a, lda, b, ldb, c, ldc, 0, alpha, 0.f, nullptr, nullptr, 0, d.batch, d.heads, strides,
                        stream);
}

int attention_forward(const Dims& d, const Saved& s, void* stream) {
    const int S = d.seq, hd = d.H / d.heads, ld = 3 * d.H;
    if (d.fused) return pd_attention_fwd_bf16(s.qkv, s.att, nullptr, s.lse2, d.batch, S, d.heads, hd, stream);
    const int64_t SS = (int64_t)S * S, head = hd, row = (int64_t)S * ld;
    PD_STEP(batched(0, 1, S, S, hd, s.qkv, ld, s.qkv + d.H, ld, s.probs, S, (float)(1.0 / sqrt((double)hd)), d,
                    {row, head, row, head, d.heads * SS, SS}, stream));
    PD_STEP(pd_softmax_fwd_bf16(s.probs, s.probs, (int64_t)d.batch * d.heads * S, S, stream));
    return batched(0, 0, S, hd, S, s.probs, S, s.qkv + 2 * d.H, ld, s.att, d.H, 1.f, d,
                   {d.heads * SS, SS, row, head, (int64_t)S * d.H, head}, stream);
}

int attention_backward(const Dims& d, const Saved& s, const Work& w, void* stream) {
    const int S = d.seq, H = d.H, hd = H / d.heads, ld = 3 * H;
    if (d.fused)
        return pd_attention_bwd_bf16(s.qkv, s.att, w.datt, s.lse2, w.delta, w.dqkv, d.batch, S, d.heads, hd, stream);
    const float scale = (float)(1.0 / sqrt((double)hd));
    const int64_t SS = (int64_t)S * S, head = hd, row = (int64_t)S * ld, orow = (int64_t)S * H, hs = d.heads * SS;
    PD_STEP(batched(0, 1, S, S, hd, w.datt, H, s.qkv + 2 * H, ld, w.dscores, S, 1.f, d, {orow, head, row, head, hs, SS}, stream));
    PD_STEP(batched(1, 0, S, hd, S, s.probs, S, w.datt, H, w.dqkv + 2 * H, ld, 1.f, d, {hs, SS, orow, head, row, head}, stream));
    PD_STEP(pd_softmax_bwd_bf16(s.probs, w.dscores, w.dscores, (int64_t)d.batch * d.heads * S, S, stream));
    PD_STEP(batched(0, 0, S, hd, S, w.dscores, S, s.qkv + H, ld, w.dqkv, ld, scale, d, {hs, SS, row, head, row, head}, stream));
    return batched(1, 0, S, hd, S, w.dscores, S, s.qkv, ld, w.dqkv + H, ld, scale, d, {hs, SS, row, head, row, head}, stream);
}

// dw [n][k] (+)= dy^T x
int weight_gradient(const uint16_t* dy, const uint16_t* x, float* dw, bool add, uint64_t T, int n, int k, float* partials,
                    void* stream) {
    const int splits = pd_gemm_bf16_wgrad_splits(T, n, k);
    if (splits == 1)
        return pd_gemm_bf16(1, 0, n, k, (int)T, dy, n, x, k, dw, k, 1, 1.f, add ? 1.f : 0.f, nullptr, nullptr, 0, 1, 1, nullptr, stream);
    const int rows = (int)(T / splits);
    const int64_t strides[6] = {(int64_t)rows * n, 0, (int64_t)rows * k, 0, (int64_t)n * k, 0};
    PD_STEP(pd_gemm_bf16(1, 0, n, k, rows, dy, n, x, k, partials, k, 1, 1.f, 0.f, nullptr, nullptr, 0, splits, 1, strides, stream));
    return pd_splitk_reduce_f32(partials, splits, n, k, nullptr, 0, add ? 1.f : 0.f, dw, k, stream);
}

enum { LN1_W, LN1_B, QKV_W, QKV_B, PROJ_W, PROJ_B, LN2_W, LN2_B, FC1_W, FC1_B, FC2_W, FC2_B, N_PARAMS };

int check_params(const char* who, const void* const* params) {
    PD_REQUIRE(params, PD_EINVAL, "%s: NULL pointer", who);
    for (int i = 0; i < N_PARAMS; ++i) PD_REQUIRE(params[i], PD_EINVAL, "%s: NULL parameter", who);
    return PD_OK;
}

}  // namespace

extern "C" int pd_gemm_bf16_wgrad_splits(uint64_t T, int n, int k) {
    if (n <= 0 || k <= 0) return 1;
    const long tiles = (long)((n + 127) / 128) * ((k + 127) / 128);
    if (tiles > 64) return 1;
    long s = 256 / tiles;
    if ((long)(T / 1024) < s) s = (long)(T / 1024);
    if (s > 8) s = 8;
    return s < 2 || T % (s * 128) != 0 || n % 4 != 0 || k % 4 != 0 ? 1 : (int)s;
}

extern "C" int pd_transformer_layer_saved_offsets(int batch, int seq, int heads, int hidden, int ffn, uint64_t* offsets) {
    Dims d;
    PD_STEP(make_dims("pd_transformer_layer_saved_offsets", batch, seq, heads, hidden, ffn, &d));
    PD_REQUIRE(offsets, PD_EINVAL, "pd_transformer_layer_saved_offsets: NULL pointer");
    Saved(d, nullptr, offsets);
    return PD_OK;
}

extern "C" int pd_transformer_layer_bytes(int batch, int seq, int heads, int hidden, int ffn, uint64_t* saved, uint64_t* work) {
    Dims d;
    PD_STEP(make_dims("pd_transformer_layer_bytes", batch, seq, heads, hidden, ffn, &d));
    PD_REQUIRE(saved && work, PD_EINVAL, "pd_transformer_layer_bytes: NULL pointer");
    *saved = Saved(d, nullptr).bytes;
    *work = Work(d, nullptr).bytes;
    return PD_OK;
}

extern "C" int pd_transformer_layer_fwd_bf16(const void* const* params, const uint16_t* x, void* saved, uint16_t* y, int batch,
                                             int seq, int heads, int hidden, int ffn, float eps, void* stream) {
    const char* who = "pd_transformer_layer_fwd_bf16";
    Dims d;
    PD_STEP(make_dims(who, batch, seq, heads, hidden, ffn, &d));
    PD_STEP(check_params(who, params));
    PD_REQUIRE(x && saved && y && pd_aligned(saved, 256), PD_EINVAL, "%s: NULL pointer or saved not 256-byte aligned", who);
    const Saved s(d, saved);
    const auto F = [&](int i) { return (const float*)params[i]; };
    const auto W = [&](int i) { return (const uint16_t*)params[i]; };
    const int T = (int)d.T, H = d.H;
    PD_STEP(pd_layernorm_fwd_bf16(x, F(LN1_W), F(LN1_B), s.h1, s.mean1, s.rstd1, T, H, eps, stream));
    PD_STEP(pd_gemm_bf16(0, 1, T, 3 * H, H, s.h1, H, W(QKV_W), H, s.qkv, 3 * H, 0, 1.f, 0.f, F(QKV_B), nullptr, 0, 1, 1, nullptr, stream));
    PD_STEP(attention_forward(d, s, stream));
    PD_STEP(pd_gemm_bf16(0, 1, T, H, H, s.att, H, W(PROJ_W), H, s.x2, H, 0, 1.f, 0.f, F(PROJ_B), x, H, 1, 1, nullptr, stream));
    PD_STEP(pd_layernorm_fwd_bf16(s.x2, F(LN2_W), F(LN2_B), s.h2, s.mean2, s.rstd2, T, H, eps, stream));
    PD_STEP(pd_gemm_bf16_gelu(0, 0, 1, T, ffn, H, s.h2, H, W(FC1_W), H, s.f, ffn, F(FC1_B), s.g, ffn, stream));
    return pd_gemm_bf16(0, 1, T, H, ffn, s.g, ffn, W(FC2_W), ffn, y, H, 0, 1.f, 0.f, F(FC2_B), s.x2, H, 1, 1, nullptr, stream);
}

extern "C" int pd_transformer_layer_bwd_bf16(const void* const* params, float* const* grads, uint32_t add, const uint16_t* x,
                                             void* saved, const uint16_t* dy, void* work, uint16_t* dx, int batch, int seq,
                                             int heads, int hidden, int ffn, void* stream) {
    const char* who = "pd_transformer_layer_bwd_bf16";
    Dims d;
    PD_STEP(make_dims(who, batch, seq, heads, hidden, ffn, &d));
    PD_STEP(check_params(who, params));
    PD_STEP(check_params(who, (const void* const*)grads));
    PD_REQUIRE(x && saved && dy && work && dx && pd_aligned(saved, 256) && pd_aligned(work, 256), PD_EINVAL,
               "%s: NULL pointer, or saved or work not 256-byte aligned", who);
    const Saved s(d, saved);
    const Work w(d, work);
    const auto F = [&](int i) { return (const float*)params[i]; };
    const auto W = [&](int i) { return (const uint16_t*)params[i]; };
    const int T = (int)d.T, H = d.H;
    const auto input_grad = [&](const uint16_t* g, int n, int p, uint16_t* out) {
        return pd_gemm_bf16(0, 0, T, H, n, g, n, W(p), H, out, H, 0, 1.f, 0.f, nullptr, nullptr, 0, 1, 1, nullptr, stream);
    };
    const auto weight_grad = [&](const uint16_t* g, const uint16_t* in, int n, int k, int p) {
        return weight_gradient(g, in, grads[p], add >> p & 1, d.T, n, k, w.partials, stream);
    };
    // y = fc2(gelu(fc1(LN2(x2)))) + x2
    PD_STEP(weight_grad(dy, s.g, H, ffn, FC2_W));
    PD_STEP(pd_gemm_bf16_gelu(1, 0, 0, T, ffn, H, dy, H, W(FC2_W), ffn, w.df, ffn, nullptr, s.f, ffn, stream));
    PD_STEP(weight_grad(w.df, s.h2, ffn, H, FC1_W));
    PD_STEP(input_grad(w.df, ffn, FC1_W, w.dh2));
    PD_STEP(pd_layernorm_bwd_bf16(w.dh2, s.x2, F(LN2_W), s.mean2, s.rstd2, w.dx2, dy, w.ln[0], w.ln[1], T, H, stream));
    // x2 = proj(attention(qkv(LN1(x)))) + x
    PD_STEP(weight_grad(w.dx2, s.att, H, H, PROJ_W));
    PD_STEP(input_grad(w.dx2, H, PROJ_W, w.datt));
    PD_STEP(attention_backward(d, s, w, stream));
    PD_STEP(weight_grad(w.dqkv, s.h1, 3 * H, H, QKV_W));
    PD_STEP(input_grad(w.dqkv, 3 * H, QKV_W, w.dh1));
    PD_STEP(pd_layernorm_bwd_bf16(w.dh1, x, F(LN1_W), s.mean1, s.rstd1, dx, w.dx2, w.ln[2], w.ln[3], T, H, stream));
    // the bias gradients and the sums over the LayerNorm kernels' partial results
    const void* xs[8] = {dy, w.df, w.ln[0], w.ln[1], w.dx2, w.dqkv, w.ln[2], w.ln[3]};
    const int kinds[8] = {1, 1, 0, 0, 1, 1, 0, 0};
    const int at[8] = {FC2_B, FC1_B, LN2_W, LN2_B, PROJ_B, QKV_B, LN1_W, LN1_B};
    const int cols[8] = {H, ffn, H, H, H, 3 * H, H, H};
    float* outs[8];
    uint64_t rows[8], lds[8];
    float betas[8];
    for (int i = 0; i < 8; ++i) {
        outs[i] = grads[at[i]];
        rows[i] = kinds[i] ? d.T : (uint64_t)w.ln_rows;
        lds[i] = cols[i];
        betas[i] = add >> at[i] & 1 ? 1.f : 0.f;
    }
    return pd_colsum_batch(8, xs, kinds, outs, rows, cols, lds, betas, w.sums, w.sums_floats, COLSUM_SPLITS, stream);
}
