// rh_train.cpp -- the training pass behind include/rustane_hip.h:
// full_model::forward + backward_ws (full_model.rs:915-991, 592-702) with
// layer::backward_into (layer.rs:7037-7366) per layer.
//
// The forward is the inference forward's kernels with every activation the
// backward needs kept per layer (the ForwardCache of layer.rs:79-126): the
// layer input and post-attention residuals (fp32), the normalised GEMM
// operands, q/k/v, the attention output and its log-sum-exp, the SwiGLU
// pre-activations and gate.  The backward then runs, per layer in reverse:
//
//   dW2 += dffn^T gate          dgate = dffn W2          (SiLU backward) -> dh1|dh3
//   dx_ffn = dh1 W1^T + dh3 W3^T    dW1, dW3 += x2n^T dh{1,3}
//   dx2 = RMSNorm2'(dx_ffn) + dy    da = (a dx2) Wo^T    dWo += attn^T (a dx2)
//   attention backward -> dq, dk, dv   (RoPE backward on dq, dk)
//   dxn = dq Wq^T + dk Wk^T + dv Wv^T   dWq, dWk, dWv += xn^T d{q,k,v}
//   dy' = RMSNorm1'(dxn) + dx2
//
// Every product is an NT GEMM of the forward's kernel: the data-gradient
// GEMMs stream transposed copies of the weights (built once per weight
// version), the weight-gradient GEMMs contract over tokens (whole blocks of
// 128 read in place by transposing LDS reads; ragged counts, and short first
// stores of large outputs, from token-inner copies of the operands), and
// accumulate into the fp32 gradients in their epilogue (C += kappa * acc).
// Gradients keep the reference's tensor shapes and orientation and accumulate
// across calls.
#include "rh_ctx.h"

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <vector>

namespace rhrt {

struct TrainState {
    // M: token capacity of the buffers; Mp: this call's token count B * S
    // rounded up to 128 (the K of the weight-gradient GEMMs, <= capacity's)
    int M = 0, Mp = 0, B = 0, S = 0;
    uint64_t packs_gen = 0;            // weight version the transposed copies hold
    bool zero = true;  // every gradient is 0: the weight-gradient GEMMs store instead of accumulating
    bool have_static = false;  // the gradients and transposed weights below are allocated
    // fp32 gradients, reference orientation (RSTK order per layer)
    float *dembed = nullptr, *dgf = nullptr;
    std::vector<std::array<float*, 9>> dlay;  // value-initialised: null until allocated
    // transposed fp16 weights (fragment order)
    f16* embed_t = nullptr;  // [D][Vp]
    struct WT { f16 *qkvt = nullptr, *ot = nullptr, *w13t = nullptr, *w2t = nullptr; };
    std::vector<WT> wt;
    // per-layer forward caches
    struct Cache {
        float *xin, *x2, *lse;
        f16 *xn, *q, *k, *v, *attn, *x2n, *h13, *gate;
    };
    std::vector<Cache> c;
    float* xlast = nullptr;  // residual after the last layer
    f16* xf = nullptr;       // final RMSNorm rows (fragment order)
    // backward workspace
    // Activation gradients in fp16 fragment order, one buffer per role so each
    // is rewritten only once per layer: H1 = the layer's output gradient times
    // alpha (dffn), H1m = alpha * dx2, H2 = [dh1 | dh3], H2q = [dq | dk | dv].
    f16 *dlh = nullptr, *H1 = nullptr, *H1m = nullptr, *H2 = nullptr, *H2q = nullptr;
    // The weight-gradient GEMMs run on the side stream in four groups per
    // layer (0: dW2, 1: dW1 dW3, 2: dWo, 3: dWq dWk dWv), from the activation
    // gradient above and a forward cache, or (enqueue_backward says when) from
    // token-inner copies of them, tx[g] and dlT (written on the side stream too).
    // ready[g] (main): group g's activation gradient is written; read[g]
    // (side): it has been read (by the GEMM, or by the copy), so the main
    // stream may rewrite that buffer a layer later.
    f16 *tx[4][2] = {}, *dlT = nullptr;
    int txM = 0;  // token capacity of the copies (0: none allocated)
    hipStream_t side = nullptr;
    hipEvent_t ready[5] = {}, read[4] = {};  // ready[4]: the logits gradient
    f16* dOh = nullptr;
    float *gout = nullptr, *dres = nullptr, *Drow = nullptr, *dgp = nullptr;
    uint32_t* utok = nullptr;
    int *ustart = nullptr, *uidx = nullptr;
    // optimizer: the fp32 master weights (created by the first fp32 weight
    // load or optimizer call) and ModelOptState's moments (first optimizer call)
    struct Opt {
        float* emb = nullptr;                  // master embedding [V][D]
        std::vector<std::array<float*, 7>> w;  // masters of the 7 matrices per layer
        uint64_t synced = 0;                   // weight version the masters hold
        bool moments = false;                  // moments and norm partials allocated
        float *emb_m = nullptr, *emb_v = nullptr, *gf_m = nullptr, *gf_v = nullptr;
        std::vector<std::array<float*, 9>> m, v;
    };
    Opt* opt = nullptr;
    // gradient norm: per-block sums of squares of every gradient tensor, their sum
    float* norm_part = nullptr;
    double* norm_sum = nullptr;
    // The kept forward (ForwardResult, full_model.rs:120-129): the caches
    // above, ctx->logits and ctx->d_tgt hold the forward of fwd_B sequences of
    // fwd_S tokens run at ctx->work_epoch == fwd_epoch with logit softcap
    // fwd_softcap; utok/ustart/uidx hold the embedding backward's index.
    uint64_t fwd_epoch = 0, fwd_id = 0;
    int fwd_B = 0, fwd_S = 0, fwd_nuniq = 0;
    float fwd_softcap = 0.f;
    std::vector<uint32_t> fwd_tokens;
    ~TrainState() {
        if (side) {
            (void)hipStreamSynchronize(side);
            (void)hipStreamDestroy(side);
        }
        for (hipEvent_t e : ready)
            if (e) (void)hipEventDestroy(e);
        for (hipEvent_t e : read)
            if (e) (void)hipEventDestroy(e);
        delete opt;
    }
};

void train_state_free(TrainState* t) { delete t; }

int zero_moments(rh_ctx* ctx);

int weights_written(rh_ctx* ctx, bool masters_hold_them) {
    TrainState* T = ctx->train;
    if (!T || !T->opt) return RH_OK;
    if (masters_hold_them) T->opt->synced = ctx->wgen;
    if (T->opt->moments) RCK(zero_moments(ctx));
    return RH_OK;
}

const float* train_master(const rh_ctx* ctx, int l, int j) {
    const TrainState* T = ctx->train;
    if (!T || !T->opt || T->opt->synced != ctx->wgen) return nullptr;
    return j < 0 ? T->opt->emb : T->opt->w[l][j];
}

}  // namespace rhrt

using namespace rhrt;

namespace {

size_t round_up(size_t x, size_t m) { return (x + m - 1) / m * m; }

// The host side of the training state (no device memory yet).
int ensure_train_host(rh_ctx* ctx) {
    if (ctx->train) return RH_OK;
    ctx->train = new (std::nothrow) TrainState;
    return ctx->train ? RH_OK : fail(ctx, RH_ENOMEM, "out of host memory");
}

// Gradients and transposed weights: allocated once per context (a call that
// could not allocate them all is continued by the next).
int ensure_train_static(rh_ctx* ctx) {
    RCK(ensure_train_host(ctx));
    TrainState* T = ctx->train;
    if (T->have_static) return RH_OK;
    const rh_config& c = ctx->cfg;
    const size_t D = c.dim, F = c.hidden, V = c.vocab, Vp = round_up(V, 128);
    if (!T->side)  // the weight-gradient GEMMs' stream (default priority, like the context's)
        HCK(hipStreamCreateWithFlags(&T->side, hipStreamNonBlocking));
    for (hipEvent_t& e : T->ready)
        if (!e) HCK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    for (hipEvent_t& e : T->read)
        if (!e) HCK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    auto once = [&](auto*& p, size_t n) { return p ? RH_OK : dalloc(ctx, &p, n); };
    RCK(once(T->dembed, V * D));
    RCK(once(T->dgf, D));
    T->dlay.resize(c.nlayers);
    const size_t sz[9] = {D * D, D * D, D * D, D * D, D * F, D * F, D * F, D, D};
    size_t nparts = rh::sumsq_blocks(V * D) + rh::sumsq_blocks(D);
    for (auto& g : T->dlay)
        for (int j = 0; j < 9; ++j) {
            RCK(once(g[j], sz[j]));
            nparts += rh::sumsq_blocks(sz[j]);
        }
    RCK(once(T->norm_part, nparts));
    RCK(once(T->norm_sum, 1));
    RCK(once(T->embed_t, D * Vp));
    T->wt.resize(c.nlayers);
    for (auto& w : T->wt) {
        RCK(once(w.qkvt, D * 3 * D));
        RCK(once(w.ot, D * D));
        RCK(once(w.w13t, D * 2 * F));
        RCK(once(w.w2t, F * D));
    }
    T->zero = true;
    T->have_static = true;
    return RH_OK;
}

// Whether the store-wave kernel takes the first store of a gradient [rows][cols]
// (store_waves: of this call's).
bool store_wave_size(const rh_ctx* ctx, size_t rows, size_t cols) {
    return ctx->train->Mp <= 1024 && rows * cols >= (size_t)4096 * 4096;
}
bool store_waves(const rh_ctx* ctx, int rows, int cols) {
    return ctx->train->zero && store_wave_size(ctx, rows, cols);
}

void drop_copies(rh_ctx* ctx) {
    TrainState* T = ctx->train;
    T->txM = 0;
    drop(ctx, T->dlT);
    for (auto& pr : T->tx)
        for (f16*& p : pr) drop(ctx, p);
}

// The token-inner copies (0.8 GB at 4096 wide, vocabulary 32000 and 4096
// tokens), sized for the buffers' capacity by the first call that needs them:
// a token count that is no multiple of 128, or outputs that the store-wave
// kernel takes when they are next zeroed.
int ensure_copies(rh_ctx* ctx) {
    TrainState* T = ctx->train;
    const size_t d = ctx->cfg.dim, f = ctx->cfg.hidden, v = ctx->cfg.vocab;
    const bool need = T->B * T->S != T->Mp || store_wave_size(ctx, d, std::max({d, f, v}));
    if (!need || T->txM >= T->M) return RH_OK;
    HCK(hipStreamSynchronize(T->side));  // reads them
    drop_copies(ctx);
    const rh_config& c = ctx->cfg;
    const size_t D = c.dim, F = c.hidden, Vp = round_up(c.vocab, 128), mp = round_up(T->M, 128);
    RCK(dalloc(ctx, &T->dlT, Vp * mp));
    const size_t rows[4][2] = {{D, F}, {D, 2 * F}, {D, D}, {D, 3 * D}};
    for (int g = 0; g < 4; ++g)
        for (int i = 0; i < 2; ++i) RCK(dalloc(ctx, &T->tx[g][i], rows[g][i] * mp));
    T->txM = T->M;
    return RH_OK;
}

// Caches and workspace for B sequences of S tokens (grow-only).
int ensure_train_ws(rh_ctx* ctx, int B, int S) {
    TrainState* T = ctx->train;
    const int M = B * S;
    if (M <= T->M) {  // every buffer is indexed with the current B, S: any B*S within capacity fits
        T->B = B;
        T->S = S;
        T->Mp = (int)round_up((size_t)M, 128);
        return RH_OK;
    }
    HCK(hipStreamSynchronize(ctx->stream));
    if (T->side) HCK(hipStreamSynchronize(T->side));  // the weight-gradient stream reads some of them
    // free the old per-shape buffers; no capacity until every new one is there
    T->M = 0;
    for (auto& cc : T->c) {
        drop(ctx, cc.xin); drop(ctx, cc.x2); drop(ctx, cc.lse); drop(ctx, cc.xn); drop(ctx, cc.q); drop(ctx, cc.k);
        drop(ctx, cc.v); drop(ctx, cc.attn); drop(ctx, cc.x2n); drop(ctx, cc.h13); drop(ctx, cc.gate);
    }
    drop(ctx, T->xlast); drop(ctx, T->xf); drop(ctx, T->dlh); drop(ctx, T->H1); drop(ctx, T->H1m);
    drop(ctx, T->H2); drop(ctx, T->H2q); drop(ctx, T->dOh); drop(ctx, T->gout); drop(ctx, T->dres);
    drop(ctx, T->Drow); drop(ctx, T->dgp); drop(ctx, T->utok); drop(ctx, T->ustart); drop(ctx, T->uidx);
    drop_copies(ctx);
    const rh_config& c = ctx->cfg;
    const size_t D = c.dim, F = c.hidden, V = c.vocab, Vp = round_up(V, 128);
    const size_t m = M, m16 = round_up(m, 16), mp = round_up(m, 128);
    T->c.assign(c.nlayers, TrainState::Cache{});
    for (auto& cc : T->c) {
        RCK(dalloc(ctx, &cc.xin, m * D));
        RCK(dalloc(ctx, &cc.x2, m * D));
        RCK(dalloc(ctx, &cc.lse, (size_t)M * c.heads));
        RCK(dalloc(ctx, &cc.xn, m16 * D));
        RCK(dalloc(ctx, &cc.q, m * D));
        RCK(dalloc(ctx, &cc.k, m * D));
        RCK(dalloc(ctx, &cc.v, m * D));
        RCK(dalloc(ctx, &cc.attn, m16 * D));
        RCK(dalloc(ctx, &cc.x2n, m16 * D));
        RCK(dalloc(ctx, &cc.h13, 2 * m * F));
        RCK(dalloc(ctx, &cc.gate, m16 * F));
    }
    RCK(dalloc(ctx, &T->xlast, m * D));
    RCK(dalloc(ctx, &T->xf, m16 * D));
    RCK(dalloc(ctx, &T->dlh, m16 * Vp));
    RCK(dalloc(ctx, &T->H1, m16 * D));
    RCK(dalloc(ctx, &T->H1m, m16 * D));
    RCK(dalloc(ctx, &T->H2, m16 * 2 * F));
    RCK(dalloc(ctx, &T->H2q, m16 * 3 * D));
    RCK(dalloc(ctx, &T->dOh, m * D));
    RCK(dalloc(ctx, &T->gout, m * D));  // an unsplit data-gradient product [M][D]
    RCK(dalloc(ctx, &T->dres, m * D));
    RCK(dalloc(ctx, &T->Drow, (size_t)M * c.heads));
    RCK(dalloc(ctx, &T->dgp, (size_t)rh::rms_backward_blocks(M, (int)D) * D));
    RCK(dalloc(ctx, &T->utok, m));
    RCK(dalloc(ctx, &T->ustart, m + 1));
    RCK(dalloc(ctx, &T->uidx, m));
    T->M = M;
    T->Mp = (int)mp;
    T->B = B;
    T->S = S;
    return RH_OK;
}

// Transposed weight copies for the data-gradient GEMMs, rebuilt when the
// weights changed since they were made.
int ensure_packs(rh_ctx* ctx) {
    TrainState* T = ctx->train;
    if (T->packs_gen == ctx->wgen) return RH_OK;
    const rh_config& c = ctx->cfg;
    const int D = c.dim, F = c.hidden, V = c.vocab, Vp = (int)round_up(V, 128);
    hipStream_t st = ctx->stream;
    LCK(rh::launch_transpose_frag(ctx->embed, T->embed_t, V, D, Vp, 0, st));
    for (int l = 0; l < c.nlayers; ++l) {
        const Layer& W = ctx->L[l];
        LCK(rh::launch_transpose_frag(W.wqkv, T->wt[l].qkvt, 3 * D, D, 3 * D, 0, st));
        LCK(rh::launch_transpose_frag(W.wo, T->wt[l].ot, D, D, D, 0, st));
        LCK(rh::launch_transpose_frag(W.w13, T->wt[l].w13t, 2 * F, D, 2 * F, 1, st));
        LCK(rh::launch_transpose_frag(W.w2, T->wt[l].w2t, D, F, D, 0, st));
    }
    T->packs_gen = ctx->wgen;
    return RH_OK;
}

// The forward token loop of enqueue_body with the caches kept per layer.
int enqueue_forward_train(rh_ctx* ctx, int B, int S) {
    TrainState* T = ctx->train;
    const rh_config& c = ctx->cfg;
    const int M = B * S, D = c.dim, F = c.hidden;
    const float alpha = 1.0f / std::sqrt(2.0f * (float)c.nlayers);
    hipStream_t st = ctx->stream;
    // The residual stream moves out of place through the per-layer caches the
    // backward reads: xin[l] -> (Wo) x2[l] -> (W2) xin[l + 1] ... -> xlast.
    LCK(rh::launch_embed(ctx->d_tok, ctx->embed, T->c[0].xin, M, D, c.vocab, ctx->d_err, st));
    LCK(rh::launch_rmsnorm(T->c[0].xin, ctx->L[0].g1, T->c[0].xn, M, D, c.rms_eps, st, true));
    for (int l = 0; l < c.nlayers; ++l) {
        const Layer& W = ctx->L[l];
        const TrainState::Cache& cc = T->c[l];
        rh::GemmArgs g{};
        g.W = W.wqkv; g.X = cc.xn; g.M = M; g.N = 3 * D; g.K = D;
        g.q = cc.q; g.kc = cc.k; g.vc = cc.v; g.rope = ctx->rope;
        g.S = S; g.D = D; g.H = c.heads; g.hd = c.head_dim; g.ctx = S; g.pos0 = 0;
        set_sk(ctx, g);
        RCK(timed(ctx, RH_K_GEMM_QKV, [&] { return rh::launch_gemm(rh::EPI_QKV, g, st); }));
        RCK(timed(ctx, RH_K_ATTN, [&] {
            return rh::launch_attn_prefill(cc.q, cc.k, cc.v, cc.attn, B, c.heads, S, c.head_dim, S, st, cc.lse);
        }));
        g = rh::GemmArgs{};
        g.W = W.wo; g.X = cc.attn; g.M = M; g.N = D; g.K = D;
        g.resid_in = cc.xin; g.out_f32 = cc.x2; g.ldo = D; g.alpha = alpha;
        set_sk(ctx, g);
        RCK(timed(ctx, RH_K_GEMM_WO, [&] { return rh::launch_gemm_resid_norm(g, W.g2, c.rms_eps, cc.x2n, st); }));
        g = rh::GemmArgs{};
        g.W = W.w13; g.X = cc.x2n; g.M = M; g.N = 2 * F; g.K = D;
        g.out_f16 = cc.gate; g.ldo = F; g.h13 = cc.h13;
        set_sk(ctx, g);
        RCK(timed(ctx, RH_K_GEMM_W13, [&](hipEvent_t t0, hipEvent_t t1) {
            g.prof_start = t0; g.prof_stop = t1;
            return rh::launch_gemm(rh::EPI_SWIGLU_SAVE, g, st);
        }));
        const bool last = l + 1 == c.nlayers;
        g = rh::GemmArgs{};
        g.W = W.w2; g.X = cc.gate; g.M = M; g.N = D; g.K = F;
        g.resid_in = cc.x2; g.out_f32 = last ? T->xlast : T->c[l + 1].xin; g.ldo = D; g.alpha = alpha;
        set_sk(ctx, g);
        const float* ng = last ? ctx->gfinal : ctx->L[l + 1].g1;
        f16* nxn = last ? T->xf : T->c[l + 1].xn;
        RCK(timed(ctx, RH_K_GEMM_W2, [&] { return rh::launch_gemm_resid_norm(g, ng, c.rms_eps, nxn, st); }));
    }
    return enqueue_tail(ctx, B, S, true, T->xf, T->fwd_softcap);
}

// dgamma (+)= kappa * the partial sums of rms_backward (stores while the
// gradients are logically zero).
int gamma_grad(rh_ctx* ctx, int nblk, int D, float kappa, float* dgamma) {
    LCK(rh::launch_dgamma_reduce(ctx->train->dgp, nblk, D, kappa, dgamma, ctx->train->zero, ctx->stream));
    return RH_OK;
}

// C[rows][cols] += kappa * X W^T with X [rows][Mp], W [cols][Mp] (token-inner).
// When every gradient is still zero the epilogue stores kappa * acc instead
// (the same values; it skips reading the fp32 gradient back).  The tile model
// picks the tile (no stream-K: its workspace belongs to the main stream's
// GEMMs); its picks at K = 4096, accumulating, against the best of the other
// tiles (us): 4096 x 4096 256x256 112 | 122, 4096 x 11008 256x256 355 | 394,
// 8192 x 4096 256x256 223 | 252; 1024 x 1024 128x128 28 | 39, 1024 x 2816
// 128x128 31 | 40, 8192 x 1024 256x128 62 | 68.  A short K after a zero leaves
// the fp32 output most of the time; large outputs then take the kernel whose
// store waves write a tile while the next one is computed.
// trx, trw > 0: X and W are token-major instead, [Mp][trx] and [Mp][trw].
int grad_gemm(rh_ctx* ctx, const f16* X, const f16* W, int rows, int cols, float kappa, float* out,
              hipStream_t st, int trx = 0, int trw = 0) {
    rh::GemmArgs g{};
    g.trx = trx; g.trw = trw;
    g.X = X; g.W = W; g.M = rows; g.N = cols; g.K = ctx->train->Mp;
    g.out_f32 = out; g.ldo = cols; g.alpha = kappa;
    g.nt_out = true;  // read only by the optimizer
    if (store_waves(ctx, rows, cols)) {
        LCK(rh::launch_gemm_wgrad(g, false, st));
        return RH_OK;
    }
    LCK(rh::launch_gemm(ctx->train->zero ? rh::EPI_F32 : rh::EPI_RESID, g, st));
    return RH_OK;
}

// Whether n (2 or 3) gradients [rows][cols] of one X (dWq | dWk | dWv and dW1 |
// dW3) run as one product with n outputs: where that fills the CUs better than
// n products (the tile model's estimate): 1024 wide at K = 4096, dWq..dWv 85 ->
// 32 us, dW1 dW3 62 -> 50; 4096 wide three products of one round each stay (334
// against 358 us).  Outputs whose first store the
// store-wave kernel takes stay n products up to 512 tokens, where writing them
// is most of the time: forward + backward of two layers after a zero, joint ->
// n products, 128 - 512 tokens: 2560 wide 0 - 2% faster, 3072 wide 1 - 4% (512
// tokens 1510 -> 1455 us), 5120 wide 6% (128 tokens, 1750 -> 1652 us) to -1%
// (512); at 1024 tokens 3072 wide 1% faster, 5120 wide 4% slower.
bool joint(const rh_ctx* ctx, int rows, int cols, int n) {
    if (n == 1 || (ctx->train->Mp <= 512 && store_waves(ctx, rows, cols))) return false;
    return rh::gemm_tile_cost(rows, n * cols) < (float)n * rh::gemm_tile_cost(rows, cols);
}

// n gradients [rows][cols] of one X, the W of each after the other.
int grad_gemms(rh_ctx* ctx, const f16* X, const f16* W, int rows, int cols, float kappa, float* const* out, int n,
               hipStream_t st, int trx = 0, int trw = 0) {
    if (!joint(ctx, rows, cols, n)) {
        for (int j = 0; j < n; ++j)
            RCK(grad_gemm(ctx, X, W + (size_t)j * cols * (trw ? 16 : ctx->train->Mp), rows, cols, kappa, out[j], st,
                          trx, trw));
        return RH_OK;
    }
    rh::GemmArgs g{};
    g.X = X; g.W = W; g.M = rows; g.N = n * cols; g.K = ctx->train->Mp;
    g.out_f32 = out[0]; g.out_part1 = out[1]; g.out_part2 = n > 2 ? out[2] : nullptr;
    g.part_cols = g.ldo = cols; g.alpha = kappa;
    g.trx = trx; g.trw = trw;
    g.nt_out = true;
    LCK(rh::launch_gemm(ctx->train->zero ? rh::EPI_F32 : rh::EPI_RESID, g, st));
    return RH_OK;
}

// out [M][N] fp32 = A W^T with A [M][K] and W [N][K] (fragment order).
// As the sum of *nsplit fp32 partials at *parts, M * N floats apart: K split
// into the stream-K workspace when the output has too few tiles to fill the
// CUs (the consuming row kernel adds them up, so no fix-up kernel runs),
// otherwise the whole product in out (*nsplit = 1).
int data_gemm(rh_ctx* ctx, const f16* A, const f16* W, int M, int N, int K, float* out, const float** parts,
              int* nsplit) {
    rh::GemmArgs g{};
    g.X = A; g.W = W; g.M = M; g.N = N; g.K = K;
    g.out_f32 = out; g.ldo = N;
    set_sk(ctx, g);
    LCK(rh::launch_gemm_partials(g, nsplit, ctx->stream));
    if (*nsplit >= 2) {
        *parts = ctx->sk_part;
        return RH_OK;
    }
    LCK(rh::launch_gemm(rh::EPI_F32, g, ctx->stream));
    *parts = out;
    *nsplit = 1;
    return RH_OK;
}

int enqueue_backward(rh_ctx* ctx, int B, int S, float loss_scale, int nuniq) {
    TrainState* T = ctx->train;
    const rh_config& c = ctx->cfg;
    const int M = B * S, D = c.dim, F = c.hidden, V = c.vocab, Vp = (int)round_up(V, 128), Mp = T->Mp;
    const int H = c.heads, hd = c.head_dim;
    const float alpha = 1.0f / std::sqrt(2.0f * (float)c.nlayers);
    const float kappa = loss_scale / ((float)S * rh::GRAD_UNIT);
    const int nblk = rh::rms_backward_blocks(M, D);
    hipStream_t st = ctx->stream;
    // Main stream: the chain through the data gradients.  Side stream: the
    // weight gradients, each group after the activation
    // gradient it reads is written (ready) and before that buffer is rewritten
    // a layer later (read).  No buffer either stream writes is touched by the
    // other until the event that orders them.
    hipStream_t sd = T->side;
    for (hipEvent_t e : T->read) HCK(hipEventRecord(e, sd));  // nothing read yet
    auto publish = [&](int g) -> int {  // main -> side: group g's input is written
        HCK(hipEventRecord(T->ready[g], st));
        HCK(hipStreamWaitEvent(sd, T->ready[g], 0));
        return RH_OK;
    };
    auto rewrite = [&](int g) -> int {  // main waits: the side has copied group g's input
        HCK(hipStreamWaitEvent(st, T->read[g], 0));
        return RH_OK;
    };
    // CE gradient (internal units), dx_final = dl E, dembed += dl^T x_final
    LCK(rh::launch_ce_backward(ctx->logits, ctx->d_tgt, T->dlh, M, V, Vp, T->fwd_softcap, rh::GRAD_UNIT, st));
    RCK(publish(4));
    // Weight gradients contract over tokens.  With whole 128-token blocks the
    // tile kernels read the token-major activations and their gradients in place
    // (then read[g] is the GEMM's end); otherwise the rows past the last token
    // have to be zeros and the GEMMs take padded token-inner copies.  From 1000
    // tokens on that is 1 - 6% of a pass at nearly every width (512 - 4096; 20
    // layers of 4096, 8 x 512 accumulated: 98.2 -> 95.3 ms), at 128 - 768 tokens -3
    // to 8% at 512 - 4096 wide; a chain of the smallest kernels loses, since the
    // main stream then waits for the product instead of its copy (8 layers, 128
    // tokens: 512 wide 8%, 128 wide 12%).  The store-wave kernel keeps the copies: two
    // transposing reads for each of its 128x128 tile's operands take 4096 x
    // 11008 x 512 from 72 to 93 us beside the other stream (20 layers of 4096
    // after a zero, 1 x 512: 19.7 ms in place, 18.7 with copies).
    auto in_place = [&](int rows, int cols, int n) {
        return M == Mp && (joint(ctx, rows, cols, n) || !store_waves(ctx, rows, cols));
    };
    auto grads = [&](int g, const f16* X, int nx, f16* Xt, const f16* W, int nw, f16* Wt, int rows, int cols,
                     float* const* out, int n) -> int {
        const bool tr = in_place(rows, cols, n);
        if (!tr) {
            LCK(rh::launch_transpose_frag2(X, Xt, M, nx, W, Wt, M, nw, Mp, sd));
            if (g >= 0) HCK(hipEventRecord(T->read[g], sd));
            X = Xt;
            W = Wt;
        }
        RCK(grad_gemms(ctx, X, W, rows, cols, kappa, out, n, sd, tr ? nx : 0, tr ? nw : 0));
        if (tr && g >= 0) HCK(hipEventRecord(T->read[g], sd));
        return RH_OK;
    };
    RCK(grads(-1, T->dlh, Vp, T->dlT, T->xf, D, T->tx[0][0], V, D, &T->dembed, 1));
    const size_t MD = (size_t)M * D;  // stride of the data-gradient partials
    const float* dp;
    int ns;
    RCK(data_gemm(ctx, T->dlh, T->embed_t, M, D, Vp, T->gout, &dp, &ns));
    // final RMSNorm backward: dy -> dres, a*dy -> H1 (the last layer's dffn)
    LCK(rh::launch_rms_backward(dp, ns, MD, T->xlast, ctx->gfinal, nullptr, T->dres, T->H1, alpha, T->dgp, M, D,
                                c.rms_eps, st));
    RCK(gamma_grad(ctx, nblk, D, kappa, T->dgf));
    for (int l = c.nlayers - 1; l >= 0; --l) {
        const Layer& W = ctx->L[l];
        const TrainState::Cache& cc = T->c[l];
        const TrainState::WT& wt = T->wt[l];
        float* const* G = T->dlay[l].data();
        // dW2 += dffn^T gate (side); dgate = dffn W2 with the SiLU backward -> [dh1 | dh3]
        RCK(publish(0));
        RCK(grads(0, T->H1, D, T->tx[0][0], cc.gate, F, T->tx[0][1], D, F, G + 6, 1));
        RCK(rewrite(1));
        {
            rh::GemmArgs g{};
            g.X = T->H1; g.W = wt.w2t; g.M = M; g.N = F; g.K = D;
            g.h13 = cc.h13; g.out_f16 = T->H2; g.ldo = F;
            set_sk(ctx, g);
            LCK(rh::launch_gemm(rh::EPI_SILU_BWD, g, st));
        }
        // dx_ffn = [dh1 | dh3] [W1 | W3]^T; dW1, dW3 += x2n^T dh (side)
        RCK(publish(1));
        RCK(grads(1, cc.x2n, D, T->tx[1][0], T->H2, 2 * F, T->tx[1][1], D, F, G + 4, 2));
        RCK(data_gemm(ctx, T->H2, wt.w13t, M, D, 2 * F, T->gout, &dp, &ns));
        // dx2 = RMSNorm2'(dx_ffn) + dy (in place in dres); a*dx2 -> H1m
        RCK(rewrite(2));
        LCK(rh::launch_rms_backward(dp, ns, MD, cc.x2, W.g2, T->dres, T->dres, T->H1m, alpha, T->dgp, M, D,
                                    c.rms_eps, st));
        RCK(gamma_grad(ctx, nblk, D, kappa, G[8]));
        // da = (a dx2) Wo^T; dWo += attn^T (a dx2) (side)
        RCK(publish(2));
        RCK(grads(2, cc.attn, D, T->tx[2][0], T->H1m, D, T->tx[2][1], D, D, G + 3, 1));
        RCK(data_gemm(ctx, T->H1m, wt.ot, M, D, D, T->gout, &dp, &ns));
        // attention backward -> dq | dk | dv with the RoPE backward, as the fp16
        // operand H2q (rewritten: the side stream has copied the previous layer's)
        RCK(rewrite(3));
        LCK(rh::launch_attn_backward(cc.q, cc.k, cc.v, cc.attn, dp, ns, MD, cc.lse, T->dOh, T->Drow, T->H2q,
                                     ctx->rope, B, H, S, hd, st));
        // dxn = dqkv [Wq | Wk | Wv]^T; dWq, dWk, dWv += xn^T d{q,k,v} (side)
        RCK(publish(3));
        RCK(grads(3, cc.xn, D, T->tx[3][0], T->H2q, 3 * D, T->tx[3][1], D, D, G, 3));
        RCK(data_gemm(ctx, T->H2q, wt.qkvt, M, D, 3 * D, T->gout, &dp, &ns));
        // dy' = RMSNorm1'(dxn) + dx2 (in place); a*dy' -> H1 (the next layer's dffn)
        RCK(rewrite(0));
        LCK(rh::launch_rms_backward(dp, ns, MD, cc.xin, W.g1, T->dres, T->dres, T->H1, alpha, T->dgp, M, D,
                                    c.rms_eps, st));
        RCK(gamma_grad(ctx, nblk, D, kappa, G[7]));
    }
    // every weight gradient is written before anything after the backward reads them
    HCK(hipEventRecord(T->ready[4], sd));
    HCK(hipStreamWaitEvent(st, T->ready[4], 0));
    LCK(rh::launch_embed_backward(T->dres, T->utok, T->ustart, T->uidx, nuniq, kappa, T->dembed, D, st));
    T->zero = false;
    return RH_OK;
}

const size_t* tensor_sizes(const rh_config& c, size_t out[9]) {
    const size_t D = c.dim, F = c.hidden;
    const size_t sz[9] = {D * D, D * D, D * D, D * D, D * F, D * F, D * F, D, D};
    std::copy(sz, sz + 9, out);
    return out;
}

}  // namespace

// fp32 master weights (reference orientation), allocated together: the
// tensors are published only once every allocation has succeeded, so a
// failed call leaves no partial set behind for a later call to mistake for
// a complete one.
int rhrt::ensure_masters(rh_ctx* ctx) {
    RCK(ensure_train_host(ctx));
    TrainState* T = ctx->train;
    if (!T->opt) {
        T->opt = new (std::nothrow) TrainState::Opt;
        if (!T->opt) return fail(ctx, RH_ENOMEM, "out of host memory");
    }
    auto* o = T->opt;
    if (o->emb) return RH_OK;
    const rh_config& c = ctx->cfg;
    size_t sz[9];
    tensor_sizes(c, sz);
    float* emb = nullptr;
    std::vector<std::array<float*, 7>> w(c.nlayers);
    for (auto& a : w) a.fill(nullptr);
    int rc = dalloc(ctx, &emb, (size_t)c.vocab * c.dim);
    for (int l = 0; l < c.nlayers && rc == RH_OK; ++l)
        for (int j = 0; j < 7 && rc == RH_OK; ++j) rc = dalloc(ctx, &w[l][j], sz[j]);
    if (rc != RH_OK) {
        dfree(ctx, emb);
        for (auto& a : w)
            for (float* p : a) dfree(ctx, p);
        return rc;
    }
    o->w = std::move(w);
    o->emb = emb;
    o->synced = 0;  // nothing written yet
    return RH_OK;
}

bool rhrt::have_masters(const rh_ctx* ctx) { return ctx->train && ctx->train->opt && ctx->train->opt->emb; }

float* rhrt::master_ptr(rh_ctx* ctx, int l, int j) {
    return j < 0 ? ctx->train->opt->emb : ctx->train->opt->w[l][j];
}

// Frees the masters (no optimizer moments may exist: they belong together).
int rhrt::drop_masters(rh_ctx* ctx) {
    if (!have_masters(ctx)) return RH_OK;
    auto* o = ctx->train->opt;
    if (o->moments) return fail(ctx, RH_ESTATE, "the optimizer state holds the fp32 masters");
    HCK(hipStreamSynchronize(ctx->stream));
    dfree(ctx, o->emb);
    o->emb = nullptr;
    for (auto& a : o->w)
        for (float* p : a) dfree(ctx, p);
    o->w.clear();
    o->synced = 0;
    return RH_OK;
}

// Zeroes the moments (ModelOptState::zeros).
int rhrt::zero_moments(rh_ctx* ctx) {
    auto* o = ctx->train->opt;
    const rh_config& c = ctx->cfg;
    size_t sz[9];
    tensor_sizes(c, sz);
    hipStream_t st = ctx->stream;
    const size_t VD = (size_t)c.vocab * c.dim;
    LCK(rh::launch_fill_f32(o->emb_m, 0.f, VD, st));
    LCK(rh::launch_fill_f32(o->emb_v, 0.f, VD, st));
    LCK(rh::launch_fill_f32(o->gf_m, 0.f, c.dim, st));
    LCK(rh::launch_fill_f32(o->gf_v, 0.f, c.dim, st));
    for (int l = 0; l < c.nlayers; ++l)
        for (int j = 0; j < 9; ++j) {
            LCK(rh::launch_fill_f32(o->m[l][j], 0.f, sz[j], st));
            LCK(rh::launch_fill_f32(o->v[l][j], 0.f, sz[j], st));
        }
    return RH_OK;
}

namespace {

// Optimizer state: masters, moments (zeroed when created) and the norm's
// partials.  Masters older than the device weights (rh_init_weights_normal)
// are re-read from the fp16 device copy.
int ensure_opt(rh_ctx* ctx) {
    RCK(ensure_train_static(ctx));
    RCK(ensure_masters(ctx));
    TrainState* T = ctx->train;
    auto* o = T->opt;
    const rh_config& c = ctx->cfg;
    const size_t D = c.dim, V = c.vocab;
    size_t sz[9];
    tensor_sizes(c, sz);
    hipStream_t st = ctx->stream;
    if (!o->moments) {
        auto once = [&](float*& p, size_t n) { return p ? RH_OK : dalloc(ctx, &p, n); };
        RCK(once(o->emb_m, V * D));
        RCK(once(o->emb_v, V * D));
        RCK(once(o->gf_m, D));
        RCK(once(o->gf_v, D));
        o->m.resize(c.nlayers);
        o->v.resize(c.nlayers);
        for (int l = 0; l < c.nlayers; ++l)
            for (int j = 0; j < 9; ++j) {
                RCK(once(o->m[l][j], sz[j]));
                RCK(once(o->v[l][j], sz[j]));
            }
        o->moments = true;
        RCK(zero_moments(ctx));
    }
    if (o->synced != ctx->wgen) {
        LCK(rh::launch_unpack_rows(ctx->embed, o->emb, (int)V, (int)D, st));
        for (int l = 0; l < c.nlayers; ++l)
            for (int j = 0; j < 7; ++j) {
                const TensorMap mp = layer_map(ctx, l, j);
                if (mp.map < 0) {
                    LCK(rh::launch_unpack_rows(mp.dst, o->w[l][j], mp.R, mp.C, st));
                } else {
                    LCK(rh::launch_unpack_transpose(mp.dst, o->w[l][j], mp.R, mp.C, mp.ldd, mp.map, mp.row_off, st));
                }
            }
        o->synced = ctx->wgen;
    }
    return RH_OK;
}

// 1 - b^t in fp32 by repeated squaring (f32::powi of the bias corrections).
float powi_f32(float b, uint32_t t) {
    float r = 1.0f, x = b;
    for (uint32_t e = t; e; e >>= 1) {
        if (e & 1u) r *= x;
        x *= x;
    }
    return r;
}

}  // namespace

extern "C" {

void rh_train_config_default(rh_train_config* tc) {
    if (!tc) return;
    *tc = rh_train_config{3e-4f, 0.1f, 100u, 10000u, 0.9f, 0.95f, 1e-8f, 0.1f, 0.05f, 5.0f, 256.0f, 10u, 1.0f, 0.0f};
}

float rh_learning_rate(uint32_t step, const rh_train_config* tc) {
    if (!tc) return 0.f;
    if (step < tc->warmup_steps) return tc->max_lr * (float)(step + 1) / (float)tc->warmup_steps;
    const float decay = (float)(step - tc->warmup_steps) / (float)(tc->total_steps - tc->warmup_steps);
    const float min_lr = tc->max_lr * tc->min_lr_frac;
    return min_lr + 0.5f * (1.0f + std::cos(3.14159265358979323846f * decay)) * (tc->max_lr - min_lr);
}

int rh_grad_norm(rh_ctx* ctx, float* norm_out) {
    if (!ctx || !norm_out) return fail(ctx, RH_EINVAL, "null argument");
    TrainState* T = ctx->train;
    if (!T || !T->have_static || T->zero) {
        *norm_out = 0.f;
        return RH_OK;
    }
    HCK(hipSetDevice(ctx->device));
    const rh_config& c = ctx->cfg;
    size_t sz[9];
    tensor_sizes(c, sz);
    hipStream_t st = ctx->stream;
    // grad_norm's tensor order (full_model.rs:1403-1450)
    std::vector<std::pair<const float*, size_t>> ts{{T->dembed, (size_t)c.vocab * c.dim}, {T->dgf, (size_t)c.dim}};
    for (int l = 0; l < c.nlayers; ++l)
        for (int j = 0; j < 9; ++j) ts.emplace_back(T->dlay[l][j], sz[j]);
    // per-block partials of every tensor, then their sum in double on the device
    size_t off = 0;
    for (auto& t : ts) {
        LCK(rh::launch_sumsq(t.first, t.second, T->norm_part + off, st));
        off += rh::sumsq_blocks(t.second);
    }
    LCK(rh::launch_sum_parts(T->norm_part, off, T->norm_sum, st));
    double total = 0.0;
    HCK(hipMemcpyAsync(&total, T->norm_sum, sizeof(double), hipMemcpyDeviceToHost, st));
    HCK(hipStreamSynchronize(st));
    *norm_out = (float)std::sqrt(total);
    return RH_OK;
}

int rh_update_weights(rh_ctx* ctx, uint32_t t, float lr, const rh_train_config* tc, float grad_scale) {
    if (!ctx || !tc) return fail(ctx, RH_EINVAL, "null argument");
    if (t == 0) return fail(ctx, RH_EINVAL, "the Adam step count t starts at 1");
    HCK(hipSetDevice(ctx->device));
    RCK(ensure_opt(ctx));
    TrainState* T = ctx->train;
    auto* o = T->opt;
    const rh_config& c = ctx->cfg;
    const size_t D = c.dim, V = c.vocab;
    size_t sz[9];
    tensor_sizes(c, sz);
    hipStream_t st = ctx->stream;
    const bool zg = T->zero;  // gradients logically zero: no grad reads
    rh::AdamArgs a{};
    a.beta1 = tc->beta1;
    a.beta2 = tc->beta2;
    a.omb1 = 1.0f - tc->beta1;
    a.omb2 = 1.0f - tc->beta2;
    a.eps = tc->eps;
    a.gscale = grad_scale;
    a.bc1 = 1.0f / (1.0f - powi_f32(tc->beta1, t));
    a.bc2 = 1.0f / (1.0f - powi_f32(tc->beta2, t));
    // update_weights (full_model.rs:1123-1241): embed at lr * embed_lr_scale, gamma_final at lr, no decay
    rh::AdamArgs ae = a;
    ae.lr = lr * tc->embed_lr_scale;
    ae.wd = 0.f;
    LCK(rh::launch_adam_rows(o->emb, zg ? nullptr : T->dembed, o->emb_m, o->emb_v, V * D, ae, ctx->embed, (int)D,
                             st));
    rh::AdamArgs ag = a;
    ag.lr = lr;
    ag.wd = 0.f;
    LCK(rh::launch_adam_rows(ctx->gfinal, zg ? nullptr : T->dgf, o->gf_m, o->gf_v, D, ag, nullptr, 0, st));
    // update_layer (:1243-1400): matrices at lr * matrix_lr_scale with decay, gammas at lr without
    rh::AdamArgs am = a;
    am.lr = lr * tc->matrix_lr_scale;
    am.wd = tc->weight_decay;
    for (int l = 0; l < c.nlayers; ++l) {
        for (int j = 0; j < 7; ++j) {
            const TensorMap mp = layer_map(ctx, l, j);
            const float* g = zg ? nullptr : T->dlay[l][j];
            if (mp.map < 0) {
                LCK(rh::launch_adam_rows(o->w[l][j], g, o->m[l][j], o->v[l][j], sz[j], am, mp.dst, mp.C, st));
            } else {
                LCK(rh::launch_adam_transpose(o->w[l][j], g, o->m[l][j], o->v[l][j], mp.R, mp.C, am, mp.dst,
                                              mp.ldd, mp.map, mp.row_off, st));
            }
        }
        LCK(rh::launch_adam_rows(ctx->L[l].g1, zg ? nullptr : T->dlay[l][7], o->m[l][7], o->v[l][7], D, ag,
                                 nullptr, 0, st));
        LCK(rh::launch_adam_rows(ctx->L[l].g2, zg ? nullptr : T->dlay[l][8], o->m[l][8], o->v[l][8], D, ag,
                                 nullptr, 0, st));
    }
    HCK(hipStreamSynchronize(st));
    ++ctx->wgen;  // the transposed copies of the backward are rebuilt on its next call
    o->synced = ctx->wgen;
    return RH_OK;
}

}  // extern "C"

namespace {
int train_step_body(rh_ctx* ctx, const rh_tokens* data, uint32_t step, const rh_train_config* tc,
                    uint64_t max_pos, float* loss_out, float* grad_norm_out);
int forward_backward_impl(rh_ctx* ctx, const uint32_t* tokens, const uint32_t* targets, int batch, int seq,
                          float softcap, float loss_scale, float* mean_loss_out);
}  // namespace

extern "C" {

int rh_train_step(rh_ctx* ctx, const rh_tokens* data, uint32_t step, const rh_train_config* tc, float* loss_out,
                  float* grad_norm_out) {
    if (!ctx || !data || !tc) return fail(ctx, RH_EINVAL, "null argument");
    if (tc->accum_steps == 0 || !(tc->loss_scale > 0.f))
        return fail(ctx, RH_EINVAL, "accum_steps must be >= 1 and loss_scale > 0");
    const int S = ctx->cfg.seq;
    const int64_t n = rh_tokens_len(data);
    if (n < (int64_t)S + 2) return fail(ctx, RH_ERANGE, "token data shorter than seq + 2");
    const uint64_t max_pos = (uint64_t)(n - S - 1);
    // The training forward uses tc->softcap; the context's own softcap (the
    // one forwards and decodes use) is not touched.
    const int rc = train_step_body(ctx, data, step, tc, max_pos, loss_out, grad_norm_out);
    return rc;
}

}  // extern "C"

namespace {

int train_step_body(rh_ctx* ctx, const rh_tokens* data, uint32_t step, const rh_train_config* tc,
                    uint64_t max_pos, float* loss_out, float* grad_norm_out) {
    const int S = ctx->cfg.seq;
    RCK(rh_zero_grads(ctx));
    // train_step_with_options (full_model.rs:1510-1600): accum_steps sequences
    // at pseudo-random positions (step*7919 + micro*104729) % max_pos, run as
    // batches of up to max_batch independent sequences.
    const int mb = std::max(1, std::min<int>((int)tc->accum_steps, ctx->max_batch));
    std::vector<uint32_t> buf((size_t)S + 1), tok((size_t)mb * S), tgt((size_t)mb * S);
    std::vector<float> losses(mb);
    float total = 0.f;
    for (uint32_t i0 = 0; i0 < tc->accum_steps; i0 += mb) {
        const int nb = std::min<int>(mb, (int)(tc->accum_steps - i0));
        for (int j = 0; j < nb; ++j) {
            const uint64_t pos = ((uint64_t)step * 7919u + (uint64_t)(i0 + j) * 104729u) % max_pos;
            RCK(rh_tokens_read(data, (int64_t)pos, S + 1, buf.data()));
            std::memcpy(&tok[(size_t)j * S], buf.data(), (size_t)S * 4);
            std::memcpy(&tgt[(size_t)j * S], buf.data() + 1, (size_t)S * 4);
        }
        RCK(forward_backward_impl(ctx, tok.data(), tgt.data(), nb, S, tc->softcap, tc->loss_scale, losses.data()));
        for (int j = 0; j < nb; ++j) total += losses[j];
    }
    const float gsc = 1.0f / ((float)tc->accum_steps * tc->loss_scale);
    float raw = 0.f;
    RCK(rh_grad_norm(ctx, &raw));
    const float scaled = raw * gsc;
    const float combined = scaled > tc->grad_clip ? tc->grad_clip / raw : gsc;
    RCK(rh_update_weights(ctx, step + 1, rh_learning_rate(step, tc), tc, combined));
    if (loss_out) *loss_out = total / (float)tc->accum_steps;
    if (grad_norm_out) *grad_norm_out = scaled;
    return RH_OK;
}

}  // namespace

extern "C" {

// Zeroing is logical: the next backward's weight-gradient GEMMs and gamma
// reductions store instead of accumulating, and reads return zeros until
// then, so no pass over the gradient memory is needed.
int rh_zero_grads(rh_ctx* ctx) {
    if (!ctx) return RH_EINVAL;
    TrainState* T = ctx->train;
    if (!T) return RH_OK;  // nothing allocated yet: the first backward starts from zero
    T->zero = true;
    return RH_OK;
}

}  // extern "C"

namespace {

// Host-built index of the embedding backward: every distinct token and its
// positions, in increasing order.
struct TokenIndex {
    std::vector<uint32_t> utok;
    std::vector<int> start{0}, idx;
};

// Radix sort of the positions by token id, 11 bits a pass, so that the time
// goes with the tokens and not with the vocabulary (whose ids the caller
// checked): the GPU is idle until this is done.  16, 128, 512 and 4096 tokens of
// a vocabulary of 32000, us: 2, 3, 6 and 34; a counting sort over the whole
// vocabulary 86, 87, 94 and 99; a map of position lists 2, 13, 60 and 543.
void build_index(const uint32_t* tokens, int M, int vocab, TokenIndex& ix) {
    constexpr int BITS = 11, R = 1 << BITS;
    std::vector<int> next(M);
    ix.idx.resize(M);
    for (int i = 0; i < M; ++i) ix.idx[i] = i;
    for (int sh = 0; sh == 0 || (uint64_t)(vocab - 1) >> sh; sh += BITS) {
        int at[R + 1] = {};
        auto digit = [&](int i) { return (tokens[i] >> sh) & (R - 1); };
        for (int i = 0; i < M; ++i) ++at[digit(i) + 1];
        for (int d = 0; d < R; ++d) at[d + 1] += at[d];
        for (int i : ix.idx) next[at[digit(i)]++] = i;
        ix.idx.swap(next);
    }
    for (int i = 0; i < M; ++i) {
        const uint32_t t = tokens[ix.idx[i]];
        if (i == 0 || t != ix.utok.back()) {
            if (i) ix.start.push_back(i);
            ix.utok.push_back(t);
        }
    }
    ix.start.push_back(M);
}

// Checks a training forward's arguments and sizes every buffer it needs.
int prepare_train(rh_ctx* ctx, const uint32_t* tokens, const uint32_t* targets, int batch, int seq, float softcap) {
    if (!ctx || !tokens || !targets) return fail(ctx, RH_EINVAL, "null argument");
    if (batch <= 0 || seq <= 0 || batch > ctx->max_batch)
        return fail(ctx, RH_ERANGE, "batch must be in [1, max_batch] and seq >= 1");
    if (!(softcap >= 0.f) || !std::isfinite(softcap)) return fail(ctx, RH_EINVAL, "softcap must be >= 0");
    const rh_config& c = ctx->cfg;
    if (c.hidden % 64 != 0) return fail(ctx, RH_EINVAL, "the backward pass needs hidden % 64 == 0");
    const size_t M = (size_t)batch * seq;
    RCK(check_tokens(ctx, tokens, M));
    RCK(check_tokens(ctx, targets, M));
    HCK(hipSetDevice(ctx->device));
    RCK(ensure_workspace(ctx, (int)M));
    RCK(ensure_rope(ctx, seq));
    RCK(ensure_train_static(ctx));
    RCK(ensure_train_ws(ctx, batch, seq));
    RCK(ensure_copies(ctx));
    RCK(ensure_packs(ctx));
    return RH_OK;
}

// Uploads the tokens, targets and the embedding backward's index (ix must
// stay alive until the stream has drained) and enqueues the training forward
// whose caches the backward reads; records it as the kept forward.
int enqueue_kept_forward(rh_ctx* ctx, const uint32_t* tokens, const uint32_t* targets, int batch, int seq,
                         float softcap, TokenIndex& ix) {
    TrainState* T = ctx->train;
    hipStream_t st = ctx->stream;
    const size_t M = (size_t)batch * seq;
    build_index(tokens, (int)M, ctx->cfg.vocab, ix);
    HCK(hipMemcpyAsync(ctx->d_tok, tokens, M * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    HCK(hipMemcpyAsync(ctx->d_tgt, targets, M * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    HCK(hipMemcpyAsync(T->utok, ix.utok.data(), ix.utok.size() * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    HCK(hipMemcpyAsync(T->ustart, ix.start.data(), ix.start.size() * sizeof(int), hipMemcpyHostToDevice, st));
    HCK(hipMemcpyAsync(T->uidx, ix.idx.data(), ix.idx.size() * sizeof(int), hipMemcpyHostToDevice, st));
    T->fwd_softcap = softcap;
    T->fwd_B = batch;
    T->fwd_S = seq;
    T->fwd_nuniq = (int)ix.utok.size();
    T->fwd_tokens.assign(tokens, tokens + M);
    T->fwd_epoch = ctx->work_epoch;
    T->fwd_id += 1;
    RCK(enqueue_forward_train(ctx, batch, seq));
    return RH_OK;
}

// The backward of the kept forward, accumulating into the gradients.
int enqueue_kept_backward(rh_ctx* ctx, float loss_scale) {
    TrainState* T = ctx->train;
    const int rc = enqueue_backward(ctx, T->fwd_B, T->fwd_S, loss_scale, T->fwd_nuniq);
    if (rc != RH_OK) (void)hipStreamSynchronize(T->side);  // leave no weight-gradient work behind
    return rc;
}

int forward_backward_impl(rh_ctx* ctx, const uint32_t* tokens, const uint32_t* targets, int batch, int seq,
                          float softcap, float loss_scale, float* mean_loss_out) {
    RCK(prepare_train(ctx, tokens, targets, batch, seq, softcap));
    if (!(loss_scale > 0.f) || !std::isfinite(loss_scale)) return fail(ctx, RH_EINVAL, "loss_scale must be > 0");
    TokenIndex ix;
    RCK(enqueue_kept_forward(ctx, tokens, targets, batch, seq, softcap, ix));
    RCK(enqueue_kept_backward(ctx, loss_scale));
    hipStream_t st = ctx->stream;
    if (mean_loss_out) HCK(hipMemcpyAsync(mean_loss_out, ctx->mean, batch * sizeof(float), hipMemcpyDeviceToHost, st));
    HCK(hipStreamSynchronize(st));
    return check_err_flag(ctx);
}

}  // namespace

struct rh_forward_result {
    const rh_ctx* ctx;
    uint64_t id;
};

extern "C" {

int rh_forward_backward(rh_ctx* ctx, const uint32_t* tokens, const uint32_t* targets, int batch, int seq,
                        float loss_scale, float* mean_loss_out) {
    if (!ctx) return RH_EINVAL;
    return forward_backward_impl(ctx, tokens, targets, batch, seq, ctx->cfg.softcap, loss_scale, mean_loss_out);
}

int rh_forward_train(rh_ctx* ctx, const uint32_t* tokens, const uint32_t* targets, int batch, int seq,
                     float softcap, float* mean_loss_out, rh_forward_result** out) {
    if (!out) return fail(ctx, RH_EINVAL, "null argument");
    *out = nullptr;
    RCK(prepare_train(ctx, tokens, targets, batch, seq, softcap));
    auto* r = new (std::nothrow) rh_forward_result{ctx, 0};
    if (!r) return fail(ctx, RH_ENOMEM, "out of host memory");
    TokenIndex ix;
    int rc = enqueue_kept_forward(ctx, tokens, targets, batch, seq, softcap, ix);
    hipStream_t st = ctx->stream;
    if (rc == RH_OK && mean_loss_out &&
        hipMemcpyAsync(mean_loss_out, ctx->mean, batch * sizeof(float), hipMemcpyDeviceToHost, st) != hipSuccess)
        rc = fail(ctx, RH_EDEVICE, "hipMemcpyAsync of the losses failed");
    if (hipStreamSynchronize(st) != hipSuccess && rc == RH_OK) rc = fail(ctx, RH_EDEVICE, "stream synchronize failed");
    if (rc == RH_OK) rc = check_err_flag(ctx);
    if (rc != RH_OK) {
        ctx->train->fwd_id += 1;  // nothing may consume a failed forward
        delete r;
        return rc;
    }
    r->id = ctx->train->fwd_id;
    *out = r;
    return RH_OK;
}

int rh_backward(rh_ctx* ctx, const rh_forward_result* fwd, const uint32_t* tokens, float softcap, float loss_scale,
                float* grad_norm_out) {
    if (!ctx || !fwd || !tokens) return fail(ctx, RH_EINVAL, "null argument");
    if (!(loss_scale > 0.f) || !std::isfinite(loss_scale)) return fail(ctx, RH_EINVAL, "loss_scale must be > 0");
    TrainState* T = ctx->train;
    if (fwd->ctx != ctx || !T || fwd->id != T->fwd_id || T->fwd_epoch != ctx->work_epoch)
        return fail(ctx, RH_ESTATE,
                    "the forward result is stale: another forward, prefill or validation has run on this "
                    "context since it was made, or it belongs to another context");
    if (softcap != T->fwd_softcap) return fail(ctx, RH_EINVAL, "softcap differs from the forward's");
    if (!std::equal(T->fwd_tokens.begin(), T->fwd_tokens.end(), tokens))
        return fail(ctx, RH_EINVAL, "tokens differ from the forward's input tokens");
    HCK(hipSetDevice(ctx->device));
    RCK(ensure_packs(ctx));  // the weights may have changed since the forward
    RCK(enqueue_kept_backward(ctx, loss_scale));
    HCK(hipStreamSynchronize(ctx->stream));
    if (grad_norm_out) RCK(rh_grad_norm(ctx, grad_norm_out));
    return RH_OK;
}

void rh_forward_result_free(rh_forward_result* fwd) { delete fwd; }

int rh_read_grads_f32(rh_ctx* ctx, float* dembed, float* dgamma_final, float* const* layer_grads) {
    if (!ctx) return RH_EINVAL;
    TrainState* T = ctx->train;
    if (!T || !T->have_static) return fail(ctx, RH_ESTATE, "no gradients: run rh_forward_backward first");
    HCK(hipSetDevice(ctx->device));
    const rh_config& c = ctx->cfg;
    const size_t D = c.dim, F = c.hidden, V = c.vocab;
    hipStream_t st = ctx->stream;
    const size_t sz[9] = {D * D, D * D, D * D, D * D, D * F, D * F, D * F, D, D};
    if (T->zero) {
        if (dembed) std::memset(dembed, 0, V * D * sizeof(float));
        if (dgamma_final) std::memset(dgamma_final, 0, D * sizeof(float));
        if (layer_grads)
            for (int l = 0; l < c.nlayers; ++l)
                for (int j = 0; j < 9; ++j)
                    if (layer_grads[9 * l + j]) std::memset(layer_grads[9 * l + j], 0, sz[j] * sizeof(float));
        return RH_OK;
    }
    if (dembed) HCK(hipMemcpyAsync(dembed, T->dembed, V * D * sizeof(float), hipMemcpyDeviceToHost, st));
    if (dgamma_final) HCK(hipMemcpyAsync(dgamma_final, T->dgf, D * sizeof(float), hipMemcpyDeviceToHost, st));
    if (layer_grads)
        for (int l = 0; l < c.nlayers; ++l)
            for (int j = 0; j < 9; ++j)
                if (layer_grads[9 * l + j])
                    HCK(hipMemcpyAsync(layer_grads[9 * l + j], T->dlay[l][j], sz[j] * sizeof(float),
                                       hipMemcpyDeviceToHost, st));
    HCK(hipStreamSynchronize(st));
    return RH_OK;
}

}  // extern "C"
