// Whole layers per call (host code only: every launch goes through the entry points of the other files).  A layer is nine
// to fifteen launches; issued one by one from Python each costs about 11 us of host time, more than most of them run for
// a short slice, so the chain is built here from one descriptor per layer.
#include "gemm_epilogue.h"

#include <cmath>

namespace tp {

enum { W_LN1_G, W_LN1_B, W_QKV, B_QKV, W_OUT, B_OUT, W_LN2_G, W_LN2_B, W_FC1, B_FC1, W_FC2, B_FC2 };

enum { LD_QKV, LD_OUT, LD_FC1, LD_FC2, LD_DENSE = -1 };

// weight: which of the layer's weights B is (its rows may be a column range of a wider matrix), LD_DENSE: none of them
static tp_gemm_desc gemm_desc(const tp_layer_desc& l, int op, int epi, int M, int N, int K, const void* A, const void* B, void* C,
                              int weight = LD_DENSE) {
    tp_gemm_desc d = {};
    d.op = op; d.dtype = l.dtype; d.epilogue = epi;
    d.M = M; d.N = N; d.K = K;
    d.A = A; d.lda = op == TP_GEMM_TN ? M : K;
    d.B = B; d.ldb = weight != LD_DENSE && l.ldw[weight] ? l.ldw[weight] : op == TP_GEMM_NT ? K : N;
    d.C = C; d.ldc = N;
    return d;
}

static tp_attn_desc attn_desc(const tp_layer_desc& l) {
    tp_attn_desc d = {};
    d.dtype = l.dtype; d.batch = l.batch; d.heads = l.heads; d.head_dim = l.hidden / l.heads;
    d.T = l.T; d.cache_len = l.cache_len; d.cache_rows = l.cache_rows;
    d.q = l.q; d.k_cache = l.k_cache; d.v_cache = l.v_cache; d.o = l.o; d.lse = l.lse;
    d.q_scale = (float)pow((double)d.head_dim, -0.5);
    return d;
}

static int validate_layer(const tp_layer_desc* l, const char* what) {
    if (!l) { set_error("%s: null descriptor", what); return TP_ERR_ARG; }
    if (l->T <= 0 || l->batch <= 0 || l->heads <= 0 || l->hidden <= 0 || l->ffn <= 0 || l->cache_len < 0 || l->hidden % l->heads ||
        l->cache_rows < (int64_t)l->cache_len + l->T || (l->activation != 0 && l->activation != 1)) {
        set_error("%s: bad sizes (T=%d batch=%d heads=%d hidden=%d ffn=%d cache_len=%d cache_rows=%ld activation=%d)", what,
                  l->T, l->batch, l->heads, l->hidden, l->ffn, l->cache_len, (long)l->cache_rows, l->activation);
        return TP_ERR_ARG;
    }
    for (int i = 0; i < 12; ++i)
        if (!l->w[i]) { set_error("%s: parameter %d is null", what, i); return TP_ERR_ARG; }
    if (!l->x || !l->k_cache || !l->v_cache || !l->xn || !l->mean1 || !l->rstd1 || !l->q || !l->o || !l->lse || !l->h || !l->mean2 ||
        !l->rstd2 || !l->hn || !l->a || (l->activation == 1 && !l->z) || !l->out) {
        set_error("%s: null buffer", what);
        return TP_ERR_ARG;
    }
    return TP_OK;
}

// A product whose k-split partial sums, if the plan splits, are left to the LayerNorm that reads C; splits: how many.
static int gemm_deferred(tp_gemm_desc d, void* ws, size_t bytes, void* stream, int* splits) {
    *splits = tp_gemm_splits(&d);
    if (*splits > 1) d.defer_reduce = 1;
    return tp_gemm(&d, ws, bytes, stream);
}

// A = LayerNorm(x), then the product d that reads it: one launch where the product takes the rows itself.
static int layernorm_then(const tp_gemm_desc& d, const LayerNormOf& ln, void* ws, size_t bytes, void* stream) {
    if (gemm_takes_layernorm(d, ln)) return gemm_of_layernorm(d, ln, 1e-5f, stream);
    const int rc = tp_layernorm_fwd(ln.x, ln.gamma, ln.beta, const_cast<void*>(d.A), ln.mean, ln.rstd, d.M, d.K, 1e-5f, d.dtype, stream);
    return rc != TP_OK ? rc : tp_gemm(&d, ws, bytes, stream);
}
static LayerNormOf first_layernorm(const tp_layer_desc& l) { return {l.x, l.w[W_LN1_G], l.w[W_LN1_B], l.mean1, l.rstd1}; }

struct ForwardPlan { tp_gemm_desc qkv, out, fc1, fc2; tp_attn_desc attn; };
static ForwardPlan forward_plan(const tp_layer_desc& l) {
    const int M = l.T * l.batch, E = l.hidden, F = l.ffn;
    ForwardPlan p;
    p.attn = attn_desc(l);
    p.qkv = gemm_desc(l, TP_GEMM_NT, TP_EPI_QKV_SCATTER, M, 3 * E, E, l.xn, l.w[W_QKV], nullptr, LD_QKV);
    p.qkv.bias = l.w[B_QKV];
    p.qkv.q = l.q; p.qkv.k_cache = l.k_cache; p.qkv.v_cache = l.v_cache;
    p.qkv.batch = l.batch; p.qkv.heads = l.heads; p.qkv.head_dim = E / l.heads;
    p.qkv.cache_len = l.cache_len; p.qkv.cache_rows = l.cache_rows; p.qkv.q_scale = p.attn.q_scale;
    p.out = gemm_desc(l, TP_GEMM_NT, TP_EPI_BIAS_RESIDUAL, M, E, E, l.o, l.w[W_OUT], l.h, LD_OUT);
    p.out.bias = l.w[B_OUT]; p.out.residual = l.x; p.out.ldr = E;
    p.fc1 = gemm_desc(l, TP_GEMM_NT, l.activation ? TP_EPI_BIAS_GELU : TP_EPI_BIAS_RELU, M, F, E, l.hn, l.w[W_FC1], l.a, LD_FC1);
    p.fc1.bias = l.w[B_FC1];
    if (l.activation) { p.fc1.aux_out = l.z; p.fc1.ldauxo = F; }
    p.fc2 = gemm_desc(l, TP_GEMM_NT, TP_EPI_BIAS_RESIDUAL, M, E, F, l.a, l.w[W_FC2], l.out, LD_FC2);
    p.fc2.bias = l.w[B_FC2]; p.fc2.residual = l.h; p.fc2.ldr = E;
    if (l.no_backward)
        for (tp_gemm_desc* d : {&p.qkv, &p.out, &p.fc1, &p.fc2}) d->reserved = kNoBackward;
    return p;
}

struct BackwardPlan { tp_gemm_desc dz1, dhn, d_o, dxn, wg[4]; };
static BackwardPlan backward_plan(const tp_layer_bwd_desc& b) {
    const tp_layer_desc& l = b.f;
    const int M = l.T * l.batch, E = l.hidden, F = l.ffn;
    BackwardPlan p;
    p.dz1 = gemm_desc(l, TP_GEMM_NN, l.activation ? TP_EPI_GELU_GRAD : TP_EPI_RELU_GRAD, M, F, E, b.dout, l.w[W_FC2], b.dz1, LD_FC2);
    p.dz1.aux = l.activation ? l.z : l.a; p.dz1.ldaux = F;
    p.dhn = gemm_desc(l, TP_GEMM_NN, TP_EPI_STORE, M, E, F, b.dz1, l.w[W_FC1], b.dhn, LD_FC1);
    p.d_o = gemm_desc(l, TP_GEMM_NN, TP_EPI_STORE, M, E, E, b.dh, l.w[W_OUT], b.d_o, LD_OUT);
    p.dxn = gemm_desc(l, TP_GEMM_NN, TP_EPI_STORE, M, E, 3 * E, b.dqkv, l.w[W_QKV], b.dxn, LD_QKV);
    const int K = (int)b.wg_rows, epi = b.wg_accumulate ? TP_EPI_ACCUMULATE : TP_EPI_STORE;
    p.wg[0] = gemm_desc(l, TP_GEMM_TN, epi, 3 * E, E, K, b.wg_dqkv, b.wg_xn, b.wg_out[0]);
    p.wg[1] = gemm_desc(l, TP_GEMM_TN, epi, E, E, K, b.wg_dh, b.wg_o, b.wg_out[1]);
    p.wg[2] = gemm_desc(l, TP_GEMM_TN, epi, F, E, K, b.wg_dz1, b.wg_hn, b.wg_out[2]);
    p.wg[3] = gemm_desc(l, TP_GEMM_TN, epi, E, F, K, b.wg_dout, b.wg_a, b.wg_out[3]);
    return p;
}

static size_t more(size_t a, size_t b) { return a > b ? a : b; }

}  // namespace tp

extern "C" size_t tp_layers_fwd_workspace_bytes(const tp_layer_desc* layers, int n) {
    size_t need = 0;
    for (int i = 0; layers && i < n; ++i) {
        const tp_layer_desc &l = layers[i], &f = layers[0];
        if (i && l.T == f.T && l.batch == f.batch && l.hidden == f.hidden && l.ffn == f.ffn && l.heads == f.heads &&
            l.cache_len == f.cache_len && l.dtype == f.dtype && l.activation == f.activation && !l.no_backward == !f.no_backward)
            continue;           // as the first one
        if (tp::validate_layer(&layers[i], "tp_layers_fwd") != TP_OK) return 0;
        const tp::ForwardPlan p = tp::forward_plan(layers[i]);
        for (const tp_gemm_desc* d : {&p.qkv, &p.out, &p.fc1, &p.fc2}) need = tp::more(need, tp_gemm_workspace_bytes(d));
        need = tp::more(need, tp_attn_fwd_workspace_bytes(&p.attn));
    }
    return need;
}

extern "C" int tp_layers_fwd(const tp_layer_desc* layers, int n, void* ws, size_t bytes, void* stream) {
    using namespace tp;
    if (!layers || n < 1) { set_error("tp_layers_fwd: no layers"); return TP_ERR_ARG; }
    for (int i = 0; i < n; ++i) {
        const int rc = validate_layer(&layers[i], "tp_layers_fwd");
        if (rc != TP_OK) return rc;
        if (i && (layers[i].x != layers[i - 1].out || layers[i].T != layers[0].T || layers[i].batch != layers[0].batch ||
                  layers[i].hidden != layers[0].hidden || layers[i].dtype != layers[0].dtype)) {
            set_error("tp_layers_fwd: layer %d does not continue layer %d", i, i - 1);
            return TP_ERR_ARG;
        }
    }
    int rc, pending = 1;        // k splits of the previous layer's fc2 whose sums are still to be added
    for (int i = 0; i < n; ++i) {
        const tp_layer_desc& l = layers[i];
        const int M = l.T * l.batch, E = l.hidden;
        const ForwardPlan p = forward_plan(l);
        if (pending > 1) {
            rc = tp_layernorm_fwd_partials((const float*)ws, pending, layers[i - 1].w[B_FC2], layers[i - 1].h, layers[i - 1].out,
                                           l.w[W_LN1_G], l.w[W_LN1_B], l.xn, l.mean1, l.rstd1, M, E, 1e-5f, l.dtype, stream);
            if (rc == TP_OK) rc = tp_gemm(&p.qkv, ws, bytes, stream);
        } else {
            rc = layernorm_then(p.qkv, first_layernorm(l), ws, bytes, stream);
        }
        if (rc != TP_OK) return rc;
        if ((rc = tp_attn_prefix_fwd(&p.attn, ws, bytes, stream)) != TP_OK) return rc;
        int splits;
        if ((rc = gemm_deferred(p.out, ws, bytes, stream, &splits)) != TP_OK) return rc;
        if (splits > 1) {
            rc = tp_layernorm_fwd_partials((const float*)ws, splits, l.w[B_OUT], l.x, l.h, l.w[W_LN2_G], l.w[W_LN2_B], l.hn, l.mean2,
                                           l.rstd2, M, E, 1e-5f, l.dtype, stream);
            if (rc == TP_OK) rc = tp_gemm(&p.fc1, ws, bytes, stream);
        } else {
            rc = layernorm_then(p.fc1, {l.h, l.w[W_LN2_G], l.w[W_LN2_B], l.mean2, l.rstd2}, ws, bytes, stream);
        }
        if (rc != TP_OK) return rc;
        // (a LayerNorm that its product takes has its sums in its own order: the layers of a chain take it as one alone does)
        pending = 1;
        if (i + 1 < n && !gemm_takes_layernorm(forward_plan(layers[i + 1]).qkv, first_layernorm(layers[i + 1])))
            rc = gemm_deferred(p.fc2, ws, bytes, stream, &pending);
        else
            rc = tp_gemm(&p.fc2, ws, bytes, stream);
        if (rc != TP_OK) return rc;
    }
    return TP_OK;
}

extern "C" size_t tp_layer_bwd_workspace_bytes(const tp_layer_bwd_desc* b) {
    if (!b || tp::validate_layer(&b->f, "tp_layer_bwd") != TP_OK) return 0;
    const tp::BackwardPlan p = tp::backward_plan(*b);
    size_t need = 0;
    for (const tp_gemm_desc* d : {&p.dz1, &p.dhn, &p.d_o, &p.dxn}) need = tp::more(need, tp_gemm_workspace_bytes(d));
    if (b->wg_rows)
        for (const tp_gemm_desc& d : p.wg) need = tp::more(need, tp_gemm_workspace_bytes(&d));
    return need;
}

extern "C" int tp_layer_bwd(const tp_layer_bwd_desc* b, void* ws, size_t bytes, void* stream) {
    using namespace tp;
    int rc = validate_layer(b ? &b->f : nullptr, "tp_layer_bwd");
    if (rc != TP_OK) return rc;
    if (!b->dout || !b->dz1 || !b->dhn || !b->dh || !b->d_o || !b->dqkv || !b->dxn || !b->dx || !b->delta || !b->small_acc) {
        set_error("tp_layer_bwd: null buffer");
        return TP_ERR_ARG;
    }
    if (b->f.no_backward) { set_error("tp_layer_bwd: the forward was asked for as one that no backward follows"); return TP_ERR_ARG; }
    const tp_layer_desc& l = b->f;
    const int M = l.T * l.batch, E = l.hidden, F = l.ffn;
    const BackwardPlan p = backward_plan(*b);
    int splits;
    if ((rc = tp_gemm(&p.dz1, ws, bytes, stream)) != TP_OK) return rc;
    if ((rc = gemm_deferred(p.dhn, ws, bytes, stream, &splits)) != TP_OK) return rc;
    if (splits > 1)
        rc = tp_layernorm_bwd_partials((const float*)ws, splits, b->dhn, l.h, l.mean2, l.rstd2, l.w[W_LN2_G], b->dout, b->dh, nullptr,
                                       nullptr, nullptr, nullptr, M, E, l.dtype, stream);
    else
        rc = tp_layernorm_bwd(b->dhn, l.h, l.mean2, l.rstd2, l.w[W_LN2_G], b->dout, b->dh, nullptr, nullptr, nullptr, nullptr, M, E,
                              l.dtype, stream);
    if (rc != TP_OK) return rc;
    if ((rc = tp_gemm(&p.d_o, ws, bytes, stream)) != TP_OK) return rc;
    tp_attn_desc at = attn_desc(l);
    at.d_o = b->d_o; at.delta = b->delta; at.dqkv = b->dqkv;
    at.dk_cache = b->dk_cache; at.dv_cache = b->dv_cache;
    at.grad_cache_dtype = b->dk_cache ? b->grad_cache_dtype : l.dtype;
    at.accumulate_prefix = b->accumulate_prefix; at.has_incoming = b->has_incoming; at.zero_slice_rows = b->zero_slice_rows;
    at.whole_grad_caches = b->whole_grad_caches;
    if (b->whole_grad_caches) { at.dk_in = b->dk_in; at.dv_in = b->dv_in; }
    if ((rc = tp_attn_prefix_bwd(&at, nullptr, 0, stream)) != TP_OK) return rc;
    if ((rc = gemm_deferred(p.dxn, ws, bytes, stream, &splits)) != TP_OK) return rc;
    if (splits > 1)
        rc = tp_layernorm_bwd_partials((const float*)ws, splits, b->dxn, l.x, l.mean1, l.rstd1, l.w[W_LN1_G], b->dh, b->dx, nullptr,
                                       nullptr, nullptr, nullptr, M, E, l.dtype, stream);
    else
        rc = tp_layernorm_bwd(b->dxn, l.x, l.mean1, l.rstd1, l.w[W_LN1_G], b->dh, b->dx, nullptr, nullptr, nullptr, nullptr, M, E,
                              l.dtype, stream);
    if (rc != TP_OK) return rc;
    // the eight vector-parameter gradients, in the order LN1 gain, LN1 offset, in_proj, out_proj, LN2 gain, LN2 offset,
    // fc1, fc2
    const int sizes[8] = {E, E, 3 * E, E, E, E, F, E};
    float* acc[8];
    int64_t total = 0;
    for (int i = 0; i < 8; ++i) { acc[i] = b->small_acc + total; total += sizes[i]; }
    // Up to 1024 rows one launch takes every column's rows in one workgroup and puts the sums where they go; beyond, 256 rows
    // a workgroup, fp32 atomics, and launches that zero and cast (a layer 1600 wide, 256 rows: 22.7 us for the three -> 6.9;
    // 1024 wide, 4096 rows: 34 against 51)
    if (M <= 1024) {
        void* none[8] = {};
        void* const* out = b->small_out[0] ? b->small_out : none;
        const VecSum sums[kVecSums] = {
            {b->dz1, nullptr, nullptr, nullptr, acc[6], nullptr, out[6], nullptr, F, M, F},
            {b->dqkv, nullptr, nullptr, nullptr, acc[2], nullptr, out[2], nullptr, 3 * E, M, 3 * E},
            {b->dxn, l.x, l.mean1, l.rstd1, acc[0], acc[1], out[0], out[1], E, M, E},
            {b->dhn, l.h, l.mean2, l.rstd2, acc[4], acc[5], out[4], out[5], E, M, E},
            {b->dh, nullptr, nullptr, nullptr, acc[3], nullptr, out[3], nullptr, E, M, E},
            {b->dout, nullptr, nullptr, nullptr, acc[7], nullptr, out[7], nullptr, E, M, E},
        };
        if ((rc = vec_param_sums(sums, !b->small_zero, b->small_accumulate, l.dtype, stream)) != TP_OK) return rc;
        return b->wg_rows ? tp_gemm_grouped(p.wg, 4, ws, bytes, stream) : TP_OK;
    }
    if (b->small_zero && (rc = tp_zero_words(b->small_acc, total, stream)) != TP_OK) return rc;
    const tp_vecgrad_desc vg[6] = {
        {b->dqkv, nullptr, nullptr, nullptr, acc[2], nullptr, 3 * E, M, 3 * E},
        {b->dh, nullptr, nullptr, nullptr, acc[3], nullptr, E, M, E},
        {b->dz1, nullptr, nullptr, nullptr, acc[6], nullptr, F, M, F},
        {b->dout, nullptr, nullptr, nullptr, acc[7], nullptr, E, M, E},
        {b->dxn, l.x, l.mean1, l.rstd1, acc[0], acc[1], E, M, E},
        {b->dhn, l.h, l.mean2, l.rstd2, acc[4], acc[5], E, M, E},
    };
    rc = b->wg_rows ? tp_gemm_grouped_vec(p.wg, 4, vg, 6, ws, bytes, stream) : tp_vec_param_grads(vg, 6, l.dtype, stream);
    if (rc != TP_OK) return rc;
    if (b->small_out[0]) rc = tp_accum_cast_parts(b->small_out, sizes, 8, b->small_acc, b->small_accumulate, l.dtype, stream);
    return rc;
}
