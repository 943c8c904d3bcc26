/* forward.c -- fox_eval on the GPU (RustFox src/forward.c:56-132, 295-438 semantics).
 *
 * One decode pass, per layer (src/forward.c:318-397):
 *   xb = rmsnorm(x, attn_norm); q, k, v = W xb; rope(q, k) at pos + t and
 *   store k, v in the layer's cache (one launch for ternary weights);
 *   xb = attention; x += W_o xb (residual fused into the gemv);
 *   xb = rmsnorm(x, ffn_norm); hb = silu(W_gate xb) * (W_up xb) (one launch
 *   for ternary weights); x += W_down hb.
 * then xb = rmsnorm(x_last, output_norm) and logits = W_out xb.
 *
 * The K cache is f32 [n_layer][n_ctx][n_head_kv * head_dim] as in the
 * reference, the V cache the device's position-quad interleaved layout
 * (fox_gpu.h) per layer; the RoPE tables are built on the host in double exactly as
 * src/forward.c:104-118 and uploaded.  fox_eval cuts its input into passes:
 * of at most FOX_GPU_MAX_TOKENS tokens (the decode kernels), or, where
 * n_batch is larger than that and as many tokens are left, of up to n_batch
 * (by default FOX_GPU_BATCH_TOKENS; the batched kernels; a 1024-token prompt of the
 * 4B-class layers in passes of 8 read the weights 128 times).  The result is
 * that of the reference's n_batch chunks because a token depends only on the
 * cache rows before it (batched == stepped, tests/test_forward.c:258-272).
 */
#include "fox_host_internal.h"

#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>

typedef struct {
    const fox_gpu_tensor *attn_q, *attn_k, *attn_v, *attn_out, *ffn_gate, *ffn_up, *ffn_down;
    float *attn_norm, *ffn_norm;   /* device f32 [n_embd] */
} dev_layer;

/* device activations of a pass of up to `cap` tokens: one allocation, carved,
 * and hb2, which only a gate/up that runs as two products needs */
typedef struct {
    void  *block;
    float *x, *xb, *q, *k, *v, *hb, *hb2;
    uint32_t *tok, *pos;           /* pos[i]: the position of token 8 i */
    size_t cap;
} pass_buffers;

#define HEAD_ROWS 64               /* logits rows of one product of a batched fox_eval_all */

struct fox_context {
    fox_model          *m;
    fox_context_config  cfg;
    fox_gpu_ctx        *gpu;
    uint32_t            pos;
    size_t              d, nq, nkv, wide, ff, hd, vocab;
    dev_layer          *L;
    const fox_gpu_tensor *embd, *out;
    float              *out_norm;
    /* device activations */
    float *x, *xb, *q, *k, *v, *hb, *hb2, *dlogits;
    float *kc, *vc, *rc, *rs;
    uint32_t *dtok, *dpos, *dhist, *dzero;
    float *norms;                  /* all norm vectors, n_embd floats each */
    /* pinned host memory (copies to pageable memory pin it page by page each
     * time): the row fox_eval hands out, then log_rows rows that
     * fox_eval_all's logits pass through */
    float *logits, *log_stage;
    size_t log_rows;
    double last_seconds;
    uint64_t reads_at_start;
    /* batched passes: allocated at the first one and again at a larger one
     * (cap 0 before, and where the memory is not there: passes of
     * FOX_GPU_MAX_TOKENS then) */
    pass_buffers B;
    size_t pass_max;               /* most tokens of a pass (n_batch) */
    float *blogits;                /* HEAD_ROWS rows, at the first batched fox_eval_all */
    int no_batch;
    fox_gpu_graph *greedy;
    int attn_mode;                 /* FOX_GPU_ATTN_EXACT or FOX_GPU_ATTN_SPLIT */
    void *allocs[32];
    int n_allocs;
};

static double now_s(void)
{
    struct timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return (double)ts.tv_sec + (double)ts.tv_nsec * 1e-9;
}

#define GPU(call, what)                                       \
    do {                                                      \
        fox_gpu_status gs_ = (call);                          \
        if (gs_ != FOX_GPU_OK) return fox_gpu_failed(gs_, what); \
    } while (0)

static fox_status dalloc(fox_context *c, size_t bytes, void **out)
{
    fox_gpu_status gs;
    if (c->n_allocs == (int)(sizeof(c->allocs) / sizeof(c->allocs[0])))
        return fox_fail(FOX_ERR_INTERNAL, "context: too many buffers");
    gs = fox_gpu_malloc(c->gpu, bytes ? bytes : 4, out);
    if (gs != FOX_GPU_OK)
        return fox_gpu_failed(gs, "context: cannot allocate working memory; try a smaller n_ctx");
    c->allocs[c->n_allocs++] = *out;
    return FOX_OK;
}

static const fox_gpu_tensor *dev_tensor(fox_model *m, size_t idx)
{
    return m->weights->dev[idx];
}

static int streaming(const fox_context *c)
{
    return c->m->weights->mode == FOX_WEIGHTS_STREAM;
}

void fox_context_config_default(fox_context_config *cfg, const fox_model *m)
{
    if (!cfg) return;
    memset(cfg, 0, sizeof(*cfg));
    cfg->n_ctx = m ? m->info.n_ctx_train : 2048;
    cfg->n_batch = FOX_BATCH_DEFAULT;
    cfg->n_threads = 0;
    if (cfg->n_ctx == 0) cfg->n_ctx = 2048;
}

static void batch_free(fox_context *c)
{
    fox_gpu_free(c->gpu, c->B.hb2);
    fox_gpu_free(c->gpu, c->B.block);
    memset(&c->B, 0, sizeof(c->B));
}

void fox_context_destroy(fox_context *c)
{
    int i;
    if (!c) return;
    if (c->greedy) fox_gpu_graph_free(c->greedy);
    if (c->gpu) {
        fox_gpu_sync(c->gpu);
        batch_free(c);
        for (i = 0; i < c->n_allocs; i++) fox_gpu_free(c->gpu, c->allocs[i]);
    }
    if (c->logits) fox_gpu_host_free(c->gpu, c->logits);
    free(c->L);
    free(c);
}

/* device f32 copy of a norm vector into `dst` (src/forward.c:167-186
 * dequantises it per use; it never changes, so it is dequantised once) */
static fox_status norm_vector(fox_context *c, const fox_gpu_tensor *t, float *dst)
{
    GPU(fox_gpu_get_rows(c->gpu, t, c->dzero, 1, dst, c->d, NULL), "context: norm weights");
    return FOX_OK;
}

fox_status fox_context_create(fox_model *m, const fox_context_config *cfg, fox_context **out)
{
    fox_context *c;
    fox_context_config k;
    const fox_model_info *mi;
    fox_status st;
    size_t nb, half, p, i, pass_max;
    float *tc, *ts;
    uint32_t l, zero = 0;

    if (!m || !out) return fox_fail(FOX_ERR_ARG, "context: null argument");
    *out = NULL;
    if (m->weights->mode == FOX_WEIGHTS_RESIDENT)
        return fox_fail(FOX_ERR_UNSUPPORTED,
                        "context: rustfox_amd computes on the GPU; open the model with "
                        "FOX_WEIGHTS_DEVICE or FOX_WEIGHTS_STREAM");
    if (cfg) k = *cfg;
    else fox_context_config_default(&k, m);
    if (k.n_ctx == 0) k.n_ctx = m->info.n_ctx_train;
    if (k.n_ctx == 0) k.n_ctx = 2048;
    if (k.n_batch == 0) k.n_batch = FOX_BATCH_DEFAULT;
    pass_max = k.n_batch == FOX_BATCH_DEFAULT || k.n_batch > FOX_GPU_BATCH_TOKENS
                   ? FOX_GPU_BATCH_TOKENS : k.n_batch;
    if (pass_max > k.n_ctx) pass_max = k.n_ctx;
    if (k.n_batch > k.n_ctx) k.n_batch = k.n_ctx;
    mi = &m->info;

    c = (fox_context *)calloc(1, sizeof(*c));
    if (!c) return fox_fail(FOX_ERR_NOMEM, "context: handle");
    c->m = m;
    c->cfg = k;
    c->pass_max = pass_max;
    c->gpu = m->weights->gpu;
    c->d = mi->n_embd;
    c->hd = mi->head_dim;
    c->nq = (size_t)mi->n_head * mi->head_dim;
    c->nkv = (size_t)mi->n_head_kv * mi->head_dim;
    c->wide = c->nq > c->d ? c->nq : c->d;
    c->ff = mi->n_ff;
    c->vocab = mi->n_vocab;
    c->attn_mode = FOX_GPU_ATTN_EXACT;
    {
        const char *e = getenv("FOX_ATTENTION");
        if (e && strcmp(e, "split") == 0) c->attn_mode = FOX_GPU_ATTN_SPLIT;
    }
    nb = FOX_GPU_MAX_TOKENS;

    /* (fox_eval_all's way out: up to nb rows where they are small) */
    c->log_rows = c->vocab ? ((size_t)1 << 18) / c->vocab : 1;
    if (c->log_rows < 1) c->log_rows = 1;
    if (c->log_rows > nb) c->log_rows = nb;
    if (fox_gpu_host_alloc(c->gpu, ((1 + c->log_rows) * c->vocab + 1) * sizeof(float),
                           (void **)&c->logits) == FOX_GPU_OK) {
        memset(c->logits, 0, c->vocab * sizeof(float));
        c->log_stage = c->logits + c->vocab;
    }
    c->L = (dev_layer *)calloc(mi->n_layer, sizeof(dev_layer));
    if (!c->logits || !c->L) { fox_context_destroy(c); return fox_fail(FOX_ERR_NOMEM, "context: tables"); }

#define ALLOC(ptr, bytes) \
    if ((st = dalloc(c, (bytes), (void **)&(ptr))) != FOX_OK) { fox_context_destroy(c); return st; }
    ALLOC(c->x, nb * c->d * 4)
    ALLOC(c->xb, nb * c->wide * 4)
    ALLOC(c->q, nb * c->nq * 4)
    ALLOC(c->k, nb * c->nkv * 4)
    ALLOC(c->v, nb * c->nkv * 4)
    ALLOC(c->hb, nb * c->ff * 4)
    ALLOC(c->hb2, nb * c->ff * 4)
    ALLOC(c->dlogits, nb * c->vocab * 4)          /* nb rows for fox_eval_all */
    ALLOC(c->kc, (size_t)mi->n_layer * k.n_ctx * c->nkv * 4)
    ALLOC(c->vc, (size_t)mi->n_layer * FOX_GPU_V_CACHE_FLOATS(k.n_ctx, c->nkv) * 4)
    ALLOC(c->rc, (size_t)k.n_ctx * (c->hd / 2) * 4)
    ALLOC(c->rs, (size_t)k.n_ctx * (c->hd / 2) * 4)
    ALLOC(c->dtok, (nb + 1) * 4)                  /* the tokens, then the position */
    ALLOC(c->dhist, (size_t)k.n_ctx * 4)
    ALLOC(c->dzero, 4)
    ALLOC(c->norms, (2 * (size_t)mi->n_layer + 1) * c->d * 4)
#undef ALLOC
    c->dpos = c->dtok + nb;
    if (fox_gpu_memcpy_h2d(c->gpu, c->dzero, &zero, 4) != FOX_GPU_OK ||
        fox_gpu_memset(c->gpu, c->kc, 0, (size_t)mi->n_layer * k.n_ctx * c->nkv * 4) != FOX_GPU_OK ||
        fox_gpu_memset(c->gpu, c->vc, 0,
                       (size_t)mi->n_layer * FOX_GPU_V_CACHE_FLOATS(k.n_ctx, c->nkv) * 4) !=
            FOX_GPU_OK) {
        st = fox_gpu_failed(FOX_GPU_ERR_INTERNAL, "context: initialise buffers");
        fox_context_destroy(c);
        return st;
    }

    /* RoPE tables, src/forward.c:104-118 */
    half = c->hd / 2;
    tc = (float *)malloc((size_t)k.n_ctx * half * 4);
    ts = (float *)malloc((size_t)k.n_ctx * half * 4);
    if (!tc || !ts) {
        free(tc); free(ts);
        fox_context_destroy(c);
        return fox_fail(FOX_ERR_NOMEM, "context: rope tables");
    }
    for (p = 0; p < k.n_ctx; p++)
        for (i = 0; i < half; i++) {
            double ex = -2.0 * (double)i / (double)c->hd;
            double th = (double)p * pow((double)mi->rope_freq_base, ex);
            tc[p * half + i] = (float)cos(th);
            ts[p * half + i] = (float)sin(th);
        }
    st = FOX_OK;
    if (fox_gpu_memcpy_h2d(c->gpu, c->rc, tc, (size_t)k.n_ctx * half * 4) != FOX_GPU_OK ||
        fox_gpu_memcpy_h2d(c->gpu, c->rs, ts, (size_t)k.n_ctx * half * 4) != FOX_GPU_OK)
        st = fox_gpu_failed(FOX_GPU_ERR_INTERNAL, "context: upload rope tables");
    free(tc);
    free(ts);
    if (st != FOX_OK) { fox_context_destroy(c); return st; }

    if ((st = fox_weights_use(m->weights, m->token_embd, &c->embd)) != FOX_OK ||
        (st = fox_weights_use(m->weights, m->output, &c->out)) != FOX_OK) {
        fox_context_destroy(c);
        return st;
    }
    for (l = 0; l < mi->n_layer; l++) {
        const fox_layer_tensors *t = &m->layers[l];
        dev_layer *D = &c->L[l];
        const fox_gpu_tensor *an, *fn;
        D->attn_norm = c->norms + (2 * (size_t)l) * c->d;
        D->ffn_norm = c->norms + (2 * (size_t)l + 1) * c->d;
        if (streaming(c)) {
            /* the layer's matrices are taken from its slot at every pass;
             * its norm vectors are copied out once here */
            const fox_gpu_tensor *lt[FOX_LAYER_ROLES];
            st = fox_weights_use_layer(m->weights, l, lt);
            an = lt[FOX_ROLE_ATTN_NORM];
            fn = lt[FOX_ROLE_FFN_NORM];
        } else {
            D->attn_q = dev_tensor(m, t->attn_q);
            D->attn_k = dev_tensor(m, t->attn_k);
            D->attn_v = dev_tensor(m, t->attn_v);
            D->attn_out = dev_tensor(m, t->attn_out);
            D->ffn_gate = dev_tensor(m, t->ffn_gate);
            D->ffn_up = dev_tensor(m, t->ffn_up);
            D->ffn_down = dev_tensor(m, t->ffn_down);
            an = dev_tensor(m, t->attn_norm);
            fn = dev_tensor(m, t->ffn_norm);
            st = FOX_OK;
        }
        if (st == FOX_OK) st = norm_vector(c, an, D->attn_norm);
        if (st == FOX_OK) st = norm_vector(c, fn, D->ffn_norm);
        if (streaming(c)) fox_weights_done_layer(m->weights, l);
        if (st != FOX_OK) {
            fox_context_destroy(c);
            return st;
        }
    }
    c->out_norm = c->norms + 2 * (size_t)mi->n_layer * c->d;
    {
        const fox_gpu_tensor *on;
        if ((st = fox_weights_use(m->weights, m->output_norm, &on)) != FOX_OK ||
            (st = norm_vector(c, on, c->out_norm)) != FOX_OK) {
            fox_context_destroy(c);
            return st;
        }
    }
    if (fox_gpu_sync(c->gpu) != FOX_GPU_OK) {
        st = fox_gpu_failed(FOX_GPU_ERR_INTERNAL, "context: setup");
        fox_context_destroy(c);
        return st;
    }
    *out = c;
    return FOX_OK;
}

void fox_context_reset(fox_context *c)
{
    if (c) c->pos = 0;
}

uint32_t fox_context_position(const fox_context *c) { return c ? c->pos : 0; }
double fox_context_last_eval_seconds(const fox_context *c) { return c ? c->last_seconds : 0.0; }
uint64_t fox_context_weight_reads(const fox_context *c)
{
    return c ? fox_weights_reads(c->m->weights) : 0;
}

static int same_type(const fox_gpu_tensor *a, const fox_gpu_tensor *b)
{
    int ta, tb;
    uint64_t ka, kb;
    fox_gpu_tensor_info(a, &ta, &ka, NULL, NULL, NULL);
    fox_gpu_tensor_info(b, &tb, &kb, NULL, NULL, NULL);
    return ta == tb && ka == kb;
}

/* y_i = W_i rmsnorm(x, norm_w) for matrices sharing the input, xb scratch for
 * the normed rows: one product for each run of equal types (q/k/v, gate/up),
 * the norm in its input stage where the type has one */
static fox_status project_group(fox_context *c, size_t n, const fox_gpu_tensor *const *ws,
                                const float *x, float *xb, size_t M, const float *norm_w,
                                float *const *outs, const size_t *strides)
{
    const float eps = c->m->info.rms_eps;
    size_t i = 0;
    int normed = 0;
    while (i < n) {
        size_t j = i + 1;
        fox_gpu_status gs = FOX_GPU_ERR_UNSUPPORTED;
        while (j < n && same_type(ws[i], ws[j])) j++;
        if (M > 1)
            gs = fox_gpu_batch_gemv_rmsnorm(c->gpu, j - i, ws + i, x, c->d, M, norm_w, eps, outs + i,
                                            strides + i, 0);
        if (gs == FOX_GPU_ERR_UNSUPPORTED) {
            if (!normed)
                GPU(fox_gpu_rmsnorm(c->gpu, xb, c->wide, x, c->d, norm_w, c->d, M, eps),
                    "forward: norm");
            normed = 1;
            gs = M > FOX_GPU_MAX_TOKENS
                     ? fox_gpu_batch_gemv(c->gpu, j - i, ws + i, xb, c->wide, M, outs + i,
                                          strides + i, 0)
                     : fox_gpu_gemv_multi(c->gpu, j - i, ws + i, xb, c->wide, M, outs + i,
                                          strides + i, 0);
        }
        if (gs != FOX_GPU_OK) return fox_gpu_failed(gs, "forward: projection");
        i = j;
    }
    return FOX_OK;
}

/* layer l's matrices: resident, or from the layer's slot (*SD; loaded now if
 * the prefetch did not reach it; the compute stream waits for its upload) */
static fox_status layer_of(fox_context *c, uint32_t l, dev_layer *SD, const dev_layer **D)
{
    const fox_gpu_tensor *lt[FOX_LAYER_ROLES];
    fox_status st;
    *D = &c->L[l];
    if (!streaming(c)) return FOX_OK;
    if ((st = fox_weights_use_layer(c->m->weights, l, lt)) != FOX_OK) return st;
    *SD = c->L[l];
    SD->attn_q = lt[FOX_ROLE_ATTN_Q];
    SD->attn_k = lt[FOX_ROLE_ATTN_K];
    SD->attn_v = lt[FOX_ROLE_ATTN_V];
    SD->attn_out = lt[FOX_ROLE_ATTN_OUT];
    SD->ffn_gate = lt[FOX_ROLE_FFN_GATE];
    SD->ffn_up = lt[FOX_ROLE_FFN_UP];
    SD->ffn_down = lt[FOX_ROLE_FFN_DOWN];
    *D = SD;
    return FOX_OK;
}

/* the layer-ahead load (src/forward.c:333-337): the next layer, or the first
 * one of the next pass, goes up on the copy stream while this one computes */
static fox_status layer_done(fox_context *c, uint32_t l)
{
    if (!streaming(c)) return FOX_OK;
    fox_weights_done_layer(c->m->weights, l);
    return fox_weights_prefetch_layer(c->m->weights, (l + 1) % c->m->info.n_layer);
}

/* output norm and head (src/forward.c:401-408) over rows of a pass: each
 * row's are independent of the others */
static fox_status head(fox_context *c, const float *x, float *xb, size_t rows, float *logits)
{
    GPU(fox_gpu_rmsnorm(c->gpu, xb, c->wide, x, c->d, c->out_norm, c->d, rows,
                        c->m->info.rms_eps), "forward: output_norm");
    if (rows > FOX_GPU_MAX_TOKENS)
        GPU(fox_gpu_batch_gemv(c->gpu, 1, &c->out, xb, c->wide, rows, &logits, &c->vocab, 0),
            "forward: output");
    else
        GPU(fox_gpu_gemv(c->gpu, c->out, xb, c->wide, rows, logits, c->vocab, 0),
            "forward: output");
    return FOX_OK;
}

/* one pass over all layers for M <= FOX_GPU_MAX_TOKENS tokens already in
 * dtok, at the position held in dpos; queued on the stream, no host sync.
 * want_logits: 0 none, 1 the last token's (dlogits row 0), 2 every token's
 * (dlogits rows 0 .. M-1) */
static fox_status forward_pass(fox_context *c, size_t M, int want_logits)
{
    const fox_model_info *mi = &c->m->info;
    const size_t kvl = (size_t)c->cfg.n_ctx * c->nkv;
    const size_t vl = FOX_GPU_V_CACHE_FLOATS(c->cfg.n_ctx, c->nkv);
    uint32_t l;
    fox_status st;
    fox_gpu_status gs;

    GPU(fox_gpu_get_rows(c->gpu, c->embd, c->dtok, M, c->x, c->d, NULL), "forward: embed");
    for (l = 0; l < mi->n_layer; l++) {
        dev_layer SD;
        const dev_layer *D;
        if ((st = layer_of(c, l, &SD, &D)) != FOX_OK) return st;
        const fox_gpu_tensor *qkv[3] = { D->attn_q, D->attn_k, D->attn_v };
        float *qkv_out[3] = { c->q, c->k, c->v };
        size_t qkv_str[3] = { c->nq, c->nkv, c->nkv };
        const fox_gpu_tensor *gu[2] = { D->ffn_gate, D->ffn_up };
        float *gu_out[2] = { c->hb, c->hb2 };
        size_t gu_str[2] = { c->ff, c->ff };

        /* ternary layers: norm, quantisation, q/k/v and RoPE + cache store in
         * one launch; other types (or activations too wide for one
         * workgroup) take the separate steps */
        gs = fox_gpu_qkv_rope(c->gpu, D->attn_q, D->attn_k, D->attn_v, c->x, c->d, M,
                              D->attn_norm, mi->rms_eps, c->q, c->nq, c->rc, c->rs, c->dpos,
                              c->cfg.n_ctx, c->kc + l * kvl, c->vc + l * vl, c->hd);
        if (gs == FOX_GPU_ERR_UNSUPPORTED) {
            if ((st = project_group(c, 3, qkv, c->x, c->xb, M, D->attn_norm, qkv_out, qkv_str)) !=
                FOX_OK)
                return st;
            GPU(fox_gpu_rope_store(c->gpu, c->q, c->nq, c->k, c->nkv, c->v, c->nkv, mi->n_head,
                                   mi->n_head_kv, c->hd, M, c->rc, c->rs, c->dpos, c->cfg.n_ctx,
                                   c->kc + l * kvl, c->vc + l * vl), "forward: rope");
        } else if (gs != FOX_GPU_OK) {
            return fox_gpu_failed(gs, "forward: q/k/v");
        }
        GPU(fox_gpu_attention(c->gpu, c->xb, c->wide, c->q, c->nq, c->kc + l * kvl,
                              c->vc + l * vl, mi->n_head, mi->n_head_kv, c->hd, M, c->dpos,
                              c->cfg.n_ctx, c->attn_mode), "forward: attention");
        GPU(fox_gpu_gemv(c->gpu, D->attn_out, c->xb, c->wide, M, c->x, c->d,
                         FOX_GPU_GEMV_ACCUMULATE), "forward: attn_output");
        gs = fox_gpu_gate_up_silu(c->gpu, D->ffn_gate, D->ffn_up, c->x, c->d, M, D->ffn_norm,
                                  mi->rms_eps, c->hb, c->ff);
        if (gs == FOX_GPU_ERR_UNSUPPORTED && M > 1)        /* (K-quants, several tokens) */
            gs = fox_gpu_batch_gate_up_silu(c->gpu, D->ffn_gate, D->ffn_up, c->x, c->d, M,
                                            D->ffn_norm, mi->rms_eps, c->hb, c->ff);
        if (gs == FOX_GPU_ERR_UNSUPPORTED) {
            if ((st = project_group(c, 2, gu, c->x, c->xb, M, D->ffn_norm, gu_out, gu_str)) !=
                FOX_OK)
                return st;
            GPU(fox_gpu_silu_mul(c->gpu, c->hb, c->hb2, c->ff, M, c->ff), "forward: swiglu");
        } else if (gs != FOX_GPU_OK) {
            return fox_gpu_failed(gs, "forward: gate/up");
        }
        GPU(fox_gpu_gemv(c->gpu, D->ffn_down, c->hb, c->ff, M, c->x, c->d,
                         FOX_GPU_GEMV_ACCUMULATE), "forward: ffn_down");
        if ((st = layer_done(c, l)) != FOX_OK) return st;
    }
    if (!want_logits) return FOX_OK;
    {
        const size_t rows = want_logits == 2 ? M : 1;
        return head(c, c->x + (M - rows) * c->d, c->xb, rows, c->dlogits);
    }
}

static fox_status batch_add(fox_context *c, const fox_gpu_tensor *w, const float *x, size_t stride,
                            size_t M)
{
    float *out = c->B.x;
    GPU(fox_gpu_batch_gemv(c->gpu, 1, &w, x, stride, M, &out, &c->d, FOX_GPU_GEMV_ACCUMULATE),
        "forward: projection");
    return FOX_OK;
}

/* Attention of a batched pass of M tokens in calls of FOX_GPU_MAX_TOKENS: in
 * split mode always, in exact mode where they are few for the positions they
 * read.  The batched kernels run a token's sums one add at a time in one lane,
 * 48 ns a position and a little more with more heads, whatever M (up to about
 * 64); a call of the decode kernels spreads them over a workgroup and takes
 * 7 ns a position and 1.1 more per 1024 query and per 1024 key columns (4
 * more above 128 dimensions), beside 14 us of launches.  Measured per layer,
 * batched / in calls of eight, us: 32 heads over 8 of 128: 9 tokens at 256
 * positions 29 / 29, at 1024 69 / 45, at 8192 433 / 171; 24 tokens at 1024
 * 69 / 87, at 8192 431 / 340; 40 at 8192 474 / 568; 8 heads over 8 of 64: 40
 * at 8192 413 / 362, 64 there 418 / 581; 80 over 16 of 128: 16 at 4096 253 /
 * 199, 24 there 256 / 300. */
static int attention_in_eights(const fox_context *c, size_t M)
{
    const double p = (double)(c->pos + M), calls = (double)((M + FOX_GPU_MAX_TOKENS - 1) / FOX_GPU_MAX_TOKENS);
    const double nq = (double)c->nq / 1024, nkv = (double)c->nkv / 1024;
    if (c->attn_mode != FOX_GPU_ATTN_EXACT) return 1;
    return calls * (14e3 + p * (6.5 + 1.1 * (nq + nkv) + (c->hd > 128 ? 4 : 0))) <
           17e3 + p * (48 + 1.1 * nq);
}

/* forward_pass for M > FOX_GPU_MAX_TOKENS tokens in B.tok at position
 * B.pos[0] (eights: attention in calls of FOX_GPU_MAX_TOKENS, at B.pos[0 ..]);
 * the residual stream of every token ends in B.x */
static fox_status batch_pass(fox_context *c, size_t M, int eights)
{
    const fox_model_info *mi = &c->m->info;
    pass_buffers *B = &c->B;
    const size_t kvl = (size_t)c->cfg.n_ctx * c->nkv;
    const size_t vl = FOX_GPU_V_CACHE_FLOATS(c->cfg.n_ctx, c->nkv);
    uint32_t l;
    fox_status st;
    fox_gpu_status gs;

    GPU(fox_gpu_get_rows(c->gpu, c->embd, B->tok, M, B->x, c->d, NULL), "forward: embed");
    for (l = 0; l < mi->n_layer; l++) {
        dev_layer SD;
        const dev_layer *D;
        float *kc = c->kc + l * kvl, *vc = c->vc + l * vl;
        if ((st = layer_of(c, l, &SD, &D)) != FOX_OK) return st;
        {
            const fox_gpu_tensor *qkv[3] = { D->attn_q, D->attn_k, D->attn_v };
            float *out[3] = { B->q, B->k, B->v };
            size_t str[3] = { c->nq, c->nkv, c->nkv };
            if ((st = project_group(c, 3, qkv, B->x, B->xb, M, D->attn_norm, out, str)) != FOX_OK)
                return st;
        }
        GPU(fox_gpu_batch_rope_store(c->gpu, B->q, c->nq, B->k, c->nkv, B->v, c->nkv, mi->n_head,
                                     mi->n_head_kv, c->hd, M, c->rc, c->rs, B->pos, c->cfg.n_ctx,
                                     kc, vc), "forward: rope");
        if (!eights) {
            GPU(fox_gpu_batch_attention(c->gpu, B->xb, c->wide, B->q, c->nq, kc, vc, mi->n_head,
                                        mi->n_head_kv, c->hd, M, B->pos, c->cfg.n_ctx),
                "forward: attention");
        } else {
            size_t t;
            for (t = 0; t < M; t += FOX_GPU_MAX_TOKENS) {
                const size_t m = M - t < FOX_GPU_MAX_TOKENS ? M - t : FOX_GPU_MAX_TOKENS;
                GPU(fox_gpu_attention(c->gpu, B->xb + t * c->wide, c->wide, B->q + t * c->nq, c->nq,
                                      kc, vc, mi->n_head, mi->n_head_kv, c->hd, m,
                                      B->pos + t / FOX_GPU_MAX_TOKENS, c->cfg.n_ctx, c->attn_mode),
                    "forward: attention");
            }
        }
        if ((st = batch_add(c, D->attn_out, B->xb, c->wide, M)) != FOX_OK) return st;
        gs = fox_gpu_batch_gate_up_silu(c->gpu, D->ffn_gate, D->ffn_up, B->x, c->d, M, D->ffn_norm,
                                        mi->rms_eps, B->hb, c->ff);
        if (gs == FOX_GPU_ERR_UNSUPPORTED) {
            const fox_gpu_tensor *gu[2] = { D->ffn_gate, D->ffn_up };
            float *out[2] = { B->hb, B->hb2 };
            size_t str[2] = { c->ff, c->ff };
            if (!B->hb2) {
                GPU(fox_gpu_malloc(c->gpu, B->cap * c->ff * 4, (void **)&B->hb2), "forward: swiglu");
                out[1] = B->hb2;
            }
            if ((st = project_group(c, 2, gu, B->x, B->xb, M, D->ffn_norm, out, str)) != FOX_OK)
                return st;
            GPU(fox_gpu_silu_mul(c->gpu, B->hb, B->hb2, c->ff, M, c->ff), "forward: swiglu");
        } else if (gs != FOX_GPU_OK) {
            return fox_gpu_failed(gs, "forward: gate/up");
        }
        if ((st = batch_add(c, D->ffn_down, B->hb, c->ff, M)) != FOX_OK) return st;
        if ((st = layer_done(c, l)) != FOX_OK) return st;
    }
    return FOX_OK;
}

/* `rows` rows of logits to the caller's memory, through the pinned rows */
static fox_status logits_out(fox_context *c, float *dst, const float *src, size_t rows)
{
    size_t i, r;
    for (i = 0; i < rows; i += r) {
        r = rows - i < c->log_rows ? rows - i : c->log_rows;
        GPU(fox_gpu_memcpy_d2h(c->gpu, c->log_stage, src + i * c->vocab, r * c->vocab * 4),
            "eval: logits");
        memcpy(dst + i * c->vocab, c->log_stage, r * c->vocab * 4);
    }
    return FOX_OK;
}

/* the buffers of batched passes of n tokens, or of as many as can be had (B.cap);
 * 0 where none can.  Sized in steps, so that a short prompt does not pay for a
 * long one's memory; they grow with the prompts.  (Nine allocations for 1024
 * tokens in a context's first prompt of nine: 364 us for a 4B-class layer,
 * two passes of the decode kernels 285, here 201, warm 167.) */
static int batch_ready(fox_context *c, size_t n)
{
    pass_buffers b;
    struct { void *p; size_t row; } part[8] = {
        { &b.x, c->d }, { &b.xb, c->wide }, { &b.q, c->nq }, { &b.k, c->nkv }, { &b.v, c->nkv },
        { &b.hb, c->ff }, { &b.tok, 1 }, { &b.pos, 1 }
    };
    size_t step = 64, i;
    if (c->B.cap >= n) return 1;
    if (c->no_batch) return 0;
    while (step < n) step *= 4;
    const size_t asked = step;
    batch_free(c);
    for (; step >= 64; step /= 4) {
        const size_t cap = step < c->pass_max ? step : c->pass_max;
        size_t bytes = 0;
        memset(&b, 0, sizeof(b));
        for (i = 0; i < 8; i++) bytes += (cap * part[i].row * 4 + 255) & ~(size_t)255;
        if (fox_gpu_malloc(c->gpu, bytes, &b.block) != FOX_GPU_OK) continue;
        bytes = 0;
        for (i = 0; i < 8; i++) {
            *(void **)part[i].p = (char *)b.block + bytes;
            bytes += (cap * part[i].row * 4 + 255) & ~(size_t)255;
        }
        b.cap = cap;
        c->B = b;
        if (step < asked) c->pass_max = cap;               /* (not tried again at every pass) */
        return 1;
    }
    c->no_batch = 1;
    return 0;
}

/* tokens [done, done + M) as one batched pass; the logits wanted (all: every
 * row's into `all`; else the last row's into dlogits when `last`) */
static fox_status batch_eval(fox_context *c, const uint32_t *tokens, size_t M, int last, float *all)
{
    uint32_t pos[FOX_GPU_BATCH_TOKENS / FOX_GPU_MAX_TOKENS + 1];
    const size_t np = (M + FOX_GPU_MAX_TOKENS - 1) / FOX_GPU_MAX_TOKENS;
    const int eights = attention_in_eights(c, M);
    const size_t stored = eights ? np : 1;
    size_t i, r;
    fox_status st;
    for (i = 0; i < np; i++) pos[i] = c->pos + (uint32_t)(i * FOX_GPU_MAX_TOKENS);
    GPU(fox_gpu_memcpy_h2d(c->gpu, c->B.tok, tokens, M * 4), "eval: tokens");
    if (stored <= 16)
        GPU(fox_gpu_store_u32(c->gpu, c->B.pos, pos, stored), "eval: position");
    else
        GPU(fox_gpu_memcpy_h2d(c->gpu, c->B.pos, pos, stored * 4), "eval: position");
    if ((st = batch_pass(c, M, eights)) != FOX_OK) return st;
    if (!all) return last ? head(c, c->B.x + (M - 1) * c->d, c->B.xb, 1, c->dlogits) : FOX_OK;
    if (!c->blogits &&
        (st = dalloc(c, HEAD_ROWS * c->vocab * 4, (void **)&c->blogits)) != FOX_OK)
        return st;
    for (i = 0; i < M; i += r) {
        r = M - i < HEAD_ROWS ? M - i : HEAD_ROWS;
        if ((st = head(c, c->B.x + i * c->d, c->B.xb, r, c->blogits)) != FOX_OK) return st;
        if ((st = logits_out(c, all + i * c->vocab, c->blogits, r)) != FOX_OK) return st;
    }
    return FOX_OK;
}

static fox_status check_tokens(const fox_context *c, const uint32_t *t, size_t n)
{
    size_t i;
    for (i = 0; i < n; i++)
        if (t[i] >= c->vocab)
            return fox_fail(FOX_ERR_ARG, "forward: token %u is outside the %zu entry vocabulary",
                            t[i], c->vocab);
    return FOX_OK;
}

/* chunk [done, done + chunk) of an evaluation at position `pos` */
static fox_status check_chunk(const fox_context *c, const uint32_t *tokens, size_t chunk, size_t pos)
{
    if (pos + chunk > c->cfg.n_ctx)
        return fox_fail(FOX_ERR_ARG, "forward: %zu tokens past position %zu would overrun the "
                        "%u token context", chunk, pos, c->cfg.n_ctx);
    return check_tokens(c, tokens, chunk);
}

/* all == NULL: the last token's logits into c->logits, else every token's
 * into all.  The input is checked in chunks of at most n_batch (and
 * FOX_GPU_MAX_TOKENS): the chunks before a bad one are evaluated, then its
 * error is returned.  The good tokens run in batched passes of at most pass_max
 * where that and what is left are more than FOX_GPU_MAX_TOKENS, in such chunks
 * otherwise. */
static fox_status eval_chunks(fox_context *c, const uint32_t *tokens, size_t n, float *all)
{
    size_t done = 0, good = 0, cap = c->cfg.n_batch;
    double t0;
    fox_status st, bad = FOX_OK;

    t0 = now_s();
    c->reads_at_start = fox_weights_reads(c->m->weights);
    if (cap > FOX_GPU_MAX_TOKENS) cap = FOX_GPU_MAX_TOKENS;
    while (good < n) {
        const size_t chunk = n - good < cap ? n - good : cap;
        if ((bad = check_chunk(c, tokens + good, chunk, (size_t)c->pos + good)) != FOX_OK) break;
        good += chunk;
    }
    while (done < good) {
        size_t left = good - done, chunk = left < cap ? left : cap;
        int last;
        if (left > FOX_GPU_MAX_TOKENS && c->pass_max > FOX_GPU_MAX_TOKENS &&
            batch_ready(c, left < c->pass_max ? left : c->pass_max)) {
            /* passes of about one size, whole groups of 64 tokens */
            const size_t most = c->B.cap < c->pass_max ? c->B.cap : c->pass_max;
            const size_t np = (left + most - 1) / most;
            chunk = ((left + np - 1) / np + 63) & ~(size_t)63;
            if (chunk > most) chunk = most;
            if (chunk > left) chunk = left;
        }
        last = done + chunk == n;
        if (chunk > FOX_GPU_MAX_TOKENS) {
            st = batch_eval(c, tokens + done, chunk, last, all ? all + done * c->vocab : NULL);
            if (st == FOX_ERR_NOMEM && fox_gpu_sync(c->gpu) == FOX_GPU_OK) {
                /* a workspace or the logits rows could not be had: the same
                 * tokens again in passes of the decode kernels (they write
                 * the same cache rows; what the pass queued has ended, so
                 * nothing reads a layer's slot that is loaded again) */
                batch_free(c);
                c->no_batch = 1;
                continue;
            }
            if (st != FOX_OK) return st;
        } else {
            uint32_t in[FOX_GPU_MAX_TOKENS + 1] = { 0 };
            memcpy(in, tokens + done, chunk * 4);
            in[FOX_GPU_MAX_TOKENS] = c->pos;               /* (dpos follows dtok) */
            GPU(fox_gpu_store_u32(c->gpu, c->dtok, in, FOX_GPU_MAX_TOKENS + 1), "eval: tokens");
            if ((st = forward_pass(c, chunk, all ? 2 : last)) != FOX_OK) return st;
            if (all &&
                (st = logits_out(c, all + done * c->vocab, c->dlogits, chunk)) != FOX_OK)
                return st;
        }
        c->pos += (uint32_t)chunk;
        done += chunk;
    }
    /* (the check again: the message of its failure is the last one) */
    if (bad != FOX_OK)
        return check_chunk(c, tokens + good, n - good < cap ? n - good : cap, c->pos);
    if (!all) GPU(fox_gpu_memcpy_d2h(c->gpu, c->logits, c->dlogits, c->vocab * 4), "eval: logits");
    c->last_seconds = now_s() - t0;
    return FOX_OK;
}

fox_status fox_eval(fox_context *c, const uint32_t *tokens, size_t n, float **logits_out)
{
    fox_status st;
    if (!c || !tokens || n == 0) return fox_fail(FOX_ERR_ARG, "eval: nothing to evaluate");
    if ((st = eval_chunks(c, tokens, n, NULL)) != FOX_OK) return st;
    if (logits_out) *logits_out = c->logits;
    return FOX_OK;
}

fox_status fox_eval_all(fox_context *c, const uint32_t *tokens, size_t n, float *logits)
{
    if (!c || !tokens || n == 0 || !logits)
        return fox_fail(FOX_ERR_ARG, "eval_all: nothing to evaluate");
    return eval_chunks(c, tokens, n, logits);
}

/* one greedy step: forward at dpos with the token in dtok[0], then
 * dtok[0] = argmax, dhist[dpos] = argmax, dpos += 1 */
static fox_status greedy_step(fox_context *c)
{
    fox_status st = forward_pass(c, 1, 1);
    if (st != FOX_OK) return st;
    GPU(fox_gpu_argmax(c->gpu, c->dlogits, c->vocab, c->dtok, c->dpos, 1, c->dhist),
        "decode: argmax");
    return FOX_OK;
}

fox_status fox_decode_greedy(fox_context *c, uint32_t token, size_t n_steps, uint32_t *out_ids)
{
    double t0;
    size_t s;
    fox_status st;

    if (!c || (!out_ids && n_steps)) return fox_fail(FOX_ERR_ARG, "decode: null argument");
    if (n_steps == 0) return FOX_OK;
    if ((size_t)c->pos + n_steps > c->cfg.n_ctx)
        return fox_fail(FOX_ERR_ARG, "decode: %zu steps past position %u would overrun the %u "
                        "token context", n_steps, c->pos, c->cfg.n_ctx);
    if ((st = check_tokens(c, &token, 1)) != FOX_OK) return st;
    t0 = now_s();
    GPU(fox_gpu_store_u32(c->gpu, c->dtok, &token, 1), "decode: token");
    GPU(fox_gpu_store_u32(c->gpu, c->dpos, &c->pos, 1), "decode: position");
    /* the first step runs eagerly (it also sizes every workspace), the rest
     * replay one captured graph; FOX_GRAPHS=0 keeps every step eager (for
     * profilers that cannot follow graph launches), and so does streaming
     * (each step reloads layer slots from the host) */
    if ((st = greedy_step(c)) != FOX_OK) return st;
    {
        const char *e = getenv("FOX_GRAPHS");
        if ((e && strcmp(e, "0") == 0) || streaming(c)) {
            for (s = 1; s < n_steps; s++)
                if ((st = greedy_step(c)) != FOX_OK) return st;
            GPU(fox_gpu_memcpy_d2h(c->gpu, out_ids, c->dhist + c->pos, n_steps * 4), "decode: ids");
            c->pos += (uint32_t)n_steps;
            c->last_seconds = now_s() - t0;
            return FOX_OK;
        }
    }
    if (n_steps > 1 && !c->greedy) {
        GPU(fox_gpu_graph_begin(c->gpu), "decode: capture");
        st = greedy_step(c);
        {
            fox_gpu_status gs = fox_gpu_graph_end(c->gpu, &c->greedy);
            if (st != FOX_OK) return st;
            if (gs != FOX_GPU_OK) return fox_gpu_failed(gs, "decode: capture");
        }
    }
    for (s = 1; s < n_steps; s++) GPU(fox_gpu_graph_launch(c->gpu, c->greedy), "decode: replay");
    GPU(fox_gpu_memcpy_d2h(c->gpu, out_ids, c->dhist + c->pos, n_steps * 4), "decode: ids");
    c->pos += (uint32_t)n_steps;
    c->last_seconds = now_s() - t0;
    return FOX_OK;
}

fox_status fox_context_set_kv(fox_context *c, uint32_t layer, uint32_t p0, uint32_t n,
                              const float *k, const float *v)
{
    size_t bytes;
    float *tmp;
    fox_gpu_status gs;
    if (!c || !k || !v) return fox_fail(FOX_ERR_ARG, "set_kv: null argument");
    if (layer >= c->m->info.n_layer || (size_t)p0 + n > c->cfg.n_ctx)
        return fox_fail(FOX_ERR_ARG, "set_kv: rows %u..%u of layer %u are outside the cache",
                        p0, p0 + n, layer);
    if (n == 0) return FOX_OK;
    bytes = (size_t)n * c->nkv * 4;
    GPU(fox_gpu_malloc(c->gpu, 2 * bytes, (void **)&tmp), "set_kv: staging");
    gs = fox_gpu_memcpy_h2d(c->gpu, tmp, k, bytes);
    if (gs == FOX_GPU_OK) gs = fox_gpu_memcpy_h2d(c->gpu, tmp + (size_t)n * c->nkv, v, bytes);
    if (gs == FOX_GPU_OK)
        gs = fox_gpu_kv_write(c->gpu, c->kc + (size_t)layer * c->cfg.n_ctx * c->nkv,
                              c->vc + (size_t)layer * FOX_GPU_V_CACHE_FLOATS(c->cfg.n_ctx, c->nkv),
                              c->nkv, c->cfg.n_ctx, p0, n, tmp, tmp + (size_t)n * c->nkv);
    if (gs == FOX_GPU_OK) gs = fox_gpu_sync(c->gpu);
    fox_gpu_free(c->gpu, tmp);
    if (gs != FOX_GPU_OK) return fox_gpu_failed(gs, "set_kv");
    return FOX_OK;
}

fox_status fox_context_set_position(fox_context *c, uint32_t pos)
{
    if (!c) return fox_fail(FOX_ERR_ARG, "set_position: null context");
    if (pos > c->cfg.n_ctx) return fox_fail(FOX_ERR_ARG, "set_position: %u > n_ctx", pos);
    c->pos = pos;
    return FOX_OK;
}

fox_status fox_context_set_attention(fox_context *c, int exact)
{
    if (!c) return fox_fail(FOX_ERR_ARG, "set_attention: null context");
    c->attn_mode = exact ? FOX_GPU_ATTN_EXACT : FOX_GPU_ATTN_SPLIT;
    if (c->greedy) {
        fox_gpu_sync(c->gpu);
        fox_gpu_graph_free(c->greedy);
        c->greedy = NULL;
    }
    return FOX_OK;
}
