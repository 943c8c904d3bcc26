/* gpu_stub.c -- the device library's entry points on host memory, for tests
 * of the host library's own decisions (passes, buffers, fallbacks) without a
 * GPU.  No arithmetic: an embedding row holds its token's id, everything up
 * to the output head passes it on, and the head's logits are id * rows + row,
 * so a logits row says which token it belongs to.  Calls are counted and
 * allocations can be made to fail from the test. */
#include "../include/fox_gpu.h"

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

struct fox_gpu_tensor { int type; uint64_t ne0, ne1; };

size_t stub_fail_above;      /* fox_gpu_malloc of more bytes fails; 0: none */
int    stub_fail_attention;  /* the next so many batched attentions fail (NOMEM) */
size_t stub_mallocs, stub_live, stub_max_batch, stub_eights, stub_batches, stub_small_attn;
size_t stub_head_rows;       /* rows of a matrix that is the output head */

static struct { void *p; size_t n; } blocks[4096];

fox_gpu_status fox_gpu_init(int device, fox_gpu_ctx **out)
{
    (void)device;
    *out = (fox_gpu_ctx *)calloc(1, 64);
    return FOX_GPU_OK;
}
void fox_gpu_shutdown(fox_gpu_ctx *ctx) { free(ctx); }
const char *fox_gpu_last_error(void) { return "stub"; }
const char *fox_gpu_status_str(fox_gpu_status s) { (void)s; return "stub"; }
fox_gpu_status fox_gpu_set_max_workgroups(fox_gpu_ctx *c, int n) { (void)c; (void)n; return FOX_GPU_OK; }

fox_gpu_status fox_gpu_malloc(fox_gpu_ctx *ctx, size_t bytes, void **out)
{
    size_t i = 0;
    (void)ctx;
    *out = NULL;
    if (stub_fail_above && bytes > stub_fail_above) return FOX_GPU_ERR_NOMEM;
    while (blocks[i].p) i++;
    *out = blocks[i].p = calloc(1, bytes);
    blocks[i].n = bytes;
    stub_live += bytes;
    stub_mallocs++;
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_free(fox_gpu_ctx *ctx, void *p)
{
    size_t i;
    (void)ctx;
    for (i = 0; p && i < sizeof(blocks) / sizeof(blocks[0]); i++)
        if (blocks[i].p == p) {
            stub_live -= blocks[i].n;
            blocks[i].p = NULL;
            free(p);
            return FOX_GPU_OK;
        }
    if (p) { fprintf(stderr, "stub: free of an unknown pointer\n"); abort(); }
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_host_alloc(fox_gpu_ctx *c, size_t n, void **out) { (void)c; *out = malloc(n); return FOX_GPU_OK; }
fox_gpu_status fox_gpu_host_free(fox_gpu_ctx *c, void *p) { (void)c; free(p); return FOX_GPU_OK; }
fox_gpu_status fox_gpu_memcpy_h2d(fox_gpu_ctx *c, void *d, const void *s, size_t n) { (void)c; memcpy(d, s, n); return FOX_GPU_OK; }
fox_gpu_status fox_gpu_memcpy_d2h(fox_gpu_ctx *c, void *d, const void *s, size_t n) { (void)c; memcpy(d, s, n); return FOX_GPU_OK; }
fox_gpu_status fox_gpu_memset(fox_gpu_ctx *c, void *d, int v, size_t n) { (void)c; memset(d, v, n); return FOX_GPU_OK; }
fox_gpu_status fox_gpu_store_u32(fox_gpu_ctx *c, uint32_t *d, const uint32_t *w, size_t n) { (void)c; memcpy(d, w, 4 * n); return FOX_GPU_OK; }
fox_gpu_status fox_gpu_sync(fox_gpu_ctx *c) { (void)c; return FOX_GPU_OK; }

fox_gpu_status fox_gpu_tensor_alloc(fox_gpu_ctx *c, int type, uint64_t ne0, uint64_t ne1, fox_gpu_tensor **out)
{
    (void)c;
    *out = (fox_gpu_tensor *)calloc(1, sizeof(**out));
    (*out)->type = type;
    (*out)->ne0 = ne0;
    (*out)->ne1 = ne1 ? ne1 : 1;
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_tensor_upload(fox_gpu_ctx *c, int type, uint64_t ne0, uint64_t ne1, const void *h,
                                     uint64_t bytes, fox_gpu_tensor **out)
{
    (void)h; (void)bytes;
    return fox_gpu_tensor_alloc(c, type, ne0, ne1, out);
}
fox_gpu_status fox_gpu_tensor_info(const fox_gpu_tensor *t, int *type, uint64_t *ne0, uint64_t *ne1,
                                   uint64_t *g, uint64_t *d)
{
    if (type) *type = t->type;
    if (ne0) *ne0 = t->ne0;
    if (ne1) *ne1 = t->ne1;
    if (g) *g = 0;
    if (d) *d = 0;
    return FOX_GPU_OK;
}
void fox_gpu_tensor_free(fox_gpu_ctx *c, fox_gpu_tensor *t) { (void)c; free(t); }

fox_gpu_status fox_gpu_get_rows(fox_gpu_ctx *c, const fox_gpu_tensor *t, const uint32_t *rows, size_t n,
                                float *out, size_t stride, uint32_t *bad)
{
    size_t i;
    (void)c; (void)t; (void)bad;
    for (i = 0; i < n; i++) out[i * stride] = (float)rows[i];
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_rmsnorm(fox_gpu_ctx *c, float *out, size_t os, const float *x, size_t xs, const float *w,
                               size_t n, size_t M, float eps)
{
    size_t i;
    (void)c; (void)w; (void)n; (void)eps;
    for (i = 0; i < M; i++) out[i * os] = x[i * xs];
    return FOX_GPU_OK;
}

static void product(const fox_gpu_tensor *w, const float *x, size_t xs, size_t M, float *out, size_t os)
{
    size_t t, r;
    if (w->ne1 != stub_head_rows) return;
    for (t = 0; t < M; t++)
        for (r = 0; r < w->ne1; r++) out[t * os + r] = x[t * xs] * (float)w->ne1 + (float)r;
}
fox_gpu_status fox_gpu_gemv(fox_gpu_ctx *c, const fox_gpu_tensor *w, const float *x, size_t xs, size_t M,
                            float *out, size_t os, unsigned flags)
{
    (void)c; (void)flags;
    if (M > FOX_GPU_MAX_TOKENS) return FOX_GPU_ERR_ARG;
    product(w, x, xs, M, out, os);
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_batch_gemv(fox_gpu_ctx *c, size_t n, const fox_gpu_tensor *const *ws, const float *x,
                                  size_t xs, size_t M, float *const *outs, const size_t *os, unsigned flags)
{
    size_t i;
    (void)c; (void)flags;
    if (M > stub_max_batch) stub_max_batch = M;
    for (i = 0; i < n; i++) product(ws[i], x, xs, M, outs[i], os[i]);
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_gate_up_silu(fox_gpu_ctx *c, const fox_gpu_tensor *g, const fox_gpu_tensor *u,
                                    const float *x, size_t xs, size_t M, const float *nw, float eps, float *h,
                                    size_t hs)
{
    (void)c; (void)g; (void)u; (void)x; (void)xs; (void)nw; (void)eps; (void)h; (void)hs;
    return M > FOX_GPU_MAX_TOKENS ? FOX_GPU_ERR_ARG : FOX_GPU_OK;
}
fox_gpu_status fox_gpu_qkv_rope(fox_gpu_ctx *c, const fox_gpu_tensor *wq, const fox_gpu_tensor *wk,
                                const fox_gpu_tensor *wv, const float *x, size_t xs, size_t M, const float *nw,
                                float eps, float *q, size_t qs, const float *ct, const float *st,
                                const uint32_t *pos, size_t n_ctx, float *kc, float *vc, size_t hd)
{
    (void)c; (void)wq; (void)wk; (void)wv; (void)x; (void)xs; (void)nw; (void)eps; (void)q; (void)qs; (void)ct;
    (void)st; (void)pos; (void)n_ctx; (void)kc; (void)vc; (void)hd;
    stub_eights++;
    return M > FOX_GPU_MAX_TOKENS ? FOX_GPU_ERR_ARG : FOX_GPU_OK;
}
fox_gpu_status fox_gpu_batch_rope_store(fox_gpu_ctx *c, float *q, size_t qs, float *k, size_t ks, const float *v,
                                        size_t vs, size_t nh, size_t nkv, size_t hd, size_t M, const float *ct,
                                        const float *st, const uint32_t *pos, size_t n_ctx, float *kc, float *vc)
{
    (void)c; (void)q; (void)qs; (void)k; (void)ks; (void)v; (void)vs; (void)nh; (void)nkv; (void)hd; (void)M;
    (void)ct; (void)st; (void)pos; (void)n_ctx; (void)kc; (void)vc;
    stub_batches++;
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_batch_attention(fox_gpu_ctx *c, float *out, size_t os, const float *q, size_t qs,
                                       const float *k, const float *v, size_t nh, size_t nkv, size_t hd, size_t M,
                                       const uint32_t *pos, size_t n_ctx)
{
    (void)c; (void)out; (void)os; (void)q; (void)qs; (void)k; (void)v; (void)nh; (void)nkv; (void)hd; (void)M;
    (void)pos; (void)n_ctx;
    if (stub_fail_attention) { stub_fail_attention--; return FOX_GPU_ERR_NOMEM; }
    return FOX_GPU_OK;
}
fox_gpu_status fox_gpu_attention(fox_gpu_ctx *c, float *out, size_t os, const float *q, size_t qs, const float *k,
                                 const float *v, size_t nh, size_t nkv, size_t hd, size_t M, const uint32_t *pos,
                                 size_t n_ctx, int mode)
{
    (void)c; (void)out; (void)os; (void)q; (void)qs; (void)k; (void)v; (void)nh; (void)nkv; (void)hd; (void)pos;
    (void)n_ctx; (void)mode;
    stub_small_attn++;
    return M > FOX_GPU_MAX_TOKENS ? FOX_GPU_ERR_ARG : FOX_GPU_OK;
}

/* what the other entry points are linked to: those that need nothing done, and
 * those that no test here calls */
fox_gpu_status stub_ok(void) { return FOX_GPU_OK; }
fox_gpu_status stub_refused(void) { return FOX_GPU_ERR_INTERNAL; }
