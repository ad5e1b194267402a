/*
 * ork_mlp.c -- host side of the QAOA energy surrogate: an MLP
 * in_dim -> hidden x nhidden (GELU) -> 1 whose forward and backward passes run
 * on the BF16 MFMA kernels of k_mlp.hip, trained with Adam on fp32 master
 * weights.  No reference counterpart (the learned screening stage).
 *
 * Layer l (0..nhidden-1) maps width K_l -> hidden: W_l is kept as fp32 [K_l][hidden]
 * (master), bf16 [K_l][hidden] (for dX = dY W^T) and bf16 [hidden][K_l] (forward).
 * The head is fp32: y = h . w_out + b_out.
 */
#include "ork_host.h"

#include <math.h>
#include <string.h>
#include <hip/hip_runtime_api.h>

int ork_mlp_gemm(void *stream, int epi, const void *A, int lda, const void *B, int ldb, int M, int N, int K,
                 float *c32, int ldc, const float *bias, float *pre, void *act, void *actT, long ldt);
int ork_mlp_stage_input(void *stream, const float *x, int m0, int m1, int rows, int K, void *x16, void *x16t, long ldt,
                        const float *tgt_src, float *tgt);
int ork_mlp_pack(void *stream, int count, const float *const *src, const int *len, float *dst);
int ork_mlp_head_forward(void *stream, const void *h, const float *w, float b, int M, int K, float *y,
                         const float *target, float *dy, float *sqerr, int valid, float scale);
int ork_mlp_head_backward_t(void *stream, const float *dy, const float *w, const float *pre, int M, int K, void *dpre,
                            void *dpret, long ldt);
int ork_mlp_weight_grads(void *stream, int nl, const void *const *xt, const void *const *dt, float *const *g,
                         const int *K, int N, int rows, long ldt, int max_slices);
int ork_mlp_colsums(void *stream, int count, const void *const *a, const float *const *s, float *const *out, int M,
                    int K, float *part, const float *v0, const float *v1, float *vout);
int ork_mlp_first_layer_graph(void *stream, const float *gf, int ng, const void *w, int N, float *u);
int ork_mlp_first_layer_rows(void *stream, const float *angles, int na, long r0, int rows, int Mp, const float *u,
                             const void *wa, const float *bias, int N, void *act);
int ork_mlp_screen_ok(int na, int hidden, int nl);
int ork_mlp_screen(void *stream, const float *gf, int ng, const void *w0, const void *const *wt, void *wpk, float *u,
                   const float *const *bias, int nl, int H, const float *w_out, float b_out, const float *angles,
                   long ncand, float *y);
int ork_mlp_adam_all(void *stream, int count, float *const *w, const float *const *g, float *const *m, float *const *v,
                     void *const *wb, void *const *wtb, const int *rows, const int *cols, float lr, float b1, float b2,
                     float eps, float c1, float c2);

#define MLP_MAX_LAYERS 4
#define SPLITK_MAX 32   /* K slices of the weight-gradient products */
#define TILE 128
/* of a host batch: the host copies one chunk while the device reads the one before */
#define CHUNK_FLOATS ((size_t)1 << 17)
#define TPAD 64         /* row padding of the transposed operands: rows a power of two apart share memory channels */

typedef struct {
    int K, N;
    float *w, *g, *m, *v;        /* fp32 [K][N] */
    float *b, *gb, *mb, *vb;     /* fp32 [N] */
    void *wb, *wtb;              /* bf16 [K][N] and [N][K] */
} layer_t;

struct orkan_mlp {
    int in_dim, hidden, nl, max_batch;
    layer_t L[MLP_MAX_LAYERS];
    float *w_out, *g_out, *m_out, *v_out;   /* [hidden] */
    float b_out, mb_out, vb_out;
    /* activations (max_batch rows, padded to TILE) */
    float *x32;                 /* [M][in_dim] staged input */
    void *x16;                  /* bf16 [M][in_dim] */
    float *pre[MLP_MAX_LAYERS]; /* fp32 [M][hidden] */
    void *act[MLP_MAX_LAYERS];  /* bf16 [M][hidden] */
    /* gradients of the pre-activations, bf16 [M][hidden]: the last layer's in memory of their own, an earlier layer's in
     * place of its activations, which the backward pass does not read.  (Their transposes could take the place of the
     * pre-activations of the layer after: that made each backward product 1 us slower, 13.4 -> 14.5 at 4096 x 512.) */
    void *dpre[MLP_MAX_LAYERS];
    /* transposed operands of the weight gradients: the layers' inputs and dpre, bf16 [width][M + TPAD], in one allocation
     * (one each took 100 us and more: the padding puts them past a 2 MB page) */
    void *in_t[MLP_MAX_LAYERS], *dpre_t[MLP_MAX_LAYERS], *transposes;
    float *y, *dy, *sq, *tgt;
    float *scal;                /* sum of squared errors, d loss / d b_out; pinned */
    float *host;                /* the pinned buffer, while a batch staged in it is on its way */
    float *colpart;             /* (nl + 1) x 64 x hidden partial column sums */
    float *gf_dev, *u1;         /* screening: graph features [in_dim], their layer-1 share [hidden] */
    void *wpk;                  /* screening: the later layers' weights in fragment order */
    long step;
};

static void *dmalloc(size_t bytes, int *err) {
    void *p = NULL;
    if (*err) return NULL;
    if (ork_dev_malloc(&p, bytes ? bytes : 16) != 0) {
        *err = 1;
        return NULL;
    }
    return p;
}

static int pad_rows(int m) { return (m + TILE - 1) / TILE * TILE; }

orkan_mlp_t *orkan_mlp_create(int in_dim, int hidden, int nhidden, int max_batch) {
    if (in_dim % 32 || in_dim <= 0 || hidden % TILE || hidden <= 0 || nhidden < 1 || nhidden > MLP_MAX_LAYERS ||
        max_batch <= 0)
        return NULL;
    orkan_mlp_t *q = calloc(1, sizeof(*q));
    if (!q) return NULL;
    ork_dev();
    int err = 0;
    q->in_dim = in_dim;
    q->hidden = hidden;
    q->nl = nhidden;
    q->max_batch = pad_rows(max_batch);
    const size_t M = (size_t)q->max_batch, H = (size_t)hidden;
    for (int l = 0; l < nhidden; ++l) {
        layer_t *L = &q->L[l];
        L->K = l == 0 ? in_dim : hidden;
        L->N = hidden;
        const size_t n = (size_t)L->K * L->N;
        L->w = dmalloc(n * 4, &err); L->g = dmalloc(n * 4, &err);
        L->m = dmalloc(n * 4, &err); L->v = dmalloc(n * 4, &err);
        L->b = dmalloc(H * 4, &err); L->gb = dmalloc(H * 4, &err);
        L->mb = dmalloc(H * 4, &err); L->vb = dmalloc(H * 4, &err);
        L->wb = dmalloc(n * 2, &err); L->wtb = dmalloc(n * 2, &err);
        q->pre[l] = dmalloc(M * H * 4, &err);
        q->act[l] = dmalloc(M * H * 2, &err);
    }
    const size_t column = (M + TPAD) * 2;
    char *t = q->transposes = dmalloc(column * ((size_t)in_dim + (2 * (size_t)nhidden - 1) * H), &err);
    for (int l = 0; l < nhidden && t; ++l) {
        q->in_t[l] = t;
        q->dpre_t[l] = t += column * (size_t)q->L[l].K;
        t += column * H;
        q->dpre[l] = l == nhidden - 1 ? dmalloc(M * H * 2, &err) : q->act[l];
    }
    q->w_out = dmalloc(H * 4, &err); q->g_out = dmalloc(H * 4, &err);
    q->m_out = dmalloc(H * 4, &err); q->v_out = dmalloc(H * 4, &err);
    q->x32 = dmalloc(M * in_dim * 4, &err);
    q->x16 = dmalloc(M * in_dim * 2, &err);
    q->y = dmalloc(M * 4, &err); q->dy = dmalloc(M * 4, &err);
    q->sq = dmalloc(M * 4, &err); q->tgt = dmalloc(M * 4, &err);
    q->colpart = dmalloc((size_t)(nhidden + 1) * 64 * H * 4, &err);
    q->gf_dev = dmalloc((size_t)in_dim * 4, &err);
    q->u1 = dmalloc(H * 4, &err);
    if (ork_mlp_screen_ok(8, hidden, nhidden)) q->wpk = dmalloc((size_t)(nhidden - 1) * H * H * 2, &err);
    if (!err && hipHostMalloc((void **)&q->scal, 64, hipHostMallocDefault) != hipSuccess) err = 1;
    ork_host_prepare();
    if (err) {
        orkan_mlp_destroy(q);
        return NULL;
    }
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    for (int l = 0; l < nhidden; ++l) {
        const size_t n = (size_t)q->L[l].K * q->L[l].N;
        (void)hipMemsetAsync(q->L[l].m, 0, n * 4, st);
        (void)hipMemsetAsync(q->L[l].v, 0, n * 4, st);
        (void)hipMemsetAsync(q->L[l].mb, 0, H * 4, st);
        (void)hipMemsetAsync(q->L[l].vb, 0, H * 4, st);
    }
    (void)hipMemsetAsync(q->m_out, 0, H * 4, st);
    (void)hipMemsetAsync(q->v_out, 0, H * 4, st);
    (void)hipStreamSynchronize(st);
    return q;
}

void orkan_mlp_destroy(orkan_mlp_t *q) {
    if (!q) return;
    (void)hipStreamSynchronize((hipStream_t)ork_dev()->stream);
    for (int l = 0; l < MLP_MAX_LAYERS; ++l) {
        layer_t *L = &q->L[l];
        void *p[] = {L->w, L->g, L->m, L->v, L->b, L->gb, L->mb, L->vb, L->wb, L->wtb, q->pre[l], q->act[l],
                     l == q->nl - 1 ? q->dpre[l] : NULL};
        for (size_t i = 0; i < sizeof(p) / sizeof(p[0]); ++i)
            if (p[i]) (void)hipFree(p[i]);
    }
    void *p[] = {q->w_out, q->g_out, q->m_out, q->v_out, q->x32, q->x16, q->y, q->dy, q->sq, q->tgt,
                 q->colpart, q->gf_dev, q->u1, q->wpk, q->transposes};
    for (size_t i = 0; i < sizeof(p) / sizeof(p[0]); ++i)
        if (p[i]) (void)hipFree(p[i]);
    if (q->scal) (void)hipHostFree(q->scal);
    free(q);
}

/* one Adam launch: with `all` a step of every weight matrix, bias and the head, without it the bf16 copies of the weight
 * matrices rewritten and their moments cleared */
static int adam(orkan_mlp_t *q, int all, float lr, float b1, float b2, float eps, float c1, float c2) {
    float *w[2 * MLP_MAX_LAYERS + 1], *m[2 * MLP_MAX_LAYERS + 1], *v[2 * MLP_MAX_LAYERS + 1];
    const float *g[2 * MLP_MAX_LAYERS + 1];
    void *wb[2 * MLP_MAX_LAYERS + 1], *wtb[2 * MLP_MAX_LAYERS + 1];
    int rows[2 * MLP_MAX_LAYERS + 1], cols[2 * MLP_MAX_LAYERS + 1], n = 0;
    for (int l = 0; l < q->nl; ++l, ++n) {
        const layer_t *L = &q->L[l];
        w[n] = L->w; g[n] = all ? L->g : NULL; m[n] = L->m; v[n] = L->v;
        wb[n] = L->wb; wtb[n] = L->wtb; rows[n] = L->K; cols[n] = L->N;
    }
    for (int l = 0; all && l <= q->nl; ++l, ++n) {
        const layer_t *L = &q->L[l < q->nl ? l : 0];
        const int head = l == q->nl;
        w[n] = head ? q->w_out : L->b; g[n] = head ? q->g_out : L->gb;
        m[n] = head ? q->m_out : L->mb; v[n] = head ? q->v_out : L->vb;
        wb[n] = wtb[n] = NULL; rows[n] = 1; cols[n] = q->hidden;
    }
    return ork_mlp_adam_all(ork_dev()->stream, n, w, g, m, v, wb, wtb, rows, cols, lr, b1, b2, eps, c1, c2);
}

/* W[l]: fp32 [K_l][hidden] row-major; b[l]: [hidden]; w_out: [hidden] */
int orkan_mlp_set_weights(orkan_mlp_t *q, const float *const *W, const float *const *b, const float *w_out,
                          float b_out) {
    if (!q) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    int e = 0;
    for (int l = 0; l < q->nl && !e; ++l) {
        layer_t *L = &q->L[l];
        e |= (int)hipMemcpyAsync(L->w, W[l], (size_t)L->K * L->N * 4, hipMemcpyHostToDevice, st);
        e |= (int)hipMemcpyAsync(L->b, b[l], (size_t)L->N * 4, hipMemcpyHostToDevice, st);
    }
    if (!e) e = adam(q, 0, 0.0f, 0.0f, 0.0f, 1.0f, 1.0f, 1.0f);
    if (!e) e = (int)hipMemcpyAsync(q->w_out, w_out, (size_t)q->hidden * 4, hipMemcpyHostToDevice, st);
    q->b_out = b_out;
    if (!e) e = (int)hipStreamSynchronize(st);
    return e;
}

int orkan_mlp_get_weights(orkan_mlp_t *q, float *const *W, float *const *b, float *w_out, float *b_out) {
    if (!q) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    int e = 0;
    /* into pageable memory: packed by one kernel into pinned memory, copied from there by the host (2.4 MB of a 128 ->
     * 512 -> 512 -> 512 -> 1 network: 240 us with a copy per array, 134 so, 44 of them the kernel) */
    const float *src[2 * MLP_MAX_LAYERS + 1];
    float *dst[2 * MLP_MAX_LAYERS + 1];
    int len[2 * MLP_MAX_LAYERS + 1], n = 0, host = 1;
    size_t total = 0;
    for (int l = 0; l < q->nl; ++l) {
        const layer_t *L = &q->L[l];
        if (W && W[l]) {
            src[n] = L->w; dst[n] = W[l]; len[n++] = L->K * L->N;
        }
        if (b && b[l]) {
            src[n] = L->b; dst[n] = b[l]; len[n++] = L->N;
        }
    }
    if (w_out) {
        src[n] = q->w_out; dst[n] = w_out; len[n++] = q->hidden;
    }
    for (int i = 0; i < n; ++i) {
        total += (size_t)len[i];
        host &= ork_is_pageable(dst[i]);
    }
    float *buf = n && host && total <= ORK_HOST_FLOATS ? ork_host_take() : NULL;
    if (buf) {
        e = ork_mlp_pack(st, n, src, len, buf);
        const int es = (int)hipStreamSynchronize(st);
        if (!e) e = es;
        const float *from = buf;
        for (int i = 0; i < n && !e; from += len[i++]) memcpy(dst[i], from, (size_t)len[i] * 4);
        ork_host_give();
        if (b_out) *b_out = q->b_out;
        return e;
    }
    for (int l = 0; l < q->nl; ++l) {
        layer_t *L = &q->L[l];
        if (W && W[l]) e |= (int)hipMemcpyAsync(W[l], L->w, (size_t)L->K * L->N * 4, hipMemcpyDeviceToHost, st);
        if (b && b[l]) e |= (int)hipMemcpyAsync(b[l], L->b, (size_t)L->N * 4, hipMemcpyDeviceToHost, st);
    }
    if (w_out) e |= (int)hipMemcpyAsync(w_out, q->w_out, (size_t)q->hidden * 4, hipMemcpyDeviceToHost, st);
    if (b_out) *b_out = q->b_out;
    e |= (int)hipStreamSynchronize(st);
    return e;
}

/* forward over rows [0, Mp) of the staged bf16 input; for training it keeps the pre-activations and the transposed
 * activations */
static int forward_rows(orkan_mlp_t *q, int Mp, int training) {
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    const void *in = q->x16;
    int ld = q->in_dim;
    for (int l = 0; l < q->nl; ++l) {
        layer_t *L = &q->L[l];
        int e;
        if (training)
            e = ork_mlp_gemm(st, 1, in, ld, L->wtb, L->K, Mp, L->N, L->K, NULL, L->N, L->b, q->pre[l], q->act[l],
                                 l + 1 < q->nl ? q->in_t[l + 1] : NULL, (long)Mp + TPAD);
        else
            e = ork_mlp_gemm(st, 1, in, ld, L->wtb, L->K, Mp, L->N, L->K, NULL, L->N, L->b, NULL, q->act[l], NULL, 0);
        if (e) return e;
        in = q->act[l];
        ld = L->N;
    }
    return 0;
}

/* x (host or device) -> bf16, padding rows zero */
static int stage_input(orkan_mlp_t *q, const float *x, int rows, int Mp) {
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    int e = (int)hipMemcpyAsync(q->x32, x, (size_t)rows * q->in_dim * 4, hipMemcpyDefault, st);
    if (!e) e = ork_mlp_stage_input(st, q->x32, 0, Mp, rows, q->in_dim, q->x16, NULL, 0, NULL, NULL);
    return e;
}

/* A training batch, x and target in host or device memory: x as in stage_input, its transpose and the targets.  Pageable
 * batches that fit go through pinned memory, which the kernel reads as the host fills it, unless another thread's batch is on
 * its way there; wait_batch gives it back.  A step of 4096 rows of 128: 245 us
 * with hipMemcpy and a copy of the loss back, 195 so (130 with the batch on the device). */
static int stage_batch(orkan_mlp_t *q, const float *x, const float *target, int rows, int Mp) {
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    const size_t K = (size_t)q->in_dim;
    const long ldt = (long)Mp + TPAD;
    if (x && target && (size_t)rows * (K + 1) <= ORK_HOST_FLOATS && ork_is_pageable(x) && ork_is_pageable(target))
        q->host = ork_host_take();
    if (q->host) {
        float *hx = q->host, *ht = hx + (size_t)rows * K;
        memcpy(ht, target, (size_t)rows * 4);
        int chunk = (int)(CHUNK_FLOATS / K) & ~63, e = 0;
        if (chunk < 64) chunk = 64;
        for (int m0 = 0; m0 < Mp && !e; m0 += chunk) {
            const int m1 = Mp - m0 < chunk ? Mp : m0 + chunk, r1 = m1 < rows ? m1 : rows;
            if (r1 > m0) memcpy(hx + (size_t)m0 * K, x + (size_t)m0 * K, (size_t)(r1 - m0) * K * 4);
            e = ork_mlp_stage_input(st, hx, m0, m1, rows, q->in_dim, q->x16, q->in_t[0], ldt, ht, q->tgt);
        }
        return e;
    }
    int e = (int)hipMemcpyAsync(q->x32, x, (size_t)rows * K * 4, hipMemcpyDefault, st);
    if (!e) e = (int)hipMemcpyAsync(q->tgt, target, (size_t)rows * 4, hipMemcpyDefault, st);
    if (!e) e = ork_mlp_stage_input(st, q->x32, 0, Mp, rows, q->in_dim, q->x16, q->in_t[0], ldt, NULL, NULL);
    return e;
}

/* the end of a call that staged a batch; e: its error so far */
static int wait_batch(orkan_mlp_t *q, int e) {
    const int es = (int)hipStreamSynchronize((hipStream_t)ork_dev()->stream);
    if (q->host) ork_host_give();
    q->host = NULL;
    return e ? e : es;
}

/* y[i] for batch rows of x (host or device pointer, [batch][in_dim] fp32); any batch size */
int orkan_mlp_forward(orkan_mlp_t *q, int batch, const float *x, float *y) {
    if (!q || batch < 0) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    for (int r0 = 0; r0 < batch; r0 += q->max_batch) {
        const int rows = batch - r0 < q->max_batch ? batch - r0 : q->max_batch;
        const int Mp = pad_rows(rows);
        int e = stage_input(q, x + (size_t)r0 * q->in_dim, rows, Mp);
        if (!e) e = forward_rows(q, Mp, 0);
        if (!e) e = ork_mlp_head_forward(st, q->act[q->nl - 1], q->w_out, q->b_out, Mp, q->hidden, q->y, NULL, NULL,
                                         NULL, rows, 1.0f);
        if (!e) e = (int)hipMemcpyAsync(y + r0, q->y, (size_t)rows * 4, hipMemcpyDefault, st);
        if (e) return e;
    }
    return (int)hipStreamSynchronize(st);
}

/* Screening: rows r = 0..ncand-1 are [gf (ng floats), angles_dev[r] (in_dim - ng floats)]; y_dev receives ncand
 * predictions.  The graph features' share of layer 1 is computed once.  8 angles (p = 4) and a width of 128, 256 or 512
 * run through every layer in one kernel (k_screen.hip: a tile of activations and two workgroups fit a CU's LDS, the
 * accumulators its registers); other shapes go layer by layer, in chunks of max_batch rows.  Both give the same bits. */
int orkan_mlp_forward_candidates(orkan_mlp_t *q, const float *gf_host, int ng, const float *angles_dev, long ncand,
                                 float *y_dev) {
    if (!q || ng <= 0 || ng >= q->in_dim || ncand < 0) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    const int na = q->in_dim - ng, H = q->hidden;
    const layer_t *L0 = &q->L[0];
    int e = (int)hipMemcpyAsync(q->gf_dev, gf_host, (size_t)ng * 4, hipMemcpyHostToDevice, st);
    if (!e && ork_mlp_screen_ok(na, H, q->nl)) {
        const void *wt[MLP_MAX_LAYERS];
        const float *bias[MLP_MAX_LAYERS];
        for (int l = 0; l < q->nl; ++l) {
            bias[l] = q->L[l].b;
            if (l) wt[l - 1] = q->L[l].wtb;
        }
        e = ork_mlp_screen(st, q->gf_dev, ng, L0->wb, wt, q->wpk, q->u1, bias, q->nl, H, q->w_out, q->b_out, angles_dev,
                           ncand, y_dev);
        if (!e) e = (int)hipStreamSynchronize(st);
        return e;
    }
    if (!e) e = ork_mlp_first_layer_graph(st, q->gf_dev, ng, L0->wb, H, q->u1);
    for (long r0 = 0; r0 < ncand && !e; r0 += q->max_batch) {
        const int rows = (int)(ncand - r0 < q->max_batch ? ncand - r0 : q->max_batch);
        const int Mp = pad_rows(rows);
        e = ork_mlp_first_layer_rows(st, angles_dev, na, r0, rows, Mp, q->u1, (const char *)L0->wb + (size_t)ng * H * 2,
                                     L0->b, H, q->act[0]);
        const void *in = q->act[0];
        for (int l = 1; l < q->nl && !e; ++l) {
            layer_t *L = &q->L[l];
            e = ork_mlp_gemm(st, 1, in, L->K, L->wtb, L->K, Mp, L->N, L->K, NULL, L->N, L->b, NULL, q->act[l], NULL, 0);
            in = q->act[l];
        }
        if (!e) e = ork_mlp_head_forward(st, q->act[q->nl - 1], q->w_out, q->b_out, Mp, H, y_dev + r0, NULL, NULL,
                                         NULL, rows, 1.0f);
    }
    if (!e) e = (int)hipStreamSynchronize(st);
    return e;
}

/* gradients of the mean squared error of the staged batch into the g buffers; the sum of squared errors and
 * d loss / d b_out into scal[0] and scal[1].  Ten launches for three layers, besides the batch's and Adam's (4096 rows of a
 * 128 -> 512 -> 512 -> 512 -> 1 network: 190 us a step from a host batch, 125 from a device one; four host steps and a
 * read of the weights 895 us, 2190 with a launch per layer and operand, 37 a step) */
static int backward(orkan_mlp_t *q, int rows) {
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    const int Mp = pad_rows(rows), H = q->hidden, nl = q->nl;
    const long ldt = (long)Mp + TPAD;
    int e = forward_rows(q, Mp, 1);
    if (!e) e = ork_mlp_head_forward(st, q->act[nl - 1], q->w_out, q->b_out, Mp, H, q->y, q->tgt, q->dy, q->sq,
                                     rows, 1.0f / (float)rows);
    if (!e) e = ork_mlp_head_backward_t(st, q->dy, q->w_out, q->pre[nl - 1], Mp, H, q->dpre[nl - 1], q->dpre_t[nl - 1],
                                        ldt);
    /* dP_{l-1} = (dP_l W_l^T) * gelu'(pre_{l-1}) */
    for (int l = nl - 1; l > 0 && !e; --l) {
        layer_t *L = &q->L[l];
        e = ork_mlp_gemm(st, 2, q->dpre[l], L->N, L->wb, L->N, Mp, L->K, L->N, NULL, L->K, NULL, q->pre[l - 1],
                             q->dpre[l - 1], q->dpre_t[l - 1], ldt);
    }
    const void *xt[MLP_MAX_LAYERS], *dt[MLP_MAX_LAYERS], *cols[MLP_MAX_LAYERS + 1];
    const float *scale[MLP_MAX_LAYERS + 1];
    float *gw[MLP_MAX_LAYERS], *gc[MLP_MAX_LAYERS + 1];
    int K[MLP_MAX_LAYERS];
    for (int l = 0; l < nl; ++l) {
        xt[l] = q->in_t[l];
        dt[l] = q->dpre_t[l];
        gw[l] = q->L[l].g;
        K[l] = q->L[l].K;
        cols[l] = q->dpre[l];
        scale[l] = NULL;
        gc[l] = q->L[l].gb;
    }
    cols[nl] = q->act[nl - 1];
    scale[nl] = q->dy;
    gc[nl] = q->g_out;
    /* dW_l = X_l^T dP_l */
    if (!e) e = ork_mlp_weight_grads(st, nl, xt, dt, gw, K, H, Mp, ldt, SPLITK_MAX);
    if (!e) e = ork_mlp_colsums(st, nl + 1, cols, scale, gc, Mp, H, q->colpart, q->sq, q->dy, q->scal);
    return e;
}

int orkan_mlp_train_step(orkan_mlp_t *q, int batch, const float *x, const float *target, float lr, float *loss) {
    if (!q || batch <= 0 || batch > q->max_batch) return (int)hipErrorInvalidValue;
    int e = stage_batch(q, x, target, batch, pad_rows(batch));
    if (!e) e = backward(q, batch);
    if (e) return wait_batch(q, e);
    q->step += 1;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.0f - powf(b1, (float)q->step), c2 = 1.0f - powf(b2, (float)q->step);
    e = adam(q, 1, lr, b1, b2, eps, c1, c2);
    e = wait_batch(q, e);
    if (e) return e;
    const float *s = q->scal, gb = s[1];
    q->mb_out = b1 * q->mb_out + (1 - b1) * gb;
    q->vb_out = b2 * q->vb_out + (1 - b2) * gb * gb;
    q->b_out -= lr * (q->mb_out / c1) / (sqrtf(q->vb_out / c2) + eps);
    if (loss) *loss = s[0] / (float)batch;
    return 0;
}

/* gradients without an update (for checking against a CPU computation) */
int orkan_mlp_grads(orkan_mlp_t *q, int batch, const float *x, const float *target, float *const *dW,
                    float *const *db, float *dw_out, float *db_out, float *loss) {
    if (!q || batch <= 0 || batch > q->max_batch) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    int e = stage_batch(q, x, target, batch, pad_rows(batch));
    if (!e) e = backward(q, batch);
    for (int l = 0; l < q->nl && !e; ++l) {
        if (dW && dW[l]) e |= (int)hipMemcpyAsync(dW[l], q->L[l].g, (size_t)q->L[l].K * q->L[l].N * 4,
                                                   hipMemcpyDeviceToHost, st);
        if (db && db[l]) e |= (int)hipMemcpyAsync(db[l], q->L[l].gb, (size_t)q->L[l].N * 4, hipMemcpyDeviceToHost, st);
    }
    if (!e && dw_out) e = (int)hipMemcpyAsync(dw_out, q->g_out, (size_t)q->hidden * 4, hipMemcpyDeviceToHost, st);
    e = wait_batch(q, e);
    const float *s = q->scal;
    if (!e && db_out) *db_out = s[1];
    if (!e && loss) *loss = s[0] / (float)batch;
    return e;
}

unsigned long ork_topk_state_bytes(void);
int ork_topk(void *stream, const float *y, long n, int k, int *idx, float *vals, void *st_dev);

/* indices of the k largest entries of the device array y_dev (n floats), largest first, ties
 * by ascending index; values optional.  Selection on the device (radix select), the k
 * survivors ordered on the host. */
static int topk_after(const float *vals, const int *idx, int a, int b) {
    return vals[a] < vals[b] || (vals[a] == vals[b] && idx[a] > idx[b]);
}

/* the k positions by value, descending, then index, ascending: runs of 32 by insertion, then merges between the halves of
 * ord (2 k ints); the half that holds the result.  (By insertion alone k = 65536 took 340 to 430 ms.) */
static const int *topk_order(const float *vals, const int *idx, int k, int *ord) {
    int *from = ord, *to = ord + k;
    for (int r = 0; r < k; r += 32) {
        const int end = k - r < 32 ? k : r + 32;
        for (int a = r; a < end; ++a) {
            int b = a;
            for (; b > r && topk_after(vals, idx, from[b - 1], a); --b) from[b] = from[b - 1];
            from[b] = a;
        }
    }
    for (int len = 32; len < k; len *= 2) {
        for (int r = 0; r < k; r += 2 * len) {
            const int mid = k - r < len ? k : r + len, end = k - mid < len ? k : mid + len;
            for (int a = r, b = mid, o = r; o < end; ++o)
                to[o] = b == end || (a < mid && !topk_after(vals, idx, from[a], from[b])) ? from[a++] : from[b++];
        }
        int *t = from;
        from = to;
        to = t;
    }
    return from;
}

int orkan_topk_f32(const float *y_dev, long n, int k, int *idx_host, float *val_host) {
    if (!y_dev || !idx_host || k <= 0 || k > n || k > 65536) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    void *scratch = ork_mem_get(ork_topk_state_bytes() + (size_t)k * (sizeof(int) + sizeof(float)));
    int e = scratch ? 0 : (int)hipErrorOutOfMemory;
    float *vals = malloc((size_t)k * sizeof(float));
    int *idx = malloc((size_t)k * sizeof(int));
    int *ord = malloc((size_t)k * 2 * sizeof(int));
    if (!vals || !idx || !ord) e = (int)hipErrorOutOfMemory;
    int *idx_d = (int *)((char *)scratch + ork_topk_state_bytes());
    float *val_d = (float *)(idx_d + k);
    if (!e) e = ork_topk(st, y_dev, n, k, idx_d, val_d, scratch);
    if (!e) e = (int)hipMemcpyAsync(idx, idx_d, (size_t)k * sizeof(int), hipMemcpyDeviceToHost, st);
    if (!e) e = (int)hipMemcpyAsync(vals, val_d, (size_t)k * sizeof(float), hipMemcpyDeviceToHost, st);
    if (!e) e = (int)hipStreamSynchronize(st);
    if (!e) {
        const int *sorted = topk_order(vals, idx, k, ord);
        for (int i = 0; i < k; ++i) {
            idx_host[i] = idx[sorted[i]];
            if (val_host) val_host[i] = vals[sorted[i]];
        }
    }
    free(vals);
    free(idx);
    free(ord);
    ork_mem_put(scratch);
    return e;
}

/* C = A B^T for bf16 A [M][K], B [N][K] (device pointers), fp32 C [M][N]: exposed for testing the MFMA GEMM */
int orkan_mlp_gemm_test(int M, int N, int K, const void *A, const void *B, float *C) {
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    int e = ork_mlp_gemm(st, 0, A, K, B, K, M, N, K, C, N, NULL, NULL, NULL, NULL, 0);
    if (!e) e = (int)hipStreamSynchronize(st);
    return e;
}
