/*
 * ork_sample.c -- sample_matrix on the device (no reference implementation; the operation is
 * specified in the reference's docs/SAMPLE_MATRIX.md:1-80, its recommended algorithm in §6 there).
 *
 *   1. channels 0 .. lstar-1 are applied to iota in place (prefix shared by every leaf);
 *   2. leaves |psi_a> are built in blocks of B: copies of the prefix, M_lstar[a], then the channels after lstar, each
 *      as sum_m w[m] M[m] psi.  A channel takes T leaves at a time: every operation but the last runs on a copy of
 *      them, the last on the leaves themselves, and the copies and sums are one launch per T leaves each.  Leaf by leaf
 *      a channel of two operations took 7 launches per leaf, 5 of them copies and sums.
 *   3. for every block pair (i >= j) the block G = Phi_i^dagger diag(obs) Phi_j is one product
 *      kernel; entries with a >= b are kept and mirrored, the diagonal's imaginary part zeroed.
 * Peak: iota + 2T scratch + 2B leaves, or B leaves where one block holds them all (B from the workspace budget, at most
 * 64; T from what the leaves leave of it); every allocation happens at entry.  The operations are the caller's qop_t,
 * called on PURE states whose data are the library's device buffers, so they run through this library's gates.
 */
#include "ork_host.h"
#include "sample.h"

#include <string.h>
#include <hip/hip_runtime_api.h>

unsigned ork_sm_max_block(void);
unsigned ork_sm_parts(uint64_t N);
int ork_sm_axpy(void *stream, void *acc, const void *v, double wr, double wi, uint64_t n, int first);
int ork_sm_spread(void *stream, void *dst, const void *src, uint64_t n, uint64_t stride, int cnt);
int ork_sm_combine(void *stream, void *x, const void *a, double war, double wai, int scaled, double wr, double wi,
                   uint64_t n);
int ork_sm_block(void *stream, const void *P, int na, const void *Q, int nb, const double *obs, uint64_t N,
                 uint64_t stride, int same, void *part, void *G);

typedef struct {
    void *stream;
    qubit_t n;
    idx_t N;
    idx_t stride;            /* leaves and scratch vectors are this far apart */
    cplx_t *tmp, *acc;       /* linear-combination scratch, T vectors each */
    int T;
} lcu_t;

static void run_op(qop_t op, cplx_t *data, qubit_t n) {
    state_t s;
    s.type = PURE;
    s.data = data;
    s.qubits = n;
    op(&s);
}

/* psi <- sum_m w[m] M[m] psi for cnt <= T vectors */
static int apply_channel(lcu_t *c, cplx_t *psi, int cnt, const ansatz_channel_t *ch) {
    const idx_t len = c->stride * (idx_t)(cnt - 1) + c->N;   /* the gaps between vectors go along */
    const uint64_t M = ch->n_ops;
    for (uint64_t m = 0; m + 1 < M; ++m) {
        int e = (int)hipMemcpyAsync(c->tmp, psi, (size_t)len * sizeof(cplx_t), hipMemcpyDeviceToDevice,
                                    (hipStream_t)c->stream);
        if (e) return e;
        for (int i = 0; i < cnt; ++i) run_op(ch->ops[m], c->tmp + (size_t)i * c->stride, c->n);
        if (M > 2) e = ork_sm_axpy(c->stream, c->acc, c->tmp, creal(ch->weights[m]), cimag(ch->weights[m]), len, m == 0);
        if (e) return e;
    }
    /* the last operation needs no copy; of two operations the first one's weight waits for the sum */
    for (int i = 0; i < cnt; ++i) run_op(ch->ops[M - 1], psi + (size_t)i * c->stride, c->n);
    const cplx_t w0 = ch->weights[0], w = ch->weights[M - 1];
    return ork_sm_combine(c->stream, psi, M == 1 ? NULL : M == 2 ? c->tmp : c->acc, creal(w0), cimag(w0), M == 2,
                          creal(w), cimag(w), len);
}

/* leaves a0 .. a0 + cnt - 1 into blk (cnt vectors of N) */
static int build_leaves(lcu_t *c, cplx_t *blk, const cplx_t *prefix, const ansatz_channel_t *chs, uint64_t nch,
                        uint64_t lstar, uint64_t a0, int cnt) {
    int e = ork_sm_spread(c->stream, blk, prefix, c->N, c->stride, cnt);
    for (int i0 = 0; i0 < cnt && !e; i0 += c->T) {
        const int t = cnt - i0 < c->T ? cnt - i0 : c->T;
        cplx_t *leaves = blk + (size_t)i0 * c->stride;
        for (int i = 0; i < t; ++i) run_op(chs[lstar].ops[a0 + (uint64_t)(i0 + i)], leaves + (size_t)i * c->stride, c->n);
        for (uint64_t l = lstar + 1; l < nch && !e; ++l) e = apply_channel(c, leaves, t, &chs[l]);
    }
    return e;
}

qs_error_t sample_matrix(state_t *iota, const double *obs, const ansatz_channel_t *channels, uint64_t n_channels,
                         uint64_t lstar, size_t workspace_bytes, cplx_t *S) {
    if (!iota || !iota->data || !obs || !channels || !S) return QS_ERR_NULL;
    if (iota->type != PURE) return QS_ERR_TYPE;
    if (lstar >= n_channels) return QS_ERR_PARAM;
    for (uint64_t l = 0; l < n_channels; ++l) {
        if (channels[l].n_ops == 0 || !channels[l].ops) return QS_ERR_PARAM;
        if (l != lstar && !channels[l].weights) return QS_ERR_PARAM;
        for (uint64_t m = 0; m < channels[l].n_ops; ++m)
            if (!channels[l].ops[m]) return QS_ERR_NULL;
    }
    const qubit_t n = iota->qubits;
    const idx_t N = (idx_t)1 << n;
    const uint64_t K = channels[lstar].n_ops;
    const size_t vec = (size_t)N * sizeof(cplx_t);
    const size_t nvec = workspace_bytes / vec;
    if (nvec < 4) return QS_ERR_PARAM;
    uint64_t B = (nvec - 2) / 2;
    if (B > ork_sm_max_block()) B = ork_sm_max_block();
    if (B > K) B = K;
    /* the scratch takes what the leaves leave of the budget: at least the two vectors set aside above */
    const int one_block = B == K;
    uint64_t T = (nvec - (one_block ? B : 2 * B)) / 2;
    if (T > B) T = B;
    /* vectors a power of two apart share memory channels; the gap is left out where it would not fit the budget */
    const uint64_t held = (one_block ? B : 2 * B) + 2 * T;
    const idx_t stride = N >= 4096 && held * (vec + 64 * sizeof(cplx_t)) <= workspace_bytes ? N + 64 : N;
    const size_t svec = (size_t)stride * sizeof(cplx_t);

    /* no library lock is held while the caller's operations run (they may call exp_diag or mean,
     * which stage their arrays in the shared buffer): obs gets a buffer of its own */
    ork_dev_t *d = ork_dev();
    const size_t part_bytes = (size_t)ork_sm_parts(N) * B * B * sizeof(cplx_t);
    cplx_t *tmp = NULL, *acc = NULL, *phj = NULL, *phi = NULL, *part = NULL, *G = NULL;
    double *o = NULL;
    cplx_t *Gh = malloc((size_t)B * B * sizeof(cplx_t));
    qs_error_t rc = Gh ? QS_OK : QS_ERR_OOM;
    int sums = 0;   /* a combination of more than two operations needs a running sum */
    for (uint64_t l = 0; l < n_channels; ++l) sums |= l != lstar && channels[l].n_ops > 2;
    if (rc == QS_OK && (!(phj = ork_mem_get(svec * B)) || (!one_block && !(phi = ork_mem_get(svec * B))) ||
                        !(part = ork_mem_get(part_bytes)) || !(G = ork_mem_get((size_t)B * B * sizeof(cplx_t))) ||
                        !(o = ork_mem_get((size_t)N * sizeof(double)))))
        rc = QS_ERR_OOM;
    while (rc == QS_OK && (!(tmp = ork_mem_get(svec * T)) || (sums && !(acc = ork_mem_get(svec * T))))) {
        ork_mem_put(tmp);
        tmp = NULL;
        if (T == 1) rc = QS_ERR_OOM;
        T = 1;   /* the budget allows more than the device has left */
    }
    int e = 0;
    if (rc == QS_OK)
        e = (int)hipMemcpyAsync(o, obs, (size_t)N * sizeof(double), hipMemcpyDefault, (hipStream_t)d->stream);
    lcu_t c = {d->stream, n, N, stride, tmp, acc, (int)T};
    /* 1. prefix */
    for (uint64_t l = 0; rc == QS_OK && !e && l < lstar; ++l) e = apply_channel(&c, iota->data, 1, &channels[l]);
    /* 2-3. blocks */
    for (uint64_t j0 = 0; rc == QS_OK && !e && j0 < K; j0 += B) {
        const int nj = (int)(K - j0 < B ? K - j0 : B);
        e = build_leaves(&c, phj, iota->data, channels, n_channels, lstar, j0, nj);
        for (uint64_t i0 = j0; !e && i0 < K; i0 += B) {
            const int ni = (int)(K - i0 < B ? K - i0 : B);
            const cplx_t *P = phj;
            if (i0 != j0) {
                e = build_leaves(&c, phi, iota->data, channels, n_channels, lstar, i0, ni);
                P = phi;
            }
            if (!e) e = ork_sm_block(d->stream, P, ni, phj, nj, o, N, stride, i0 == j0, part, G);
            if (!e) e = (int)hipMemcpyAsync(Gh, G, (size_t)ni * nj * sizeof(cplx_t), hipMemcpyDeviceToHost,
                                            (hipStream_t)d->stream);
            if (!e) e = (int)hipStreamSynchronize((hipStream_t)d->stream);
            for (int a = 0; !e && a < ni; ++a)
                for (int b = 0; b < nj; ++b) {
                    const uint64_t ia = i0 + (uint64_t)a, jb = j0 + (uint64_t)b;
                    if (ia < jb) continue;
                    cplx_t v = Gh[a * nj + b];
                    if (ia == jb) v = CMPLX(creal(v), 0.0);
                    S[ia + jb * K] = v;
                    S[jb + ia * K] = conj(v);
                }
        }
    }
    (void)hipStreamSynchronize((hipStream_t)d->stream);
    void *bufs[] = {tmp, acc, phj, phi, part, G, o};
    for (size_t i = 0; i < sizeof(bufs) / sizeof(bufs[0]); ++i) ork_mem_put(bufs[i]);
    free(Gh);
    if (e) ork_hip_fail("sample_matrix", e);   /* a failed HIP call exits like every other entry point */
    return rc;
}
