/*
 * ork_qaoa.c -- host side of the batched QAOA launcher: device arenas for the
 * cost diagonals, the evaluation list and the state scratch; the launches of the
 * register kernels, one per sweep over every evaluation (12, 256: the default);
 * for the LDS shapes a hipGraph holding the counter reset and the persistent
 * kernel; and the autotuner that picks among them.
 *
 * No reference counterpart: the reference evaluates one circuit per call
 * sequence (state_plus, exp_diag, rx, mean).  Each evaluation here computes
 * exactly that sequence.
 */
#include "ork_host.h"

#include <math.h>
#include <string.h>
#include <hip/hip_runtime_api.h>

int ork_qaoa_launch(void *stream, int lt, int threads, int grid, const void *evals, const int *order,
                    const int *nevals, const void *graphs, const double *angles, const double *diag, void *states,
                    uint64_t slot_elems, double *out, unsigned *counter);
int ork_qaoa_occupancy(int lt, int threads, int *blocks_per_cu);
int ork_qaoa_sweeps(void *stream, int sym, int deep, const void *recs, const int *n, const int *p, int count, const double *angles,
                    const double *diag, void *states, double *part, double *out);
int ork_qaoa_stage(void *stream, const double *gb, uint64_t rows, double *angles, const void *recs, int nrecs, void *recs_dst);
int ork_qaoa_rescale(void *stream, const void *recs_dev, int count, double *angles);
int ork_qaoa_diag_info(void *stream, int ngraphs, int nmax, const void *graphs, const double *diag, uint64_t *info);
int ork_maxcut_diag(void *stream, double *out, int n, int ne, const int *ei, const int *ej, const double *w);

typedef struct { int graph, p, angle_off, pad; } q_eval_t;
typedef struct { uint64_t diag_off, state_off; int n, pad; } q_graph_t;
typedef struct { uint64_t diag_off, tile; int angle_off, p, n, m, out, pad; } q_rec_t;

struct orkan_qaoa {
    int ngraphs, max_evals, max_p, nmax;
    q_graph_t *graphs_h;
    void *graphs_d;
    double *diag_d;
    void *evals_d;
    int *order_d, *nevals_d;
    double *angles_d;
    unsigned *counter_d;
    void *states_d;
    size_t states_bytes;
    /* launch configuration */
    int lt, threads, grid;
    /* the graph is captured on this private stream, never on the library stream that other
     * threads' gates and reductions use, and replayed on the library stream */
    hipStream_t capture_stream;
    int nevals_h;          /* host source of the nevals_d upload */
    double *info_h;        /* per graph: largest |C|; 1 if C(x) = C(~x) for every x, else 0 */
    /* the register kernels' list: records sorted by form, then index bits, then layers, all descending; n_h: index bits */
    q_rec_t *recs_h;
    void *recs_d;
    int *n_h, *p_h, *start_h, nstaged;
    unsigned char *sym_h;
    int states_short;      /* the device had no memory for all the scratch asked for */
    size_t room;           /* tiles per round of launches, as the staged records number them */
    int deep;              /* the staged list holds a circuit that needs scalings (DEEP) */
    int wide;              /* the staged list holds a phase too large for the register kernel's sincos */
    hipGraph_t graph;
    hipGraphExec_t exec;
    int graph_ok;
    /* host staging */
    q_eval_t *evals_h;
    int *order_h;
    double *gb_h, *out_h;  /* rows of gamma, then of beta; the results */
    void *pinned;          /* gb_h, out_h and recs_h: each allocation and release of pinned memory takes 30 us and more */
};

static int cus(void) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
    return n;
}

/* the register kernels (2^12 amplitudes per workgroup of 256 threads) take phases gamma C up to this; larger ones, and ones
 * that are not finite, run through the LDS kernel, whose sincos reduces any argument */
#define REG_LT 12
#define REG_THREADS 256
#define REG_PHASE_MAX 1125899906842624.0   /* 2^50 */
#define WIDE_THREADS 512
/* qubits times layers from which a state's squared norm may outgrow the number range unless it is scaled down on the way */
#define DEEP 768
#define TILE_BYTES ((size_t)16 << REG_LT)
/* state slots of the register kernels: evaluations beyond them go in further rounds of launches. 4096 evaluations of 10 to
 * 20 qubits, half states: 15.0 ms a call with 128 to 176 MB, which the last-level cache can hold from one sweep to the next;
 * 17.3 with 64 MB, 16.2 with 256, 15.3 with 1 GB; 14.95 in one round, which takes 6.3 GB */
#define SWEEP_BYTES ((size_t)128 << 20)

static int is_reg(const orkan_qaoa_t *q) { return q->lt == REG_LT && q->threads == REG_THREADS; }

static void drop_graph(orkan_qaoa_t *q) {
    if (q->graph_ok) {
        (void)hipGraphExecDestroy(q->exec);
        (void)hipGraphDestroy(q->graph);
    }
    q->graph_ok = 0;
}

/* scratch of the register kernels: a slot for each evaluation up to SWEEP_BYTES, at least one of the largest state, and 8 B
 * per tile for the partial sums */
static size_t reg_bytes(const orkan_qaoa_t *q) {
    if (q->nmax <= REG_LT) return 16;
    const size_t slot = (size_t)16 << q->nmax;
    size_t all = 0;
    for (int g = 0; g < q->ngraphs; ++g)
        if (q->graphs_h[g].n > REG_LT) all += (size_t)16 << q->graphs_h[g].n;
    const size_t rounds = ((size_t)q->max_evals + q->ngraphs - 1) / q->ngraphs;
    size_t need = all > SWEEP_BYTES / rounds ? SWEEP_BYTES : all * rounds;
    if (need / slot > (size_t)q->max_evals) need = (size_t)q->max_evals * slot;
    if (need < slot) need = slot;
    return need + need / TILE_BYTES * sizeof(double) + 16;
}

/* The state scratch of the current configuration (and, for it, of the staged list). The LDS kernels need a slot of 2^nmax
 * for each workgroup. The register kernels take what there is, halved while memory is short down to one slot of the
 * largest state. shrink: what another configuration or list needed beyond that goes back. */
static int ensure_states(orkan_qaoa_t *q, int shrink) {
    const size_t slot = (size_t)16 << q->nmax;
    size_t need = 16, least;
    if (is_reg(q)) {
        least = (q->nmax > REG_LT ? slot + slot / TILE_BYTES * sizeof(double) : 0) + 16;
        need = reg_bytes(q);
        /* qaoa_persistent takes lists with phases beyond REG_PHASE_MAX */
        const size_t slots = q->max_evals < cus() ? (size_t)q->max_evals : (size_t)cus();
        if (q->nmax > REG_LT && q->wide && need < slots * slot) need = slots * slot;
    } else {
        if (q->nmax > q->lt) need = (size_t)q->grid * slot;
        least = need;
    }
    if ((q->states_bytes >= need || (q->states_bytes >= least && q->states_short)) &&
        !(shrink && q->states_bytes > need))
        return 0;
    if (q->states_d) {
        (void)hipStreamSynchronize((hipStream_t)ork_dev()->stream);
        (void)hipFree(q->states_d);
    }
    q->states_d = NULL;
    q->states_bytes = 0;
    q->states_short = 0;
    drop_graph(q);
    int e = ork_dev_malloc(&q->states_d, need);
    while (e && need / 2 >= least) {
        need /= 2;
        q->states_short = 1;
        e = ork_dev_malloc(&q->states_d, need);
    }
    if (e) {
        q->states_d = NULL;
        return e;
    }
    q->states_bytes = need;
    return 0;
}

/* Tiles of the register kernels that the state scratch holds, their partial sums behind them: of what they ask for, also
 * where the scratch is larger for an LDS shape or a list with wide phases, so that a list runs in the rounds that the
 * autotuner timed. */
static size_t tile_room(const orkan_qaoa_t *q) {
    const size_t want = reg_bytes(q), have = q->states_bytes < want ? q->states_bytes : want;
    return have < 16 ? 0 : (have - 16) / (TILE_BYTES + sizeof(double));
}

/* caller holds ork_lock (the state scratch may be freed and the graph dropped) */
static int set_config(orkan_qaoa_t *q, int lt, int threads, int blocks_per_cu, int shrink) {
    if (2 * lt < q->nmax) return (int)hipErrorInvalidValue;     /* pass B needs n <= 2 LT */
    int occ = 0;
    int e = ork_qaoa_occupancy(lt, threads, &occ);
    if (e) return e;
    if (occ <= 0) return (int)hipErrorInvalidConfiguration;
    if (blocks_per_cu <= 0) blocks_per_cu = occ;
    if (blocks_per_cu > occ) blocks_per_cu = occ;
    drop_graph(q);
    q->lt = lt;
    q->threads = threads;
    q->grid = cus() * blocks_per_cu;
    if (q->grid > q->max_evals) q->grid = q->max_evals;   /* a workgroup takes at least one evaluation */
    return ensure_states(q, shrink);
}

int orkan_qaoa_set_config(orkan_qaoa_t *q, int lt, int threads, int blocks_per_cu) {
    if (!q) return (int)hipErrorInvalidValue;
    ork_lock();
    const int e = set_config(q, lt, threads, blocks_per_cu, 1);
    ork_unlock();
    return e;
}

orkan_qaoa_t *orkan_qaoa_create(int ngraphs, const unsigned char *nq, const double *const *diags, int max_evals,
                                int max_p) {
    if (ngraphs <= 0 || max_evals <= 0 || max_p <= 0 || !nq || !diags) return NULL;
    orkan_qaoa_t *q = calloc(1, sizeof(*q));
    if (!q) return NULL;
    ork_dev_t *d = ork_dev();
    hipStream_t st = (hipStream_t)d->stream;
    q->ngraphs = ngraphs;
    q->max_evals = max_evals;
    q->max_p = max_p;
    q->graphs_h = calloc((size_t)ngraphs, sizeof(q_graph_t));
    q->evals_h = calloc((size_t)max_evals, sizeof(q_eval_t));
    q->order_h = calloc((size_t)max_evals, sizeof(int));
    q->info_h = calloc((size_t)ngraphs * 2, sizeof(double));
    q->sym_h = calloc((size_t)max_evals, 1);
    q->n_h = calloc((size_t)max_evals, sizeof(int));
    q->p_h = calloc((size_t)max_evals, sizeof(int));
    q->start_h = calloc((size_t)2 * 27 * (max_p + 1) + 1, sizeof(int));
    if (!q->graphs_h || !q->evals_h || !q->order_h || !q->info_h || !q->sym_h || !q->n_h || !q->p_h ||
        !q->start_h)
        goto fail;
    if (hipStreamCreateWithFlags(&q->capture_stream, hipStreamNonBlocking) != hipSuccess) {
        q->capture_stream = NULL;
        goto fail;
    }
    uint64_t total = 0;
    for (int g = 0; g < ngraphs; ++g) {
        if (nq[g] < 1 || nq[g] > 26) goto fail;
        q->graphs_h[g].n = nq[g];
        q->graphs_h[g].diag_off = total;
        total += (uint64_t)1 << nq[g];
        if (nq[g] > q->nmax) q->nmax = nq[g];
    }
    if (ork_dev_malloc((void **)&q->diag_d, total * sizeof(double)) != 0) goto fail;
    for (int g = 0; g < ngraphs; ++g)
        if (hipMemcpyAsync(q->diag_d + q->graphs_h[g].diag_off, diags[g], ((size_t)1 << nq[g]) * sizeof(double),
                           hipMemcpyDefault, st) != hipSuccess)
            goto fail;
    if (ork_dev_malloc(&q->graphs_d, (size_t)ngraphs * sizeof(q_graph_t)) != 0) goto fail;
    if (hipMemcpyAsync(q->graphs_d, q->graphs_h, (size_t)ngraphs * sizeof(q_graph_t), hipMemcpyHostToDevice, st) !=
        hipSuccess)
        goto fail;
    if (ork_dev_malloc(&q->evals_d, (size_t)max_evals * sizeof(q_eval_t)) != 0) goto fail;
    if (ork_dev_malloc(&q->recs_d, (size_t)max_evals * sizeof(q_rec_t)) != 0) goto fail;
    if (ork_dev_malloc((void **)&q->order_d, (size_t)max_evals * sizeof(int)) != 0) goto fail;
    if (ork_dev_malloc((void **)&q->nevals_d, sizeof(int)) != 0) goto fail;
    if (ork_dev_malloc((void **)&q->angles_d, (size_t)max_evals * max_p * 4 * sizeof(double)) != 0) goto fail;
    {
        const size_t rows = (size_t)max_evals * max_p * 2, info = (size_t)ngraphs * 2;
        const size_t bytes = (rows + max_evals) * sizeof(double) + (size_t)max_evals * sizeof(q_rec_t);
        if (hipHostMalloc(&q->pinned, bytes > info * sizeof(uint64_t) ? bytes : info * sizeof(uint64_t),
                          hipHostMallocDefault) != hipSuccess)
            goto fail;
        q->gb_h = q->pinned;
        q->out_h = q->gb_h + rows;
        q->recs_h = (q_rec_t *)(q->out_h + max_evals);
    }
    if (ork_dev_malloc((void **)&q->counter_d, sizeof(unsigned)) != 0) goto fail;
    {
        const size_t bytes = (size_t)ngraphs * 2 * sizeof(uint64_t);
        uint64_t *info = ork_mem_get(bytes), *host = q->pinned;
        const int bad = !info || hipMemsetAsync(info, 0, bytes, st) != hipSuccess ||
                        ork_qaoa_diag_info(st, ngraphs, q->nmax, q->graphs_d, q->diag_d, info) ||
                        hipMemcpyAsync(host, info, bytes, hipMemcpyDeviceToHost, st) != hipSuccess;
        const int waited = hipStreamSynchronize(st) == hipSuccess;
        ork_mem_put(info);
        if (bad || !waited) goto fail;
        for (int g = 0; g < ngraphs; ++g) {
            memcpy(&q->info_h[2 * g], &host[2 * g], sizeof(double));
            q->info_h[2 * g + 1] = host[2 * g + 1] == 0;
        }
    }
    {
        /* default: 4096 amplitudes in the registers of 256 threads; 8192 in LDS when the largest state needs it */
        int lt = REG_LT;
        while (2 * lt < q->nmax) ++lt;
        ork_lock();
        const int e = set_config(q, lt, lt >= 13 ? 1024 : REG_THREADS, 0, 0);
        ork_unlock();
        if (e) goto fail;
    }
    return q;
fail:
    orkan_qaoa_destroy(q);
    return NULL;
}

void orkan_qaoa_destroy(orkan_qaoa_t *q) {
    if (!q) return;
    (void)hipStreamSynchronize((hipStream_t)ork_dev()->stream);
    drop_graph(q);
    void *bufs[] = {q->graphs_d, q->diag_d, q->evals_d, q->order_d, q->nevals_d,
                    q->angles_d, q->counter_d, q->states_d, q->recs_d};
    for (size_t i = 0; i < sizeof(bufs) / sizeof(bufs[0]); ++i)
        if (bufs[i]) (void)hipFree(bufs[i]);
    if (q->pinned) (void)hipHostFree(q->pinned);
    free(q->graphs_h);
    free(q->evals_h);
    free(q->order_h);
    free(q->info_h);
    free(q->sym_h);
    free(q->n_h);
    free(q->p_h);
    free(q->start_h);
    if (q->capture_stream) (void)hipStreamDestroy(q->capture_stream);
    free(q);
}

static int capture(orkan_qaoa_t *q) {
    hipStream_t st = q->capture_stream;
    drop_graph(q);
    int e = (int)hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
    if (e) return e;
    int le = ork_qaoa_launch(st, q->lt, q->threads, q->grid, q->evals_d, q->order_d, q->nevals_d, q->graphs_d,
                             q->angles_d, q->diag_d, q->states_d, ((uint64_t)1 << q->nmax), q->out_h, q->counter_d);
    e = (int)hipStreamEndCapture(st, &q->graph);
    if (le) return le;
    if (e) return e;
    e = (int)hipGraphInstantiate(&q->exec, q->graph, NULL, NULL, 0);
    if (e) {
        (void)hipGraphDestroy(q->graph);
        return e;
    }
    q->graph_ok = 1;
    return 0;
}

static uint64_t cost(const orkan_qaoa_t *q, const q_eval_t *ev) {
    return ((uint64_t)1 << q->graphs_h[ev->graph].n) * (uint64_t)(ev->p > 0 ? ev->p : 1);
}

static const orkan_qaoa_t *g_sort_q;
static int by_cost_desc(const void *a, const void *b) {
    const q_eval_t *E = g_sort_q->evals_h;
    const uint64_t ca = cost(g_sort_q, &E[*(const int *)a]), cb = cost(g_sort_q, &E[*(const int *)b]);
    if (ca != cb) return ca < cb ? 1 : -1;
    return *(const int *)a - *(const int *)b;
}

/* half of the state: a cost with C(x) = C(~x) whose state is larger than a tile.  A tile costs the same whatever part of it
 * a state fills, and the half's X on the qubit left out takes an exchange more. */
static int is_sym(const orkan_qaoa_t *q, int graph) {
    return q->info_h[2 * graph + 1] != 0.0 && q->graphs_h[graph].n > REG_LT;
}

/* the register kernels' records: a counting sort by form (half states first), index bits and layers, all descending */
static int rec_key(const orkan_qaoa_t *q, const q_eval_t *ev) {
    const int sym = is_sym(q, ev->graph);
    return ((1 - sym) * 27 + 26 - (q->graphs_h[ev->graph].n - sym)) * (q->max_p + 1) + (q->max_p - ev->p);
}

static void sort_recs(orkan_qaoa_t *q, int nevals) {
    const int nkeys = 2 * 27 * (q->max_p + 1);
    memset(q->start_h, 0, ((size_t)nkeys + 1) * sizeof(int));
    for (int e = 0; e < nevals; ++e) ++q->start_h[rec_key(q, &q->evals_h[e]) + 1];
    for (int k = 0; k < nkeys; ++k) q->start_h[k + 1] += q->start_h[k];
    for (int e = 0; e < nevals; ++e) {
        const q_eval_t *ev = &q->evals_h[e];
        const int n = q->graphs_h[ev->graph].n, sym = is_sym(q, ev->graph);
        const int at = q->start_h[rec_key(q, ev)]++;
        const q_rec_t r = {q->graphs_h[ev->graph].diag_off, 0, ev->angle_off, ev->p, n, n - sym, e, 0};
        q->recs_h[at] = r;
        q->n_h[at] = n - sym;
        q->p_h[at] = ev->p;
        q->sym_h[at] = (unsigned char)sym;
    }
}

/* the number of records from `at` on that are of one form and whose states fit the scratch together */
static int next_round(const orkan_qaoa_t *q, int at) {
    size_t used = 0;
    int i = at;
    for (; i < q->nstaged && q->sym_h[i] == q->sym_h[at]; ++i) {
        const size_t tiles = q->n_h[i] > REG_LT ? (size_t)1 << (q->n_h[i] - REG_LT) : 0;
        if (used + tiles > q->room || used + tiles > ((size_t)1 << 31) - 1) break;
        used += tiles;
    }
    return i - at;
}

static int list_ok(const orkan_qaoa_t *q, int nevals, const int *graph, const int *p) {
    if (nevals < 0 || nevals > q->max_evals) return 0;
    for (int e = 0; e < nevals; ++e)
        if (graph[e] < 0 || graph[e] >= q->ngraphs || p[e] < 1 || p[e] > q->max_p) return 0;
    return 1;
}

/* stage the evaluation list; angles: rows of max_p gammas and betas.  any_shape: for every kernel, not only the one the
 * configuration and the list's phases call for */
static int stage(orkan_qaoa_t *q, int nevals, const int *graph, const int *p, const double *gamma, const double *beta,
                 int any_shape) {
    if (!list_ok(q, nevals, graph, p)) return (int)hipErrorInvalidValue;   /* before anything changes */
    q->wide = q->deep = 0;
    for (int e = 0; e < nevals; ++e) {
        q->evals_h[e].graph = graph[e];
        q->evals_h[e].p = p[e];
        q->evals_h[e].angle_off = e * q->max_p;
        const double *g = gamma + (size_t)e * q->max_p, *b = beta + (size_t)e * q->max_p;
        memcpy(q->gb_h + (size_t)e * q->max_p, g, (size_t)p[e] * sizeof(double));
        memcpy(q->gb_h + ((size_t)nevals + e) * q->max_p, b, (size_t)p[e] * sizeof(double));
        for (int l = 0; l < p[e]; ++l)
            if (!(fabs(g[l]) * q->info_h[2 * graph[e]] < REG_PHASE_MAX)) q->wide = 1;
        q->deep |= q->graphs_h[graph[e]].n >= (DEEP + p[e] - 1) / p[e];
        q->order_h[e] = e;
    }
    q->nstaged = nevals;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    int e = ensure_states(q, 0);
    if (e) return e;
    int nrecs = 0;
    if (nevals > 0 && (any_shape || q->deep || (is_reg(q) && !q->wide))) {
        sort_recs(q, nevals);
        /* every round numbers its tiles from 0 */
        q->room = tile_room(q);
        for (int at = 0, m; at < nevals && (m = next_round(q, at)) > 0; at += m) {
            uint64_t tile = 0;
            for (int i = at; i < at + m; ++i) {
                q->recs_h[i].tile = tile;
                if (q->n_h[i] > REG_LT) tile += (uint64_t)1 << (q->n_h[i] - REG_LT);
            }
        }
        nrecs = nevals;
    }
    if (nevals > 0) {
        e = ork_qaoa_stage(st, q->gb_h, (uint64_t)nevals * q->max_p, q->angles_d, q->recs_h, nrecs, q->recs_d);
        if (!e && q->deep) e = ork_qaoa_rescale(st, q->recs_d, nrecs, q->angles_d);
        if (e) return e;
    }
    if (any_shape || !is_reg(q) || q->wide) {
        g_sort_q = q;
        qsort(q->order_h, (size_t)nevals, sizeof(int), by_cost_desc);
        if (nevals > 0) {
            e |= (int)hipMemcpyAsync(q->evals_d, q->evals_h, (size_t)nevals * sizeof(q_eval_t), hipMemcpyHostToDevice, st);
            e |= (int)hipMemcpyAsync(q->order_d, q->order_h, (size_t)nevals * sizeof(int), hipMemcpyHostToDevice, st);
        }
        q->nevals_h = nevals;
        e |= (int)hipMemcpyAsync(q->nevals_d, &q->nevals_h, sizeof(int), hipMemcpyHostToDevice, st);
        e |= (int)hipStreamSynchronize(st);
    }
    return e;
}

/* caller holds ork_lock */
int orkan_qaoa_launch_staged(orkan_qaoa_t *q) {
    if (is_reg(q)) {
        void *st = ork_dev()->stream;
        if (q->wide) {
            const size_t slots = q->nmax > REG_LT ? q->states_bytes / ((size_t)16 << q->nmax) : (size_t)cus();
            const int grid = slots < (size_t)cus() ? (int)slots : cus();
            return ork_qaoa_launch(st, REG_LT, WIDE_THREADS, grid, q->evals_d, q->order_d, q->nevals_d, q->graphs_d,
                                   q->angles_d, q->diag_d, q->states_d, ((uint64_t)1 << q->nmax), q->out_h, q->counter_d);
        }
        /* a configuration set since then may have left less scratch than the records' tiles were numbered for */
        if (q->room > tile_room(q)) return (int)hipErrorOutOfMemory;
        for (int at = 0; at < q->nstaged;) {
            const int m = next_round(q, at);
            if (m == 0) return (int)hipErrorInvalidValue;
            const int e = ork_qaoa_sweeps(st, q->sym_h[at], q->deep, (const q_rec_t *)q->recs_d + at, q->n_h + at, q->p_h + at, m, q->angles_d,
                                          q->diag_d, q->states_d, (double *)((char *)q->states_d + q->room * TILE_BYTES),
                                          q->out_h);
            if (e) return e;
            at += m;
        }
        return 0;
    }
    if (!q->graph_ok) {
        int e = capture(q);
        if (e) return e;
    }
    return (int)hipGraphLaunch(q->exec, (hipStream_t)ork_dev()->stream);
}

int orkan_qaoa_eval(orkan_qaoa_t *q, int nevals, const int *graph, const int *p, const double *gamma,
                    const double *beta, double *out) {
    if (!q) return (int)hipErrorInvalidValue;
    ork_lock();
    int e = stage(q, nevals, graph, p, gamma, beta, 0);
    if (!e) e = orkan_qaoa_launch_staged(q);
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    /* also after an error: the next call writes the pinned list again */
    const int es = (int)hipStreamSynchronize(st);
    if (!e) e = es;
    if (!e && nevals > 0 && out) memcpy(out, q->out_h, (size_t)nevals * sizeof(double));
    ork_unlock();
    return e;
}

int orkan_qaoa_get_config(const orkan_qaoa_t *q, int *lt, int *threads, int *grid) {
    if (!q) return (int)hipErrorInvalidValue;
    if (lt) *lt = q->lt;
    if (threads) *threads = q->threads;
    if (grid) *grid = q->grid;
    return 0;
}

/* the configuration as it was before a search that found none */
static void back_to(orkan_qaoa_t *q, int lt, int threads, int grid) {
    drop_graph(q);
    q->lt = lt;
    q->threads = threads;
    q->grid = grid;
    (void)ensure_states(q, 1);
}

/* Autotuner: time every (tile, workgroup size) candidate the largest state
 * allows on the caller's evaluation list (one untimed launch, then the median
 * of `reps` launches), keep the fastest. */
int orkan_qaoa_autotune(orkan_qaoa_t *q, int nevals, const int *graph, const int *p, const double *gamma,
                        const double *beta, int reps, double *best_ms) {
    static const int cand[][2] = {{11, 256}, {11, 512}, {12, 256}, {12, 512}, {12, 1024}, {13, 512}, {13, 1024}};
    if (!q || !list_ok(q, nevals, graph, p)) return (int)hipErrorInvalidValue;
    if (reps < 1) reps = 1;
    if (reps > 15) reps = 15;
    hipStream_t st = (hipStream_t)ork_dev()->stream;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess) return (int)hipErrorOutOfMemory;
    if (hipEventCreate(&b) != hipSuccess) {
        (void)hipEventDestroy(a);
        return (int)hipErrorOutOfMemory;
    }
    /* the whole search holds the library lock: staging, every reconfiguration and launch */
    ork_lock();
    const int lt0 = q->lt, threads0 = q->threads, grid0 = q->grid;
    /* the register kernels' records number tiles of the scratch: it has its size for them first */
    if (2 * REG_LT >= q->nmax) (void)set_config(q, REG_LT, REG_THREADS, 0, 0);
    int e = stage(q, nevals, graph, p, gamma, beta, 1);
    if (e) {
        back_to(q, lt0, threads0, grid0);
        ork_unlock();
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
        return e;
    }
    double best = 1e30;
    int best_i = -1;
    for (size_t i = 0; i < sizeof(cand) / sizeof(cand[0]); ++i) {
        if (set_config(q, cand[i][0], cand[i][1], 0, 0)) continue;
        if (orkan_qaoa_launch_staged(q)) continue;
        float t[15];
        int ok = 1;
        for (int r = 0; r < reps && ok; ++r) {
            ok &= hipEventRecord(a, st) == hipSuccess;
            ok &= orkan_qaoa_launch_staged(q) == 0;
            ok &= hipEventRecord(b, st) == hipSuccess;
            ok &= hipEventSynchronize(b) == hipSuccess;
            ok &= hipEventElapsedTime(&t[r], a, b) == hipSuccess;
        }
        if (!ok) continue;
        for (int x = 0; x < reps; ++x)
            for (int y = x + 1; y < reps; ++y)
                if (t[y] < t[x]) { float tmp = t[x]; t[x] = t[y]; t[y] = tmp; }
        const double med = t[reps / 2];
        if (med < best) {
            best = med;
            best_i = (int)i;
        }
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    if (best_i < 0) {
        back_to(q, lt0, threads0, grid0);
        ork_unlock();
        return (int)hipErrorInvalidConfiguration;
    }
    if (best_ms) *best_ms = best;
    e = set_config(q, cand[best_i][0], cand[best_i][1], 0, 1);
    ork_unlock();
    return e;
}

int orkan_maxcut_diag_dev(int n, int nedges, const int *ei, const int *ej, const double *w, double *out_dev) {
    ork_dev_t *d = ork_dev();
    hipStream_t st = (hipStream_t)d->stream;
    int *ed = ork_mem_get((size_t)(2 * nedges + 1) * sizeof(int));
    double *wd = ork_mem_get((size_t)(nedges + 1) * sizeof(double));
    int e = ed && wd ? 0 : (int)hipErrorOutOfMemory;
    if (!e && nedges > 0) {
        e |= (int)hipMemcpyAsync(ed, ei, (size_t)nedges * sizeof(int), hipMemcpyHostToDevice, st);
        e |= (int)hipMemcpyAsync(ed + nedges, ej, (size_t)nedges * sizeof(int), hipMemcpyHostToDevice, st);
        e |= (int)hipMemcpyAsync(wd, w, (size_t)nedges * sizeof(double), hipMemcpyHostToDevice, st);
    }
    if (!e) e = ork_maxcut_diag(st, out_dev, n, nedges, ed, ed + nedges, wd);
    if (!e) e = (int)hipStreamSynchronize(st);
    ork_mem_put(ed);
    ork_mem_put(wd);
    return e;
}
