/*
 * Drives the library's device-memory bookkeeping on a small device that exists only here: the HIP calls below hand out
 * host memory against a capacity, in pages, and know what is live.  tests/test_host_memory.py links it with the C17 host
 * layer and empty kernels and runs one case per process.
 */
#include "ork_host.h"
#include "orkan.h"
#include "orkan_amd.h"

#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <hip/hip_runtime_api.h>

#define MB ((size_t)1 << 20)
#define PAGE ((size_t)4096)

static struct { char *p; size_t bytes; } live[65536];
static int nlive, nmallocs;
static size_t used, capacity = 64 * MB;

static size_t pages(size_t n) { return (n + PAGE - 1) / PAGE * PAGE; }

hipError_t hipMalloc(void **p, size_t n) {
    *p = NULL;
    ++nmallocs;
    if (used + pages(n) > capacity || nlive == 65536) return hipErrorOutOfMemory;
    *p = aligned_alloc(PAGE, pages(n));
    live[nlive].p = *p;
    live[nlive++].bytes = n;
    used += pages(n);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    for (int i = 0; i < nlive; ++i)
        if (live[i].p == p) {
            used -= pages(live[i].bytes);
            live[i] = live[--nlive];
            free(p);
            return hipSuccess;
        }
    return p ? hipErrorInvalidValue : hipSuccess;
}
static int is_live(const void *p) {
    for (int i = 0; i < nlive; ++i)
        if (live[i].p == p) return 1;
    return 0;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t p) {
    for (int i = 0; i < nlive; ++i)
        if ((char *)p >= live[i].p && (char *)p < live[i].p + live[i].bytes) {
            *base = live[i].p;
            *size = live[i].bytes;
            return hipSuccess;
        }
    return hipErrorInvalidValue;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    hipDeviceptr_t b;
    size_t n;
    memset(a, 0, sizeof *a);
    a->type = hipMemGetAddressRange(&b, &n, (hipDeviceptr_t)p) == hipSuccess ? hipMemoryTypeDevice
                                                                             : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return (*p = calloc(1, n ? n : 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { (void)k; (void)st; memmove(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) { (void)st; memset(d, v, n); return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = 64; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
int ork_qaoa_occupancy(int lt, int threads, int *blocks) { (void)lt; (void)threads; *blocks = 2; return 0; }

hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 1.0f; return hipSuccess; }
/* no cost is the same for x and ~x */
int ork_qaoa_diag_info(void *st, int ng, int nmax, const void *g, const double *d, uint64_t *info) {
    for (int i = 0; i < ng; ++i) info[2 * i + 1] = 1;
    return 0;
}
static int rounds;   /* rounds of register-kernel launches */
int ork_qaoa_sweeps() { ++rounds; return 0; }

typedef struct orkan_mlp orkan_mlp_t;
orkan_mlp_t *orkan_mlp_create(int in_dim, int hidden, int nhidden, int max_batch);

#define CHECK(c)                                                                       \
    do {                                                                               \
        if (!(c)) {                                                                    \
            fprintf(stderr, "host_memory: check failed: %s (line %d)\n", #c, __LINE__); \
            exit(2);                                                                   \
        }                                                                              \
    } while (0)

/* n qubits of 2^n x 16 B: 21 qubits are 32 MB */
static state_t pure(qubit_t n) {
    state_t s = {PURE, NULL, 0};
    state_init(&s, n, NULL);
    CHECK(s.data);
    return s;
}

/* leaves 32 MB of the 64 kept beside a live state of 1 MB */
static state_t fill(void) {
    state_t s = pure(16), big = pure(21);
    state_free(&big);
    CHECK(used >= 33 * MB);
    return s;
}

int main(int argc, char **argv) {
    const char *what = argc > 1 ? argv[1] : "";
    state_t s = fill();
    if (!strcmp(what, "dev_alloc")) {
        CHECK(orkan_dev_alloc(40 * MB / 8));
    } else if (!strcmp(what, "staging")) {
        double *host = calloc(40 * MB, 1);
        CHECK(ork_dev_doubles(host, 40 * MB / 8));
    } else if (!strcmp(what, "phases")) {
        /* a packed state of 8 qubits, then phase scratch of 16 B per index on a device with a page left for it */
        state_t m = {MIXED_PACKED, NULL, 0};
        state_init(&m, 8, NULL);
        capacity = used;
        double *diag = calloc(256, 8);
        CHECK(ork_dev_doubles(diag, 256));
        exp_diag(&m, diag, 0.5);
    } else if (!strcmp(what, "mlp")) {
        CHECK(orkan_mlp_create(128, 128, 3, 8192));
    } else if (!strcmp(what, "mlp_size")) {
        /* three layers of 128, 8192 rows: per row and column 12 B of pre-activations, 6 of activations, 6 of transposed
         * inputs, 2 of gradients and 6 of their transposes; 6 B per input; the parameters */
        orkan_mem_trim(0);
        const size_t before = used, mh = (size_t)8192 * 128;
        CHECK(orkan_mlp_create(128, 128, 3, 8192));
        CHECK(used - before <= 32 * mh + 6 * mh + 2 * MB);
    } else if (!strcmp(what, "qaoa")) {
        /* one 20-qubit graph: 8 MB of diagonal, 16 MB of state, and the whole scratch, not half of it */
        const unsigned char nq = 20;
        double *diag = calloc(8, 1 << 20);
        const double *d = diag;
        capacity = used + 4 * MB;
        orkan_qaoa_t *q = orkan_qaoa_create(1, &nq, &d, 1, 2);
        CHECK(q);
        CHECK(used >= 1 * MB + 8 * MB + 16 * MB);
    } else if (!strcmp(what, "qaoa_scratch")) {
        /* 64 evaluations of 20 qubits: 128 MB of scratch, 8 states in a round.  The LDS shapes' GB, in the autotuner's
         * search or a configuration, neither stay nor change the rounds. */
        capacity = (size_t)8 << 30;
        const unsigned char nq = 20;
        double *diag = calloc(8, 1 << 20), *g = calloc(64 * 2, 8), *b = calloc(64 * 2, 8), out[64];
        const double *d = diag;
        static int graph[64], p[64];
        for (int i = 0; i < 64; ++i) p[i] = 2;
        orkan_qaoa_t *q = orkan_qaoa_create(1, &nq, &d, 64, 2);
        CHECK(q);
        const size_t at_first = used;
        CHECK(orkan_qaoa_eval(q, 64, graph, p, g, b, out) == 0 && rounds == 8);
        CHECK(orkan_qaoa_autotune(q, 64, graph, p, g, b, 1, NULL) == 0);
        CHECK(orkan_qaoa_set_config(q, 12, 512, 0) == 0 && used > at_first + 64 * MB);
        CHECK(orkan_qaoa_set_config(q, 12, 256, 0) == 0 && used == at_first);
        rounds = 0;
        CHECK(orkan_qaoa_eval(q, 64, graph, p, g, b, out) == 0 && rounds == 8);
        /* nor do the slots of a list with a phase that the register kernels leave to an LDS one */
        g[0] = INFINITY;
        CHECK(orkan_qaoa_eval(q, 64, graph, p, g, b, out) == 0 && rounds == 8);
        g[0] = 0.0;
        CHECK(orkan_qaoa_eval(q, 64, graph, p, g, b, out) == 0 && rounds == 16);
        orkan_qaoa_destroy(q);
    } else if (!strcmp(what, "qaoa_refused")) {
        /* a search on a list that is refused leaves the configuration and the scratch as they were */
        capacity = (size_t)8 << 30;
        const unsigned char nq = 14;
        double *diag = calloc(8, 1 << 14), g[2] = {0}, b[2] = {0}, out[1];
        const double *d = diag;
        int graph = 0, p = 3, lt, th, gr;
        orkan_qaoa_t *q = orkan_qaoa_create(1, &nq, &d, 8, 2);
        CHECK(q && orkan_qaoa_set_config(q, 11, 512, 1) == 0);
        const size_t before = used;
        CHECK(orkan_qaoa_autotune(q, 1, &graph, &p, g, b, 1, NULL) != 0);
        CHECK(orkan_qaoa_get_config(q, &lt, &th, &gr) == 0 && lt == 11 && th == 512 && gr == 8 && used == before);
        p = 2;
        graph = 1;
        CHECK(orkan_qaoa_autotune(q, 1, &graph, &p, g, b, 1, NULL) != 0);
        CHECK(orkan_qaoa_autotune(q, 9, &graph, &p, g, b, 1, NULL) != 0);
        CHECK(orkan_qaoa_eval(q, 1, &graph, &p, g, b, out) != 0);
        CHECK(orkan_qaoa_get_config(q, &lt, &th, &gr) == 0 && lt == 11 && th == 512 && gr == 8 && used == before);
        graph = 0;
        CHECK(orkan_qaoa_autotune(q, 1, &graph, &p, g, b, 1, NULL) == 0);
        orkan_qaoa_destroy(q);
    } else if (!strcmp(what, "count")) {
        /* many tiny states: each holds a page, whatever its length, and a bounded number of them is kept */
        static state_t t[6000];
        for (int i = 0; i < 6000; ++i) t[i] = pure((qubit_t)(1 + i % 4));
        for (int i = 0; i < 6000; ++i) state_free(&t[i]);
        CHECK(used <= 1 * MB + 4096 * PAGE);
        CHECK(orkan_mem_trim((size_t)-1) == used - 1 * MB);
        /* the block for the next one is found, not allocated */
        const int before = nmallocs;
        for (int i = 0; i < 100; ++i) t[i] = pure(3);
        CHECK(nmallocs == before);
    } else if (!strcmp(what, "classes")) {
        /* for every size, a block of it or of up to an eighth more is taken, the nearest one first; a larger one is not */
        capacity = 256 * MB;
        for (size_t n = 5000; n < 24 * MB; n += n / 3 + 4096) {
            orkan_mem_trim(0);
            void *exact = ork_mem_get(n), *more = ork_mem_get(n + n / 16 + (n >= 1 * MB ? 2 * MB : 4096));
            ork_mem_put(exact);
            ork_mem_put(more);
            CHECK(ork_mem_get(n) == exact);
            ork_mem_put(exact);
            orkan_mem_trim(0);
            void *twice = ork_mem_get(2 * n + 8192);
            ork_mem_put(twice);
            void *q = ork_mem_get(n);
            CHECK(q && q != twice);
            ork_mem_put(q);
            CHECK(ork_mem_get(2 * n + 8192) == twice);
            ork_mem_put(twice);
        }
    } else if (!strcmp(what, "cap")) {
        /* five states of 4 GB (nothing touches their memory here): at most 8 GB stay, a larger block does not */
        capacity = (size_t)1 << 40;
        orkan_mem_trim(0);
        const size_t base = used;
        state_t big[5];
        for (int i = 0; i < 5; ++i) {
            big[i] = (state_t){PURE, NULL, 0};
            state_plus(&big[i], 28);
            CHECK(big[i].data);
        }
        for (int i = 0; i < 5; ++i) state_free(&big[i]);
        CHECK(used - base == 8192 * MB);
        big[0] = (state_t){PURE, NULL, 0};
        state_plus(&big[0], 30);
        state_free(&big[0]);
        CHECK(used - base <= 8192 * MB);
    } else if (!strcmp(what, "behind")) {
        /* a state's storage freed by its address: releasing the state then frees nothing else, and the address may come
         * back as somebody else's */
        state_t a = pure(12);
        void *p = a.data, *q;
        CHECK(hipFree(p) == hipSuccess);
        state_free(&a);
        CHECK(hipMalloc(&q, 16 << 11) == hipSuccess);
        state_t b = pure(12), c = pure(12);
        CHECK(b.data != c.data && (void *)b.data != q && (void *)c.data != q && is_live(q));
        state_free(&b);
        state_free(&c);
        CHECK(is_live(q));
    } else if (!strcmp(what, "trim")) {
        size_t (*trim)(size_t) = orkan_mem_trim;
        CHECK(trim((size_t)-1) >= 32 * MB);
        CHECK(used >= 33 * MB);
        CHECK(trim(0) == 0);
        CHECK(used < 2 * MB);
    } else {
        return 3;
    }
    CHECK(is_live(s.data));
    printf("host_memory ok %s\n", what);
    return 0;
}
