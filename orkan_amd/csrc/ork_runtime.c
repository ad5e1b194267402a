/*
 * ork_runtime.c -- per-device runtime of the library: one HIP stream per
 * device (default priority), the reduction partials, and the staging buffers
 * that bring caller-owned host arrays (observables, diagonals) into HBM.
 */
#include "ork_host.h"

#include <pthread.h>
#include <string.h>
#include <hip/hip_runtime_api.h>

#define ORK_MAX_DEV 64

static ork_dev_t g_dev[ORK_MAX_DEV];
static int g_ready[ORK_MAX_DEV];
static pthread_mutex_t g_mu = PTHREAD_MUTEX_INITIALIZER;        /* ork_lock: shared staging, partials */
static pthread_mutex_t g_host_mu = PTHREAD_MUTEX_INITIALIZER;   /* held by whoever has the pinned buffer */
static pthread_mutex_t g_init_mu = PTHREAD_MUTEX_INITIALIZER;   /* per-device runtime creation, so that
                                                                 * ork_dev() may be called under ork_lock */

void ork_hip_fail(const char *where, int err) {
    fprintf(stderr, "orkan: hip: %s: %s\n", where, hipGetErrorString((hipError_t)err));
    exit(EXIT_FAILURE);
}

void ork_lock(void) { pthread_mutex_lock(&g_mu); }
void ork_unlock(void) { pthread_mutex_unlock(&g_mu); }

ork_dev_t *ork_dev(void) {
    int dev = 0;
    ORK_HIP("hipGetDevice", hipGetDevice(&dev));
    if (dev < 0 || dev >= ORK_MAX_DEV) ork_hip_fail("device index", (int)hipErrorInvalidDevice);
    if (!__atomic_load_n(&g_ready[dev], __ATOMIC_ACQUIRE)) {
        pthread_mutex_lock(&g_init_mu);
        if (!__atomic_load_n(&g_ready[dev], __ATOMIC_ACQUIRE)) {
            ork_dev_t *d = &g_dev[dev];
            memset(d, 0, sizeof(*d));
            hipStream_t st;
            ORK_HIP("hipStreamCreateWithFlags", hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
            d->stream = (void *)st;
            ORK_HIP("hipHostMalloc(partials)", hipHostMalloc((void **)&d->partials, ork_partials_len() * sizeof(double),
                                                             hipHostMallocDefault));
            /* device address of the allocation-free exp_diag's scratch array on this device; a failure
             * leaves it unset, and only orkan_exp_diag_noalloc reports it */
            d->noalloc_err = ork_noalloc_setup();
            __atomic_store_n(&g_ready[dev], 1, __ATOMIC_RELEASE);
        }
        pthread_mutex_unlock(&g_init_mu);
    }
    return &g_dev[dev];
}

ork_dev_t *ork_dev_existing(void) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= ORK_MAX_DEV) return NULL;
    return __atomic_load_n(&g_ready[dev], __ATOMIC_ACQUIRE) ? &g_dev[dev] : NULL;
}

int ork_is_dev_ptr(const void *p) {
    hipPointerAttribute_t at;
    memset(&at, 0, sizeof(at));
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return at.type == hipMemoryTypeDevice;
}

int ork_is_pageable(const void *p) {
    hipPointerAttribute_t at;
    memset(&at, 0, sizeof(at));
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return at.type == hipMemoryTypeUnregistered;
}

const double *ork_dev_doubles(const double *src, size_t count) {
    if (ork_is_dev_ptr(src)) return src;
    ork_dev_t *d = ork_dev();
    const size_t bytes = count * sizeof(double);
    if (d->stage_bytes < bytes) {
        if (d->stage) {
            ORK_HIP("hipStreamSynchronize", hipStreamSynchronize((hipStream_t)d->stream));
            ORK_HIP("hipFree(stage)", hipFree(d->stage));
        }
        d->stage = NULL;
        d->stage_bytes = 0;
        ORK_HIP("hipMalloc(stage)", ork_dev_malloc(&d->stage, bytes));
        d->stage_bytes = bytes;
    }
    ORK_HIP("hipMemcpyAsync(stage)", hipMemcpyAsync(d->stage, src, bytes, hipMemcpyHostToDevice, (hipStream_t)d->stream));
    /* the caller may reuse its array as soon as the API call returns */
    ORK_HIP("hipStreamSynchronize", hipStreamSynchronize((hipStream_t)d->stream));
    return (const double *)d->stage;
}

/* ------------------------------------------------------------------------------------------------
 * device memory of states and scratch
 *
 * hipMalloc and hipFree map and unmap pages: a state_cp, relayout and precision conversion of a 12-qubit density
 * matrix (134 MB each) spent 9.2 of their 9.6 ms there, a sample_matrix call on 18 qubits about 1 of 4 ms.  Blocks given
 * back are therefore kept, per device, for the next request of nearly the same size.  At most ORK_MEM_KEEP bytes and
 * ORK_MEM_BLOCKS blocks are kept (the oldest go back to the device first, larger ones at once), and all of them go back when an allocation
 * of the library finds the device full (ork_mem_get, ork_dev_malloc) or a caller asks (orkan_mem_trim).  A block is only handed out for use on the library stream, after everything that used it.
 * ---------------------------------------------------------------------------------------------- */
#define ORK_MEM_KEEP ((size_t)8 << 30)
#define ORK_MEM_BLOCKS 4096
#define ORK_MEM_BUCKETS 1024
/* size classes, eight per power of two: a request looks at the blocks of its own and the next one or two only */
#define ORK_MEM_CLASSES (64 * 8)

typedef struct mem_block {
    void *p;
    size_t bytes;
    int dev;
    int kept;                          /* given back, in its device's list */
    struct mem_block *chain;           /* next block of the same bucket */
    struct mem_block *older, *newer;   /* kept blocks of a device, by the time they came back */
    struct mem_block *prev, *next;     /* ... of one size class */
} mem_block_t;

static pthread_mutex_t g_mem_mu = PTHREAD_MUTEX_INITIALIZER;
static mem_block_t *g_mem_table[ORK_MEM_BUCKETS];
static mem_block_t *g_mem_oldest[ORK_MAX_DEV], *g_mem_newest[ORK_MAX_DEV];
static mem_block_t *g_mem_class[ORK_MAX_DEV][ORK_MEM_CLASSES];
static size_t g_mem_kept[ORK_MAX_DEV];
static int g_mem_blocks[ORK_MAX_DEV];

/* what an allocation of `bytes` takes from the device (hipMemGetInfo): pages of 4 KB, from 2 MB on pages of 2 MB */
static size_t mem_round(size_t bytes) {
    const size_t page = (size_t)(bytes >= 2 << 20 ? 2 << 20 : 4 << 10);
    return bytes == 0 ? page : bytes > SIZE_MAX - page ? bytes : (bytes + page - 1) / page * page;
}

static int mem_class(size_t bytes) {   /* bytes >= 4096 */
    const int b = 63 - __builtin_clzll(bytes);
    return b * 8 + (int)(bytes >> (b - 3) & 7);
}

static mem_block_t **mem_slot(const void *p) {
    mem_block_t **s = &g_mem_table[((uintptr_t)p >> 12) % ORK_MEM_BUCKETS];
    while (*s && (*s)->p != p) s = &(*s)->chain;
    return s;
}

static void mem_unkeep(mem_block_t *b) {
    *(b->older ? &b->older->newer : &g_mem_oldest[b->dev]) = b->newer;
    *(b->newer ? &b->newer->older : &g_mem_newest[b->dev]) = b->older;
    *(b->prev ? &b->prev->next : &g_mem_class[b->dev][mem_class(b->bytes)]) = b->next;
    if (b->next) b->next->prev = b->prev;
    g_mem_kept[b->dev] -= b->bytes;
    g_mem_blocks[b->dev] -= 1;
    b->kept = 0;
}

static void mem_forget(const void *p) {
    mem_block_t **s = mem_slot(p), *b = *s;
    if (!b) return;
    if (b->kept) mem_unkeep(b);
    *s = b->chain;
    free(b);
}

/* kept blocks of the device back to it, the oldest first, until at most `keep` bytes are left */
static void mem_trim(int dev, size_t keep) {
    while (g_mem_kept[dev] > keep || g_mem_blocks[dev] > ORK_MEM_BLOCKS) {
        void *p = g_mem_oldest[dev]->p;
        mem_forget(p);
        (void)hipFree(p);
    }
}

/* hipMalloc, a second time with the kept blocks given back */
static int malloc_or_trim(int dev, void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess && g_mem_kept[dev] > 0) {
        (void)hipGetLastError();
        mem_trim(dev, 0);
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = NULL;
    }
    return (int)e;
}

int ork_dev_malloc(void **p, size_t bytes) {
    int dev = 0;
    *p = NULL;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= ORK_MAX_DEV) return (int)hipErrorInvalidDevice;
    pthread_mutex_lock(&g_mem_mu);
    const int r = malloc_or_trim(dev, p, bytes);
    if (!r) mem_forget(*p);   /* an entry of this address is of a block that was freed elsewhere */
    pthread_mutex_unlock(&g_mem_mu);
    return r;
}

size_t orkan_mem_trim(size_t keep_bytes) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= ORK_MAX_DEV) return 0;
    pthread_mutex_lock(&g_mem_mu);
    mem_trim(dev, keep_bytes);
    const size_t kept = g_mem_kept[dev];
    pthread_mutex_unlock(&g_mem_mu);
    return kept;
}

void *ork_mem_get(size_t bytes) {
    int dev = 0;
    void *p = NULL;
    ork_dev();
    if (hipGetDevice(&dev) != hipSuccess) return NULL;
    bytes = mem_round(bytes);
    pthread_mutex_lock(&g_mem_mu);
    /* the smallest kept block that holds the request and is at most an eighth larger */
    mem_block_t *best = NULL;
    const size_t most = bytes > SIZE_MAX - bytes / 8 ? bytes : bytes + bytes / 8;
    for (int c = mem_class(bytes); c <= mem_class(most) && !best; ++c)
        for (mem_block_t *b = g_mem_class[dev][c]; b && !(best && best->bytes == bytes); b = b->next)
            if (b->bytes >= bytes && b->bytes <= most && (!best || b->bytes < best->bytes)) best = b;
    if (best) {
        mem_unkeep(best);
        p = best->p;
    } else {
        if (malloc_or_trim(dev, &p, bytes) == 0) {
            mem_forget(p);   /* an entry of this address is of a block that was freed elsewhere */
            mem_block_t *b = calloc(1, sizeof(*b));
            if (b) {
                b->p = p;
                b->bytes = bytes;
                b->dev = dev;
                *mem_slot(p) = b;
            }
        }
    }
    pthread_mutex_unlock(&g_mem_mu);
    return p;
}

/* the block of p, if p is one that is out and still the allocation this table knows (a caller may have freed it with
 * hipFree and have been given the address again) */
static mem_block_t *mem_live(void *p) {
    mem_block_t *b = *mem_slot(p);
    if (!b || b->kept) return NULL;
    hipDeviceptr_t base = NULL;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();
        base = NULL;
    }
    if (base == (hipDeviceptr_t)p && size >= b->bytes && size - b->bytes < 4096) return b;
    mem_forget(p);
    return NULL;
}

void ork_mem_put(void *p) {
    if (!p) return;
    pthread_mutex_lock(&g_mem_mu);
    mem_block_t *b = mem_live(p);
    if (b && b->bytes <= ORK_MEM_KEEP) {
        b->kept = 1;
        b->newer = NULL;
        b->older = g_mem_newest[b->dev];
        *(b->older ? &b->older->newer : &g_mem_oldest[b->dev]) = b;
        g_mem_newest[b->dev] = b;
        mem_block_t **first = &g_mem_class[b->dev][mem_class(b->bytes)];
        b->prev = NULL;
        b->next = *first;
        if (*first) (*first)->prev = b;
        *first = b;
        g_mem_kept[b->dev] += b->bytes;
        g_mem_blocks[b->dev] += 1;
        mem_trim(b->dev, ORK_MEM_KEEP);
    } else {
        mem_forget(p);
        (void)hipFree(p);
    }
    pthread_mutex_unlock(&g_mem_mu);
}

void ork_mem_release(void *p) {
    if (!p) return;
    ork_dev();
    int cur = 0, dev = -1;
    (void)hipGetDevice(&cur);
    pthread_mutex_lock(&g_mem_mu);
    const mem_block_t *b = *mem_slot(p);
    if (b) dev = b->dev;
    pthread_mutex_unlock(&g_mem_mu);
    /* work of the caller's own streams may still use the memory, on the device it belongs to */
    if (dev >= 0 && dev != cur) (void)hipSetDevice(dev);
    (void)hipDeviceSynchronize();
    if (dev >= 0 && dev != cur) (void)hipSetDevice(cur);
    ork_mem_put(p);
}

void ork_host_prepare(void) {
    ork_dev_t *d = ork_dev();
    pthread_mutex_lock(&g_host_mu);
    if (!d->host) {
        void *p = NULL;
        if (hipHostMalloc(&p, ORK_HOST_FLOATS * sizeof(float), hipHostMallocDefault) == hipSuccess)
            d->host = memset(p, 0, ORK_HOST_FLOATS * sizeof(float));
        else
            (void)hipGetLastError();
    }
    pthread_mutex_unlock(&g_host_mu);
}

float *ork_host_take(void) {
    float *p = NULL;
    if (pthread_mutex_trylock(&g_host_mu) != 0) return NULL;
    if (!(p = ork_dev()->host)) pthread_mutex_unlock(&g_host_mu);
    return p;
}

void ork_host_give(void) { pthread_mutex_unlock(&g_host_mu); }

/* ------------------------------------------------------------------------------------------------
 * extension API: stream access, device arrays, timing
 * ---------------------------------------------------------------------------------------------- */

void *orkan_stream(void) { return ork_dev()->stream; }

int orkan_sync(void) { return (int)hipStreamSynchronize((hipStream_t)ork_dev()->stream); }

double *orkan_dev_alloc(idx_t count) {
    void *p = NULL;
    return ork_dev_malloc(&p, (size_t)count * sizeof(double)) == 0 ? (double *)p : NULL;
}

int orkan_dev_upload(double *dst_dev, const double *src_host, idx_t count) {
    ork_dev_t *d = ork_dev();
    int e = (int)hipMemcpyAsync(dst_dev, src_host, (size_t)count * sizeof(double), hipMemcpyHostToDevice,
                                (hipStream_t)d->stream);
    if (e) return e;
    return (int)hipStreamSynchronize((hipStream_t)d->stream);
}

int orkan_set_launch_shape(int kernel, int flags, int lds_bytes) {
    if (kernel == 10) return ork_sv_set_red_lds(flags, lds_bytes);
    if (kernel == 11) return ork_mlp_gemm_select(flags);
    if (kernel == 12) return ork_sv_set_pair_shape(flags, lds_bytes);
    if (kernel == 13) return ork_sv_set_nt_off(flags, lds_bytes);
    if (kernel == 17) return ork_sv_set_layer_variant(flags);
    if (kernel == 19) return ork_sv_set_exp_shape(flags, lds_bytes);
    if (kernel == 20) return ork_sv_set_mono_lds32(lds_bytes);
    if (kernel == 21) return ork_sv_set_perm_shape(flags, lds_bytes);
    if (kernel == 14) {
        ork_dm_reset_shapes();
        ork_sv_reset_tuning();
        ork_mlp_gemm_reset();
        return 0;
    }
    return ork_dm_set_shape(kernel, flags, lds_bytes);
}

int orkan_copy_to_host(void *dst_host, const void *src_dev, size_t bytes) {
    ork_dev_t *d = ork_dev();
    int e = (int)hipMemcpyAsync(dst_host, src_dev, bytes, hipMemcpyDeviceToHost, (hipStream_t)d->stream);
    if (e) return e;
    return (int)hipStreamSynchronize((hipStream_t)d->stream);
}

int orkan_copy_to_device(void *dst_dev, const void *src_host, size_t bytes) {
    ork_dev_t *d = ork_dev();
    int e = (int)hipMemcpyAsync(dst_dev, src_host, bytes, hipMemcpyHostToDevice, (hipStream_t)d->stream);
    if (e) return e;
    return (int)hipStreamSynchronize((hipStream_t)d->stream);
}

void orkan_dev_free(void *p) {
    ork_mem_release(p);
}

#define ORK_MAX_EVENTS 65536
static hipEvent_t *g_ev[ORK_MAX_DEV];

int orkan_event_record(int slot) {
    int dev = 0;
    if (slot < 0 || slot >= ORK_MAX_EVENTS) return (int)hipErrorInvalidValue;
    ork_dev_t *d = ork_dev();
    ORK_HIP("hipGetDevice", hipGetDevice(&dev));
    if (!g_ev[dev]) {
        g_ev[dev] = calloc(ORK_MAX_EVENTS, sizeof(hipEvent_t));
        if (!g_ev[dev]) return (int)hipErrorOutOfMemory;
    }
    if (!g_ev[dev][slot]) {
        int e = (int)hipEventCreate(&g_ev[dev][slot]);
        if (e) return e;
    }
    return (int)hipEventRecord(g_ev[dev][slot], (hipStream_t)d->stream);
}

double orkan_event_ms(int a, int b) {
    int dev = 0;
    float ms = -1.0f;
    if (a < 0 || b < 0 || a >= ORK_MAX_EVENTS || b >= ORK_MAX_EVENTS) return -1.0;
    ORK_HIP("hipGetDevice", hipGetDevice(&dev));
    if (!g_ev[dev] || !g_ev[dev][a] || !g_ev[dev][b]) return -1.0;
    if (hipEventSynchronize(g_ev[dev][b]) != hipSuccess) return -1.0;
    if (hipEventElapsedTime(&ms, g_ev[dev][a], g_ev[dev][b]) != hipSuccess) return -1.0;
    return (double)ms;
}
