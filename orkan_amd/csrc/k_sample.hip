// k_sample.hip -- kernels of sample_matrix: copies of the prefix, the weighted sums of a linear combination of operations,
// and the block product G = P^dagger diag(obs) Q of up to 64 x 64 leaf vectors (no reference code: the operation is
// specified in docs/SAMPLE_MATRIX.md).
#include "k_common.hpp"

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int SM_THREADS = 256;
constexpr int SM_MAX = 64;          // vectors per side
constexpr int SM_STEP = 16;         // amplitudes per step of the product
constexpr int SM_PARTS = 1024;     // x-ranges of the product at most: four workgroups per CU (512 take 144 us, 2048 132)

// dst[v] = src for v < cnt (vectors of n, `stride` apart): one read of src per 8 copies
__global__ __launch_bounds__(SM_THREADS) void spread_kernel(double2 *__restrict__ dst, const double2 *__restrict__ src,
                                                            u64 n, u64 stride, int cnt) {
    const int v0 = blockIdx.y * 8, v1 = v0 + 8 < cnt ? v0 + 8 : cnt;
    for (u64 i = (u64)blockIdx.x * SM_THREADS + threadIdx.x; i < n; i += (u64)gridDim.x * SM_THREADS) {
        const cd x = src[i];
        for (int v = v0; v < v1; ++v) dst[(u64)v * stride + i] = x;
    }
}

__device__ __forceinline__ cd wmul(double wr, double wi, cd x) {
    // the products of x.y rounded, those of x.x fused: as the compiler contracts wr x.x - wi x.y and wr x.y + wi x.x
    return cmk(fma(wr, x.x, -(wi * x.y)), fma(wi, x.x, wr * x.y));
}

// one term of a linear combination over cnt whole vectors: acc = [acc +] w v
__global__ __launch_bounds__(SM_THREADS) void axpy_kernel(double2 *__restrict__ acc, const double2 *__restrict__ v,
                                                          double wr, double wi, u64 n, int first) {
    for (u64 i = (u64)blockIdx.x * SM_THREADS + threadIdx.x; i < n; i += (u64)gridDim.x * SM_THREADS) {
        const cd t = wmul(wr, wi, v[i]);
        acc[i] = first ? t : cadd(acc[i], t);
    }
}

// the last term, in place: x = [a +] w x, or with `scaled` x = wa a + w x (a combination of two operations in one pass)
__global__ __launch_bounds__(SM_THREADS) void combine_kernel(double2 *__restrict__ x, const double2 *__restrict__ a,
                                                             double war, double wai, int scaled, double wr, double wi,
                                                             u64 n) {
    for (u64 i = (u64)blockIdx.x * SM_THREADS + threadIdx.x; i < n; i += (u64)gridDim.x * SM_THREADS) {
        const cd t = wmul(wr, wi, x[i]);
        if (!a) x[i] = t;
        else x[i] = cadd(scaled ? wmul(war, wai, a[i]) : a[i], t);
    }
}

// ---- block product ---------------------------------------------------------------------------------
// G[a][b] = sum_x conj(P[a][x]) obs[x] Q[b][x] on v_mfma_f64_16x16x4_f64 (A: row lane % 16, k lane / 16; B: column lane %
// 16, k lane / 16; D: column lane % 16, row 4 r + lane / 16).  A workgroup owns an x-range; per step of 16 amplitudes it
// loads 256 B of every vector into LDS (the next step's loads are in flight meanwhile), and each of its waves takes 16
// vectors a against all vectors b: per 16 x 16 tile four products (re re, im im, re im, im re).  Which wave takes which
// 16 turns with the workgroup, so that the unequal shares of a block with itself (only tiles on and below the diagonal
// are formed) and the idle waves of fewer than 49 vectors spread over a CU's SIMDs.  The x-ranges depend on N only and
// their partial sums are added in an order that depends on their number only: every entry's summation order is a
// function of N, so results are bit-identical whatever the block size.
// LDS rows are 17 complex apart: the 16 rows of a fragment start in distinct banks.
// 48 vectors of 2^18 amplitudes: 108 us with the partial sums (374 us with a 4 x 4 register tile per thread, padded to
// 64 x 64, and one thread per entry adding 256 partial sums); 64 vectors of 2^20: 610 us.  The matrix work alone is 45
// and 290 us at the card's 73 TFLOP/s, the vectors' bytes 35 and 165.  Fragments read straight from memory, each wave
// its own, take 119 and 610 us.  Vectors a power of two apart share memory channels and pages: the host spaces them 64
// amplitudes further (64 of 2^20: 810 us without).
constexpr int SM_ROW = SM_STEP + 1;

template <int NT, int SAME, int GUARD>
__global__ __launch_bounds__(SM_THREADS) void block_partial_kernel(const double2 *__restrict__ P, int na,
                                                                   const double2 *__restrict__ Q, int nb,
                                                                   const double *__restrict__ obs, u64 N, u64 stride,
                                                                   u64 chunk, double2 *__restrict__ part) {
    constexpr int SIDES = SAME ? 1 : 2;
    __shared__ cd lds[2][SIDES][NT * 16 * SM_ROW];
    __shared__ double lobs[2][SM_STEP];
    const int tid = threadIdx.x, lane = tid & 63;
    const int i = lane & 15, k = lane >> 4;
    const int nta = (na + 15) >> 4, ntb = (nb + 15) >> 4;
    const int ta = ((tid >> 6) + (int)blockIdx.x) & 3;
    const u64 x0 = (u64)blockIdx.x * chunk;
    // thread: row tid / 16 of each 16, amplitude tid % 16; rows past the end repeat the last vector
    const int lr = tid >> 4, lx = tid & 15;
    d2 v[SIDES][NT];   // a vector type: as structs the compiler kept them in scratch memory
    double o = 0.0;
    const auto load = [&](u64 xs) {
        const u64 x = xs + lx;
        const bool in = !GUARD || x < N;
        const u64 xc = in ? x : 0;
        if (lr == 0) o = in ? obs[xc] : 0.0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int r = t * 16 + lr;
            v[0][t] = *(const d2 *)&P[(u64)(r < na ? r : na - 1) * stride + xc];
            if (!SAME) v[SIDES - 1][t] = *(const d2 *)&Q[(u64)(r < nb ? r : nb - 1) * stride + xc];
            if (GUARD && !in) v[0][t] = v[SIDES - 1][t] = d2{0.0, 0.0};
        }
    };
    const auto stage = [&](int buf) {
        if (lr == 0) lobs[buf][lx] = o;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int h = 0; h < SIDES; ++h) lds[buf][h][(t * 16 + lr) * SM_ROW + lx] = cmk(v[h][t].x, v[h][t].y);
    };
    d4 re[NT], im[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) re[t][r] = im[t][r] = 0.0;
    load(x0);
    stage(0);
    __syncthreads();
    int buf = 0;
#pragma unroll 1
    for (u64 xs = x0; xs < x0 + chunk; xs += SM_STEP, buf ^= 1) {
        const bool more = xs + SM_STEP < x0 + chunk;
        if (more) load(xs + SM_STEP);
        if (ta < nta) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const cd p = lds[buf][0][(ta * 16 + i) * SM_ROW + 4 * s + k];
                const double ob = lobs[buf][4 * s + k];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (SAME ? t > ta : t >= ntb) continue;
                    const cd q = lds[buf][SIDES - 1][(t * 16 + i) * SM_ROW + 4 * s + k];
                    const double qr = q.x * ob, qi = q.y * ob;
                    re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(p.x, qr, re[t], 0, 0, 0);
                    im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(p.x, qi, im[t], 0, 0, 0);
                    re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(p.y, qi, re[t], 0, 0, 0);
                    im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-p.y, qr, im[t], 0, 0, 0);
                }
            }
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
    }
    if (ta >= nta) return;
    double2 *out = part + (u64)blockIdx.x * na * nb;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if (SAME && t > ta) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int a = ta * 16 + 4 * r + k, b = t * 16 + i;
            if (a < na && b < nb) out[(u64)a * nb + b] = cmk(re[t][r], im[t][r]);
        }
    }
}

// G[e] = sum of the ranges' partials of entry e: 16 entries per workgroup, 16 threads each (range g, g + 16, ...), then
// the 16 sums in ascending order.  Entries above the diagonal of a block with itself are left out (nobody reads them).
__global__ __launch_bounds__(SM_THREADS) void block_finish_kernel(const double2 *__restrict__ part, int ranges, int na,
                                                                  int nb, int same, double2 *__restrict__ G) {
    __shared__ cd red[16][17];
    const int e0 = threadIdx.x & 15, g = threadIdx.x >> 4, e = blockIdx.x * 16 + e0, total = na * nb;
    const bool on = e < total && !(same && e / nb < e % nb);
    cd s = cmk(0.0, 0.0);
    if (on) {
#pragma unroll 8
        for (int w = g; w < ranges; w += 16) s = cadd(s, part[(u64)w * total + e]);
    }
    red[g][e0] = s;
    __syncthreads();
    if (g == 0 && on) {
        for (int j = 1; j < 16; ++j) s = cadd(s, red[j][e0]);
        G[e] = s;
    }
}

unsigned grid_for(uint64_t n) {
    uint64_t g = (n + SM_THREADS - 1) / SM_THREADS;
    if (g > 65536) g = 65536;
    return (unsigned)(g < 1 ? 1 : g);
}

template <int NT>
void launch_partial(hipStream_t st, unsigned grid, const double2 *P, int na, const double2 *Q, int nb, const double *obs,
                    u64 N, u64 stride, u64 chunk, int same, double2 *part) {
    if (N < SM_STEP) {
        if (same) block_partial_kernel<NT, 1, 1><<<grid, SM_THREADS, 0, st>>>(P, na, Q, nb, obs, N, stride, chunk, part);
        else block_partial_kernel<NT, 0, 1><<<grid, SM_THREADS, 0, st>>>(P, na, Q, nb, obs, N, stride, chunk, part);
    } else {
        if (same) block_partial_kernel<NT, 1, 0><<<grid, SM_THREADS, 0, st>>>(P, na, Q, nb, obs, N, stride, chunk, part);
        else block_partial_kernel<NT, 0, 0><<<grid, SM_THREADS, 0, st>>>(P, na, Q, nb, obs, N, stride, chunk, part);
    }
}

}  // namespace

extern "C" unsigned ork_sm_max_block(void) { return SM_MAX; }

// x-ranges of the block product for N = 2^n amplitudes (a function of N only); they divide N evenly
extern "C" unsigned ork_sm_parts(uint64_t N) {
    const uint64_t steps = (N + SM_STEP - 1) / SM_STEP;
    return (unsigned)(steps < SM_PARTS ? steps : SM_PARTS);
}

extern "C" int ork_sm_spread(void *stream, void *dst, const void *src, uint64_t n, uint64_t stride, int cnt) {
    unsigned g = grid_for(n);
    if (g > 4096) g = 4096;
    spread_kernel<<<dim3(g, (cnt + 7) / 8), SM_THREADS, 0, (hipStream_t)stream>>>((double2 *)dst, (const double2 *)src, n, stride, cnt);
    ORK_LAUNCH_CHECK();
    return 0;
}

extern "C" int ork_sm_axpy(void *stream, void *acc, const void *v, double wr, double wi, uint64_t n, int first) {
    axpy_kernel<<<grid_for(n), SM_THREADS, 0, (hipStream_t)stream>>>((double2 *)acc, (const double2 *)v, wr, wi, n, first);
    ORK_LAUNCH_CHECK();
    return 0;
}

// x = [a +] w x, or x = wa a + w x (scaled); a may be null
extern "C" int ork_sm_combine(void *stream, void *x, const void *a, double war, double wai, int scaled, double wr,
                              double wi, uint64_t n) {
    combine_kernel<<<grid_for(n), SM_THREADS, 0, (hipStream_t)stream>>>((double2 *)x, (const double2 *)a, war, wai, scaled,
                                                                       wr, wi, n);
    ORK_LAUNCH_CHECK();
    return 0;
}

// G[a * nb + b] = sum_x conj(P[a][x]) obs[x] Q[b][x], vectors `stride` apart; same: P and Q are one block, entries with
// a < b are not written; part: ork_sm_parts(N) * na * nb complex
extern "C" int ork_sm_block(void *stream, const void *P, int na, const void *Q, int nb, const double *obs, uint64_t N,
                            uint64_t stride, int same, void *part, void *G) {
    if (na < 1 || nb < 1 || na > SM_MAX || nb > SM_MAX || stride < N) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    const unsigned parts = ork_sm_parts(N);
    const uint64_t steps = (N + SM_STEP - 1) / SM_STEP, chunk = steps / parts * SM_STEP;   // powers of two
    const double2 *p = (const double2 *)P, *q = (const double2 *)Q;
    double2 *w = (double2 *)part;
    switch (((na > nb ? na : nb) + 15) / 16) {
    case 1: launch_partial<1>(st, parts, p, na, q, nb, obs, N, stride, chunk, same, w); break;
    case 2: launch_partial<2>(st, parts, p, na, q, nb, obs, N, stride, chunk, same, w); break;
    case 3: launch_partial<3>(st, parts, p, na, q, nb, obs, N, stride, chunk, same, w); break;
    default: launch_partial<4>(st, parts, p, na, q, nb, obs, N, stride, chunk, same, w); break;
    }
    ORK_LAUNCH_CHECK();
    block_finish_kernel<<<(na * nb + 15) / 16, SM_THREADS, 0, st>>>(w, (int)parts, na, nb, same, (double2 *)G);
    ORK_LAUNCH_CHECK();
    return 0;
}
