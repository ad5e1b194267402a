// k_qaoa.hip -- batched QAOA evaluation: thousands of (graph, angles) circuits
// of uneven qubit counts in a few launches for all of them together.
//
// One evaluation is the reference's own QAOA call sequence:
//   state_plus(PURE, n); p x { exp_diag(C, gamma); rx(q, 2 beta) for q = 0..n-1 };
//   mean(C)
// (src/state/state_pure.c:30-43, src/circ/circ_pure.c:21-34,
//  src/gate/gate_pure.c:221-234, src/meas/meas_pure.c:20-30), with the same
// per-amplitude formulas for the phases and the rx with their common factor
// taken out (restored in the mean), so each instance matches a per-instance run
// of those calls to rounding (the rx of one layer act on distinct qubits and
// commute; states in HBM apply them in another order than 0..n-1).
//
// Execution: a state of n <= LT qubits stays on the chip for the whole circuit. A
// larger state (n <= 2 LT) lives in HBM and is swept in tiles of 2^LT
// amplitudes, alternating contiguous tiles and tiles gathered at stride 2^LT;
// each sweep finishes the previous layer's rx on the qubits the
// previous sweep could not reach and runs the next layer's exp_diag and rx on
// every qubit it holds: p + 1 sweeps for p layers instead of p (n + 1) gate
// passes; the last sweep reduces sum_x C(x) |psi_x|^2.  Where C(x) = C(~x), half of a state larger than a tile
// stands for all of it.
//
// Two forms. qaoa_sweep and qaoa_one_tile, the default: tiles of 2^12 amplitudes
// in registers, one launch per sweep with a workgroup for every tile of every
// evaluation. qaoa_persistent, the other shapes and phases of 2^50 and more: tiles in
// LDS, the workgroups of one launch pull evaluations from an atomic counter
// (largest first) and run each one start to finish.
#include "k_common.hpp"
#include "k_tile.hpp"

namespace {

struct QaoaEval {
    int graph;       // index into the diagonal table
    int p;           // layers
    int angle_off;   // first of this evaluation's layers in the angle rows
    int pad;
};

// a layer's row: gamma, cos beta, sin beta and the power of two by which the layer's phases scale the state
constexpr int ANG = 4;

struct QaoaGraph {
    u64 diag_off;    // offset (in doubles) of C in the diagonal arena
    u64 state_off;   // offset (in complex) of the state scratch in the state arena
    int n;
    int pad;
};

struct QaoaArgs {
    const QaoaEval *evals;
    const int *order;        // evaluation order (largest work first)
    const int *nevals;       // device scalar: evaluations in this launch
    const QaoaGraph *graphs;
    const double *angles;
    const double *diag;
    double2 *states;         // per-workgroup scratch slots for states larger than LDS
    u64 slot_elems;          // complex elements per scratch slot (2^nmax)
    double *out;
    unsigned *counter;
};

// rx(2 beta) on the pair (a, b): a' = c a - i s b, b' = -i s a + c b (gate_pure.c:221-234), with its
// scalar factor taken out: for |c| >= |s|, rx = c (I - i u X) with u = s / c; else rx = -i s (X + i u I)
// with u = c / s.  Either form costs 4 FMAs per pair instead of 4 products and 4 FMAs; the factor has
// modulus max(|c|, |s|) >= 1/sqrt 2 and, a global scale and phase of the whole layer, drops out of
// <C> once the sum is multiplied by the product of the squared moduli (max(c^2, s^2) per qubit).
struct RxScaled {
    double u;
    int swap;   // 1: the -i s (X + i u I) form
    __device__ RxScaled(double c, double s) {
        swap = fabs(c) < fabs(s);
        u = swap ? c / s : s / c;
    }
};

template <int SWAP>
__device__ __forceinline__ void rx_pair(cd &a, cd &b, double u) {
    if constexpr (!SWAP) {
        const cd na = cmk(fma(u, b.y, a.x), fma(-u, b.x, a.y));
        const cd nb = cmk(fma(u, a.y, b.x), fma(-u, a.x, b.y));
        a = na;
        b = nb;
    } else {
        const cd na = cmk(fma(-u, a.y, b.x), fma(u, a.x, b.y));
        const cd nb = cmk(fma(-u, b.y, a.x), fma(u, b.x, a.y));
        a = na;
        b = nb;
    }
}

// psi *= exp(-i C t) (circ_pure.c:27-32), times the power of two `scale`
__device__ __forceinline__ cd phase(cd v, double d, double t, double scale) {
    double s, c;
    sincos(d * t, &s, &c);
    s *= scale;
    c *= scale;
    return cmk(c * v.x + s * v.y, c * v.y - s * v.x);
}

// The scaled rx let the squared norm of a state of n qubits grow by up to 2^n per layer: past 2^1024 the sum overflows.
// Once it may have grown by 2^RESCALE_BITS, the next layer's phases take its root out again, a power of two that
// rx_scale puts back: exact, so circuits keep their bits wherever nothing overflowed.
constexpr double RESCALE_BITS = 512.0;

// product over layers of the squared modulus the scaled rx leave out, once per qubit, and of the scalings undone
__device__ double rx_scale(const double *ang, int p, int n) {
    double scale = 1.0;
    for (int l = 0; l < p; ++l) {
        const double c = ang[ANG * l + 1], s = ang[ANG * l + 2], d = ang[ANG * l + 3];
        const double f2 = fabs(c) < fabs(s) ? s * s : c * c;
        if (d != 1.0) scale /= d * d;
        for (int q = 0; q < n; ++q) scale *= f2;
    }
    return scale;
}

// LDS tiles are padded with one slot after every 8 amplitudes, so that a lane
// walking 8 consecutive amplitudes and its neighbours hit distinct banks
__device__ __forceinline__ int pad(int i) { return i + (i >> 3); }
constexpr int padded(int n) { return n + (n >> 3); }

// rx on LDS bits [b0, b1) of a tile of 2^lt amplitudes, qubits in ascending
// order, up to three qubits per pass: each thread holds the R = 2^r amplitudes of one
// r-bit group in registers and applies the r rx in qubit order, so every
// amplitude sees the same sequence of operations as gate-by-gate application.
// R is a template argument: full passes (R = 8) carry no run-time tests.
template <int THREADS, int SWAP, int R>
__device__ __forceinline__ void lds_rx_pass(cd *t, int lt, int b, double u) {
    constexpr int r = R == 8 ? 3 : (R == 4 ? 2 : 1);
    const int ngroups = 1 << (lt - r);
    const int lowmask = (1 << b) - 1;
    for (int gi = threadIdx.x; gi < ngroups; gi += THREADS) {
        const int base = ((gi & ~lowmask) << r) | (gi & lowmask);
        cd v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = t[pad(base | (j << b))];
#pragma unroll
        for (int k = 0; k < r; ++k) {
#pragma unroll
            for (int j = 0; j < R; ++j)
                if (!((j >> k) & 1)) rx_pair<SWAP>(v[j], v[j | (1 << k)], u);
        }
#pragma unroll
        for (int j = 0; j < R; ++j) t[pad(base | (j << b))] = v[j];
    }
    __syncthreads();
}

template <int THREADS, int SWAP>
__device__ __forceinline__ void lds_rx_form(cd *t, int lt, int b0, int b1, double u) {
    int b = b0;
    for (; b + 3 <= b1; b += 3) lds_rx_pass<THREADS, SWAP, 8>(t, lt, b, u);
    if (b1 - b == 2) lds_rx_pass<THREADS, SWAP, 4>(t, lt, b, u);
    else if (b1 - b == 1) lds_rx_pass<THREADS, SWAP, 2>(t, lt, b, u);
}

// one form per call (the form is the same for every thread), so each instantiation holds one butterfly
template <int THREADS>
__device__ __forceinline__ void lds_rx(cd *t, int lt, int b0, int b1, const RxScaled &rx) {
    if (rx.swap) lds_rx_form<THREADS, 1>(t, lt, b0, b1, rx.u);
    else lds_rx_form<THREADS, 0>(t, lt, b0, b1, rx.u);
}

template <int THREADS>
__device__ __forceinline__ double block_sum(double v, double *red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < THREADS / 64; ++w) s += red[w];
    __syncthreads();
    return s;
}

template <int LT, int THREADS>
__global__ __launch_bounds__(THREADS) void qaoa_persistent(QaoaArgs A) {
    __shared__ cd tile[padded(1 << LT)];
    __shared__ double red[THREADS / 64];
    __shared__ int item;
    constexpr int T = 1 << LT;
    // thread t holds tile elements t + THREADS u, u < PER; global loads go in batches of BT with every load of
    // a batch issued before the first is used (one load at a time left each thread waiting out the full
    // HBM latency per element)
    static_assert(T % THREADS == 0, "tile not a multiple of the workgroup");
    constexpr int PER = T / THREADS, BT = PER < 8 ? PER : 8;
    // loops that load C and evaluate a sincos per element: batches of 4, whose evaluations the compiler
    // interleaves (measured on the 4096-instance batch: 101k evaluations/s with 4, 98k with 2, 74k with 1)
    constexpr int BC = PER < 4 ? PER : 4;
    const int nev = *A.nevals;
    double2 *slot = A.states + (u64)blockIdx.x * A.slot_elems;

    for (;;) {
        if (threadIdx.x == 0) item = (int)atomicAdd(A.counter, 1u);
        __syncthreads();
        const int it = item;
        __syncthreads();
        if (it >= nev) break;
        const int e = A.order[it];
        const QaoaEval ev = A.evals[e];
        const QaoaGraph gr = A.graphs[ev.graph];
        const int n = gr.n;
        const u64 N = (u64)1 << n;
        const double *C = A.diag + gr.diag_off;
        const double *ang = A.angles + (u64)ev.angle_off * ANG;
        const double amp = 1.0 / sqrt((double)N);
        double acc = 0.0;

        if (n <= LT) {
            // ---- whole state in LDS ----
            for (int x = threadIdx.x; x < (int)N; x += THREADS) tile[pad(x)] = cmk(amp, 0.0);
            __syncthreads();
            for (int l = 0; l < ev.p; ++l) {
                const double g = ang[ANG * l], d = ang[ANG * l + 3];
                const RxScaled rx(ang[ANG * l + 1], ang[ANG * l + 2]);
                for (int u0 = 0; u0 < PER; u0 += BC) {
                    double cv[BC];
#pragma unroll
                    for (int u = 0; u < BC; ++u) {
                        const int x = threadIdx.x + (u0 + u) * THREADS;
                        cv[u] = x < (int)N ? C[x] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < BC; ++u) {
                        const int x = threadIdx.x + (u0 + u) * THREADS;
                        if (x < (int)N) tile[pad(x)] = phase(tile[pad(x)], cv[u], g, d);
                    }
                }
                __syncthreads();
                lds_rx<THREADS>(tile, n, 0, n, rx);
            }
            for (int u0 = 0; u0 < PER; u0 += BT) {
                double cv[BT];
#pragma unroll
                for (int u = 0; u < BT; ++u) {
                    const int x = threadIdx.x + (u0 + u) * THREADS;
                    cv[u] = x < (int)N ? C[x] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < BT; ++u) {
                    const int x = threadIdx.x + (u0 + u) * THREADS;
                    if (x < (int)N) {
                        const cd v = tile[pad(x)];
                        acc += cv[u] * (v.x * v.x + v.y * v.y);
                    }
                }
            }
        } else {
            // ---- state in HBM: p + 1 LDS-tiled passes ----
            // Pass k alternates between A tiles (contiguous: qubits 0..LT-1) and B tiles (all
            // 2^hb high indices x a run of 2^ls low indices: qubits 0..ls-1 and LT..n-1); both
            // hold tile bits ls..LT-1 that the other does not (A: qubits ls..LT-1, B: LT..n-1).
            // Pass k first finishes layer k-1 (rx on tile bits ls..LT-1, the qubits the previous
            // pass could not reach), then starts layer k (phase, rx on every tile bit), so one
            // pass per layer reads and writes the state; pass p reduces the mean instead.
            const int hb = n - LT;                 // qubits above the A tile
            const int ls = 2 * LT - n;             // log2 of the low run of a B tile
            const int S = 1 << ls;
            const u64 nchunk = (u64)1 << hb;
            for (int k = 0; k <= ev.p; ++k) {
                const bool btile = k & 1;
                const bool last = (k == ev.p);
                const double g = last ? 0.0 : ang[ANG * k], d = last ? 1.0 : ang[ANG * k + 3];
                const RxScaled rx(last ? 1.0 : ang[ANG * k + 1], last ? 0.0 : ang[ANG * k + 2]);
                const RxScaled rxp(k ? ang[ANG * (k - 1) + 1] : 1.0, k ? ang[ANG * (k - 1) + 2] : 0.0);
                for (u64 ch = 0; ch < nchunk; ++ch) {
                    const u64 lo0 = ch << ls;
                    // global index of tile element x
#define QIDX(x) (btile ? ((((u64)(x) >> ls) << LT) | (lo0 + (u64)((x) & (S - 1)))) : ((ch << LT) + (u64)(x)))
                    // C of the thread's elements of a batch, all loads in flight
#define LOAD_C(cv, u0)                                                                       \
    _Pragma("unroll") for (int u = 0; u < BC; ++u) cv[u] = C[QIDX(threadIdx.x + ((u0) + u) * THREADS)];
                    if (k == 0) {
                        for (int u0 = 0; u0 < PER; u0 += BC) {
                            double cv[BC];
                            LOAD_C(cv, u0)
#pragma unroll
                            for (int u = 0; u < BC; ++u)
                                tile[pad(threadIdx.x + (u0 + u) * THREADS)] = phase(cmk(amp, 0.0), cv[u], g, d);
                        }
                        __syncthreads();
                    } else {
                        for (int u0 = 0; u0 < PER; u0 += BT) {
                            cd v[BT];
#pragma unroll
                            for (int u = 0; u < BT; ++u) v[u] = slot[QIDX(threadIdx.x + (u0 + u) * THREADS)];
#pragma unroll
                            for (int u = 0; u < BT; ++u) tile[pad(threadIdx.x + (u0 + u) * THREADS)] = v[u];
                        }
                        __syncthreads();
                        lds_rx<THREADS>(tile, LT, ls, LT, rxp);
                        if (!last) {
                            for (int u0 = 0; u0 < PER; u0 += BC) {
                                double cv[BC];
                                LOAD_C(cv, u0)
#pragma unroll
                                for (int u = 0; u < BC; ++u) {
                                    const int x = threadIdx.x + (u0 + u) * THREADS;
                                    tile[pad(x)] = phase(tile[pad(x)], cv[u], g, d);
                                }
                            }
                            __syncthreads();
                        }
                    }
                    if (!last) {
                        lds_rx<THREADS>(tile, LT, 0, LT, rx);
                        for (int x = threadIdx.x; x < T; x += THREADS) slot[QIDX(x)] = tile[pad(x)];
                    } else {
                        for (int u0 = 0; u0 < PER; u0 += BT) {
                            double cv[BT];
#pragma unroll
                            for (int u = 0; u < BT; ++u) cv[u] = C[QIDX(threadIdx.x + (u0 + u) * THREADS)];
#pragma unroll
                            for (int u = 0; u < BT; ++u) {
                                const cd v = tile[pad(threadIdx.x + (u0 + u) * THREADS)];
                                acc += cv[u] * (v.x * v.x + v.y * v.y);
                            }
                        }
                    }
#undef LOAD_C
#undef QIDX
                    __syncthreads();
                }
            }
        }
        const double tot = block_sum<THREADS>(acc, red);
        if (threadIdx.x == 0) A.out[e] = tot * rx_scale(ang, ev.p, n);
        __syncthreads();
    }
}

// ---- tiles of 2^12 amplitudes in registers -----------------------------------------------------------
// qaoa_persistent keeps its tile in LDS and takes it through registers and back for every three qubits and for the
// phases: nine round trips per layer of a 20-qubit state, 288 B of LDS traffic per amplitude, half of its cycles bank
// conflicts, and that was its time.  Here a workgroup of 256 threads holds the tile in registers (k_tile.hpp): an rx on
// four qubits, a phase, a load or a store happens in one of the three layouts without LDS, and a sweep of a 17- to 20-qubit
// state changes layout three times: 96 B of LDS traffic per amplitude.
//
// The sweeps are those of qaoa_persistent (k = 0..p, alternating contiguous and gathered tiles).  Sweep k finishes layer
// k - 1 on tile bits ls..11 and runs layer k's phase and rx on every tile bit; the rx of one layer commute, so a sweep
// visits the layouts in the order that needs fewest changes: 1 (load, finish bits 4-7), 0 (finish bits 0-3, only where
// ls < 4), 2 (finish bits 8-11, phase, rx), 0 (rx), 1 (rx, store); with ls >= 8 it starts in layout 2.
// A launch is one sweep k over all tiles of all states that have it, so a single large state fills the chip as well as a
// thousand do: with a workgroup per evaluation one state of 18 qubits took 2180 us, now 77; 300 of 4 to 11 qubits
// (qaoa_one_tile) 231 and 180; with SYM = 0, 64 of 16 qubits 632 and 187, six of 21 to 24 qubits 185 and 5.2 ms, 4096
// evaluations of 10 to 20 qubits and 1 to 8 layers 38.8 and 28.2 ms a call.  Memory bounds it: 140 GB of amplitudes and cost
// diagonal in runs of 256 and 128 B take 26 ms with everything else left out, the rest alone 14.  Nontemporal accesses gain
// nothing.
//
// SYM = 1: half of the state, for a cost with C(x) = C(~x) (any sum of pair terms: MaxCut).  |+>, the phases and the rx all
// keep psi(x) = psi(~x), so m = n - 1 bits y name an amplitude: y_i = x_i ^ x_(n-1) for i < 12, y_i = x_i ^ x_v for i >= 12,
// with v the qubit of bit vb < 5.  The X of qubits i < n - 1 other than v flips y_i alone.  The X of qubit n - 1 flips y_0 to y_11,
// all inside a contiguous tile; that of v flips y_vb and y_12 to y_(m-1), all inside a gathered tile, whose low run holds bit vb.
// So either sweep still reaches what the other leaves: the contiguous one bits 0-11 without vb and qubit n - 1, the gathered
// one its tile's bits without vb and qubit v; the two wide flips ride on a change of layout (change_layout_flip).  The state
// of x_(n-1) = 0 has C(y) at y, with bits 12.. complemented where y_vb = 1: in runs of 2^vb, 128 B up to 20 qubits.  The
// product of a layer's X over all qubits is 1 here, so RxFlip.flip is not needed.  Half the bytes and the work:
// 4096 evaluations of 10 to 20 qubits 28.2 -> 16.0 ms a call (2 of them on the host), 64 of 16 qubits 187 -> 140 us, 700 of 12
// to 17 1.46 -> 0.97 ms, six of 21 to 24 5.4 -> 1.9 ms, one of 18 77 us both ways.

// a value that is the same in every lane, as a scalar: what is loaded by a computed index counts as per-lane otherwise, and
// with it every branch and address that depends on it
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ u64 uni(u64 x) {
    return (u64)(unsigned)uni((int)(unsigned)(x >> 32)) << 32 | (unsigned)uni((int)(unsigned)x);
}
__device__ __forceinline__ double uni(double x) { return __longlong_as_double((long long)uni((u64)__double_as_longlong(x))); }

// rx without its scalar factor in one form: c I - i s X = c (I - i u X) with u = s / c where |c| >= |s|, else
// -i s X (I - i u X) with u = -c / s.  The X flips every qubit of the layer; it commutes with every later rx, so the
// register version leaves it out and reads C at the complemented index from then on (RxFlip.flip).
struct RxFlip {
    double u;
    bool flip;
    __device__ RxFlip(double c, double s) {
        flip = fabs(c) < fabs(s);
        u = flip ? -c / s : s / c;
    }
};
// sin and cos of x for |x| < 2^50: reduction to [-pi/4, pi/4] by the nearest multiple k of pi/2 with pi/2 as the sum of two
// doubles (x - k P1 is exact in one fma: a multiple of 2^-52 below 1; the second fma rounds once; the sum is off by k
// 1.5e-33), then Taylor's series to x^17 / 17! and x^18 / 18!, whose next terms are below 2^-60 there.  Off by at most 2^-52.6
// (checked against 50 digits).  The library's sincos carries a reduction for any argument, whose registers did not fit
// beside 16 amplitudes.
__device__ __forceinline__ void sincos_bounded(double x, double &s, double &c) {
    const double kd = fma(x, 0.63661977236758138, 6755399441055744.0);   // k + 1.5 2^52: k in the low bits
    const int q = (int)(unsigned)(unsigned long long)__double_as_longlong(kd);
    const double k = kd - 6755399441055744.0;
    double r = fma(-k, 1.5707963267948966, x);
    r = fma(-k, 6.123233995736766e-17, r);
    const double z = r * r;
    double a = 2.8114572543455206e-15;
    a = fma(a, z, -7.647163731819816e-13);
    a = fma(a, z, 1.6059043836821613e-10);
    a = fma(a, z, -2.505210838544172e-08);
    a = fma(a, z, 2.7557319223985893e-06);
    a = fma(a, z, -0.0001984126984126984);
    a = fma(a, z, 0.008333333333333333);
    a = fma(a, z, -0.16666666666666666);
    const double sn = fma(a * z, r, r);
    double b = -1.5619206968586225e-16;
    b = fma(b, z, 4.779477332387385e-14);
    b = fma(b, z, -1.1470745597729725e-11);
    b = fma(b, z, 2.08767569878681e-09);
    b = fma(b, z, -2.755731922398589e-07);
    b = fma(b, z, 2.48015873015873e-05);
    b = fma(b, z, -0.001388888888888889);
    b = fma(b, z, 0.041666666666666664);
    b = fma(b, z, -0.5);
    const double cs = fma(b, z, 1.0);
    const double s0 = q & 1 ? cs : sn, c0 = q & 1 ? sn : cs;
    s = q & 2 ? -s0 : s0;
    c = (q + 1) & 2 ? -c0 : c0;
}

// I - i u X on the register bits of `mask`; u = 0 leaves a bit as it is, so that no branch splits the registers' lives
__device__ __forceinline__ void rx4(Amps &v, unsigned mask, double u) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        __builtin_amdgcn_sched_barrier(0);
        const double uk = (mask >> k) & 1 ? u : 0.0;
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (!((j >> k) & 1)) {
                const int i = j | (1 << k);
                const double ar = v.re[j], ai = v.im[j], br = v.re[i], bi = v.im[i];
                v.re[j] = fma(uk, bi, ar);
                v.im[j] = fma(-uk, br, ai);
                v.re[i] = fma(uk, ai, br);
                v.im[i] = fma(-uk, ar, bi);
            }
    }
}

// DEEP: the layers' scalings (rescale_kernel), in kernels of their own: beside the others the test alone cost 0.6 % of a batch
__device__ __forceinline__ void scale16(Amps &v, double d) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        v.re[u] *= d;
        v.im[u] *= d;
    }
}

// Memory index of a tile element: f(x) = (x >> ls) << 12 | (x & (2^ls - 1)) past the chunk's own offset in a gathered tile,
// x itself in a contiguous one.  f acts on bits and a thread's and a register's share of x have no bit in common, so the
// two shares join by xor, also through a further map that is linear over bits.
struct TileMap {
    unsigned chunk;   // offset of the tile's element 0
    int ls;           // 12: contiguous
    __device__ __forceinline__ unsigned f(unsigned x) const { return (x >> ls) << RT_BITS | (x & ((1u << ls) - 1)); }
    template <int LAY> __device__ __forceinline__ unsigned reg(int u) const { return chunk | f((unsigned)(u * lay_step(LAY))); }
};
// Byte offset of an amplitude in a state slot: blocks of 16 real parts and 16 imaginary parts (256 B, the run of a gathered
// tile of 20 qubits), and the blocks of each 2^12 amplitudes in an order that turns with the bits above: in index order the
// 2^(n - 12) runs of a gathered tile lie 64 KB apart, on few of the memory channels (4 to 6 % of the whole batch).
__device__ __forceinline__ unsigned slot_off(unsigned x) {
    const unsigned y = x ^ ((x >> 8) & 0xff0u);
    return (y >> 4) << 8 | (y & 15u) << 3;
}
// An array as a buffer resource: an access adds a thread's and a scalar byte offset to it in one instruction.  (Through
// pointers the compiler kept a 64-bit address per register and access alive across the sweep, over 100 VGPRs.) 
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t Buf;
__device__ __forceinline__ Buf buffer(const void *p, u64 bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)(unsigned)bytes, 0x00020000);
}
__device__ __forceinline__ double load8(Buf b, unsigned off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, (int)off, 0, 0));
}
template <int LAY> __device__ __forceinline__ void load_amps(Amps &v, Buf s, const TileMap &m, unsigned off) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int x = (int)(off ^ slot_off(m.reg<LAY>(u)));
        v.re[u] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(s, x, 0, 0));
        v.im[u] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(s, x + 128, 0, 0));
    }
}
template <int LAY> __device__ __forceinline__ void store_amps(const Amps &v, Buf s, const TileMap &m, unsigned off) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int x = (int)(off ^ slot_off(m.reg<LAY>(u)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v.re[u]), s, x, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v.im[u]), s, x + 128, 0, 0);
    }
}

// the cost diagonal, read at the complemented index while `flip` is set
struct Diag {
    Buf b;
    unsigned last;   // 2^n - 1
    bool flip;
    template <int LAY> __device__ __forceinline__ double at(const TileMap &m, int u, unsigned off) const {
        return load8(b, (off ^ m.reg<LAY>(u) ^ (flip ? last : 0u)) * 8);
    }
    // states of at most one tile, whose elements past 2^n do not exist: 0 there
    template <int LAY> __device__ __forceinline__ double at_small(int u, unsigned off) const {
        const unsigned x = off | (unsigned)(u * lay_step(LAY));
        return x <= last ? load8(b, (x ^ (flip ? last : 0u)) * 8) : 0.0;
    }
};

// the phases of the thread's 16 amplitudes in layout LAY, RT_BATCH loads and sincos at a time
template <int LAY, int SMALL, int RT_BATCH = 4>
__device__ __forceinline__ void phase16(Amps &v, const Diag &C, const TileMap &m, unsigned off, double g) {
#pragma unroll
    for (int u0 = 0; u0 < 16; u0 += RT_BATCH) {
        double cv[RT_BATCH];
#pragma unroll
        for (int u = 0; u < RT_BATCH; ++u) cv[u] = SMALL ? C.at_small<LAY>(u0 + u, off) : C.at<LAY>(m, u0 + u, off);
#pragma unroll
        for (int u = 0; u < RT_BATCH; ++u) {
            if (u == 0) __builtin_amdgcn_sched_barrier(0);
            double s, c;
            sincos_bounded(cv[u] * g, s, c);
            const double x = v.re[u0 + u], y = v.im[u0 + u];
            v.re[u0 + u] = fma(c, x, s * y);
            v.im[u0 + u] = fma(c, y, -(s * x));
        }
    }
}
template <int LAY, int SMALL>
__device__ __forceinline__ double mean16(const Amps &v, const Diag &C, const TileMap &m, unsigned off) {
    double acc = 0.0;
#pragma unroll
    for (int u0 = 0; u0 < 16; u0 += 8) {
        double cv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) cv[u] = SMALL ? C.at_small<LAY>(u0 + u, off) : C.at<LAY>(m, u0 + u, off);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += cv[u] * (v.re[u0 + u] * v.re[u0 + u] + v.im[u0 + u] * v.im[u0 + u]);
    }
    return acc;
}

// an evaluation of a launch
struct QaoaRec {
    u64 diag_off;    // of C in the diagonal arena (doubles)
    u64 tile;        // of its first tile in the state slots (tiles of 2^12 amplitudes)
    int angle_off;   // of its first layer in the angle rows
    int p, n, m;     // layers, qubits, bits of the stored index: n, or n - 1 (SYM)
    int out, pad;    // place of its result
};

// states of at most one tile: a workgroup runs the whole circuit
template <int SYM, int DEEP>
__global__ __launch_bounds__(RT_THREADS, SYM ? 2 : 3) void qaoa_one_tile(const QaoaRec *__restrict__ recs,
                                                              const double *__restrict__ angles,
                                                              const double *__restrict__ diag, double *__restrict__ out) {
    __shared__ double lds[RT_SLOTS];
    __shared__ double red[RT_THREADS / 64];
    const int t = threadIdx.x;
    const QaoaRec r = recs[blockIdx.x];
    const int n = uni(r.m), p = uni(r.p);
    const double *ang = angles + (u64)r.angle_off * ANG;
    Diag C{buffer(diag + r.diag_off, (u64)8 << n), (1u << n) - 1, false};
    // layouts 2 and 1 take turns in holding the phase, 0 in between.  Amplitudes past 2^n are 0 and stay 0 (their bits carry
    // no rx)
    const TileMap m{0, RT_BITS};
    const unsigned b0 = n >= 4 ? 15u : (1u << n) - 1, b1 = n >= 8 ? 15u : n > 4 ? (1u << (n - 4)) - 1 : 0u,
                   b2 = n > 8 ? (1u << (n - 8)) - 1 : 0u;
    const double amp = 1.0 / sqrt((double)(1u << n));
    Amps v;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        v.re[u] = (t | u << 8) < (1 << n) ? amp : 0.0;
        v.im[u] = 0.0;
    }
    for (int l = 0; l < p; ++l) {
        const double g = uni(ang[ANG * l]);
        const RxFlip rx(uni(ang[ANG * l + 1]), uni(ang[ANG * l + 2]));
        if (DEEP) scale16(v, uni(ang[ANG * l + 3]));
        if (l & 1) {
            phase16<1, 1>(v, C, m, (unsigned)lay_base<1>(t), g);
            rx4(v, b1, rx.u);
            if (SYM) change_layout_flip<1, 0>(v, lds, C.last, rx.u);
            else change_layout<1, 0>(v, lds);
            rx4(v, b0, rx.u);
            change_layout<0, 2>(v, lds);
            rx4(v, b2, rx.u);
        } else {
            phase16<2, 1>(v, C, m, (unsigned)t, g);
            rx4(v, b2, rx.u);
            if (SYM) change_layout_flip<2, 0>(v, lds, C.last, rx.u);
            else change_layout<2, 0>(v, lds);
            rx4(v, b0, rx.u);
            change_layout<0, 1>(v, lds);
            rx4(v, b1, rx.u);
        }
        if (!SYM) C.flip ^= rx.flip;
    }
    const double acc = p & 1 ? mean16<1, 1>(v, C, m, (unsigned)lay_base<1>(t)) : mean16<2, 1>(v, C, m, (unsigned)t);
    const double tot = block_sum<RT_THREADS>(acc, red);
    if (t == 0) out[r.out] = tot * rx_scale(ang, p, r.n);
}

// One sweep k of every larger state that has it (p >= k): a workgroup per tile.  The evaluations are sorted by qubits, then
// by layers, both descending, so the tiles of a sweep are a few runs of equal 2^(n - 12).
constexpr int RT_CLASSES = 12;   // 13 to 24 index bits
struct SweepArgs {
    const QaoaRec *recs;
    const double *angles, *diag;
    double2 *states;
    double *part;                     // per tile of the slots: its share of the mean
    int k, nclass;
    unsigned first[RT_CLASSES + 1];   // first workgroup of each class
    int rec[RT_CLASSES], n[RT_CLASSES];   // first record and index bits of each
};

template <int SYM, int DEEP>
__global__ __launch_bounds__(RT_THREADS, 3) void qaoa_sweep(SweepArgs A) {
    __shared__ double lds[RT_SLOTS];
    __shared__ double red[RT_THREADS / 64];
    const int t = threadIdx.x, k = A.k;
    int c = 0;
    while (c + 1 < A.nclass && blockIdx.x >= A.first[c + 1]) ++c;
    const int n = A.n[c];
    const unsigned b = blockIdx.x - A.first[c], ch = b & ((1u << (n - RT_BITS)) - 1);
    const QaoaRec r = A.recs[A.rec[c] + (int)(b >> (n - RT_BITS))];
    const double *ang = A.angles + (u64)r.angle_off * ANG;
    const bool gathered = k & 1, last = k == uni(r.p);
    // the flips of the layers before k
    bool flip = false;
    for (int l = 0; !SYM && l < k; ++l) flip ^= fabs(uni(ang[ANG * l + 1])) < fabs(uni(ang[ANG * l + 2]));
    const Diag C{buffer(A.diag + r.diag_off, (u64)8 << n), (1u << n) - 1, flip};
    const double g = last ? 0.0 : uni(ang[ANG * k]);
    const RxFlip rx(last ? 1.0 : uni(ang[ANG * k + 1]), last ? 0.0 : uni(ang[ANG * k + 2]));
    const RxFlip rxp(k ? uni(ang[ANG * k - 3]) : 1.0, k ? uni(ang[ANG * k - 2]) : 0.0);
    const int ls = 2 * RT_BITS - n;
    // layer k - 1 is left to finish on tile bits ls..11, by layout
    const unsigned f0 = ls < 4 ? 15u & (15u << ls) : 0u;
    const unsigned f1 = ls < 8 ? 15u & (15u << (ls > 4 ? ls - 4 : 0)) : 0u;
    const unsigned f2 = 15u & (15u << (ls > 8 ? ls - 8 : 0));
    const TileMap m{ch << (gathered ? ls : RT_BITS), gathered ? ls : RT_BITS};
    const unsigned off2 = m.f((unsigned)t), soff1 = slot_off(m.f((unsigned)lay_base<1>(t))), soff2 = slot_off(off2);
    const Buf S = buffer(A.states + (r.tile << RT_BITS), (u64)16 << n);
    // SYM: the bit of qubit v; the tile bits that the X of qubit n - 1 or v, whichever is in reach, flips; the place in
    // the diagonal
    const int vb = ls < 5 ? ls - 1 : 4;
    const unsigned all = SYM ? (RT_SIZE - 1) & ~(1u << vb) : RT_SIZE - 1;
    const unsigned cross = gathered ? (RT_SIZE - 1) & (~0u << ls | 1u << vb) : RT_SIZE - 1;
    const unsigned coff2 = SYM && (off2 >> vb & 1) ? off2 ^ (C.last & ~(RT_SIZE - 1)) : off2;
    Amps v;
    if (k == 0) {
        const double amp = 1.0 / sqrt((double)(1u << n));
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            v.re[u] = amp;
            v.im[u] = 0.0;
        }
    } else {
        if (f1) {
            load_amps<1>(v, S, m, soff1);
            rx4(v, f1, rxp.u);
            if (f0) {
                change_layout<1, 0>(v, lds);
                rx4(v, f0, rxp.u);
                if (SYM) change_layout_flip<0, 2>(v, lds, cross, rxp.u);
                else change_layout<0, 2>(v, lds);
            } else {
                if (SYM) change_layout_flip<1, 2>(v, lds, cross, rxp.u);
                else change_layout<1, 2>(v, lds);
            }
        } else {
            load_amps<2>(v, S, m, soff2);
            if (SYM) change_layout_flip<2, 2>(v, lds, cross, rxp.u);
        }
        rx4(v, f2, rxp.u);
    }
    double acc = 0.0;
    if (!last) {
        if (DEEP) scale16(v, uni(ang[ANG * k + 3]));
        phase16<2, 0, SYM ? 2 : 4>(v, C, m, coff2, g);   // 4 spill beside change_layout_flip
        rx4(v, 15u, rx.u);
        if (SYM) change_layout_flip<2, 0>(v, lds, cross, rx.u);
        else change_layout<2, 0>(v, lds);
        rx4(v, all & 15u, rx.u);
        change_layout<0, 1>(v, lds);
        rx4(v, all >> 4 & 15u, rx.u);
        // formed anew: kept from the loads it spills
        int t1 = t;
        asm volatile("" : "+v"(t1));
        store_amps<1>(v, S, m, slot_off(m.f((unsigned)lay_base<1>(t1))));
    } else {
        acc = mean16<2, 0>(v, C, m, coff2);
    }
    // apart from the branch above: with a divergent branch inside, the compiler keeps the amplitudes of one side alive
    // across the other
    if (last) {
        const double tot = block_sum<RT_THREADS>(acc, red);
        if (t == 0) A.part[r.tile + ch] = tot;
    }
}

// the tiles' shares of each mean, in a fixed order
__global__ __launch_bounds__(256) void qaoa_finish(const QaoaRec *__restrict__ recs, const double *__restrict__ angles,
                                                   const double *__restrict__ part, double *__restrict__ out) {
    __shared__ double red[4];
    const QaoaRec r = recs[blockIdx.x];
    double acc = 0.0;
    for (int i = threadIdx.x; i < 1 << (r.m - RT_BITS); i += 256) acc += part[r.tile + (u64)i];
    const double tot = block_sum<256>(acc, red);
    if (threadIdx.x == 0) out[r.out] = tot * rx_scale(angles + (u64)r.angle_off * ANG, r.p, r.n);
}

__global__ void reset_counter(unsigned *c) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *c = 0u;
}

// A call's list from pinned host memory: rows of gamma, then of beta, as the per-layer rows that the
// kernels read, and the records.  One launch and no wait in place of two copies from pageable memory (25 to 30 us of every
// call, one evaluation of 18 qubits 100 -> 77 us); the cosines took the host 0.7 of 16.8 ms for 4096 evaluations.
__global__ __launch_bounds__(256) void stage_kernel(const double *__restrict__ gb, u64 rows, double *__restrict__ angles,
                                                    const u64 *__restrict__ recs, u64 words, u64 *__restrict__ dst) {
    const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
    if (i < words) dst[i] = recs[i];
    if (i >= rows) return;
    const double theta = 2.0 * gb[rows + i];   // rx(q, 2 beta): the reference evaluates cos(theta / 2) and sin(theta / 2)
    double s, c;
    sincos(theta / 2.0, &s, &c);
    angles[ANG * i] = gb[i];
    angles[ANG * i + 1] = c;
    angles[ANG * i + 2] = s;
    angles[ANG * i + 3] = 1.0;
}

// the scalings of circuits deep enough to need any: one thread per evaluation
__global__ __launch_bounds__(64) void rescale_kernel(const QaoaRec *__restrict__ recs, int count, double *__restrict__ angles) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= count) return;
    const QaoaRec r = recs[i];
    double *ang = angles + (u64)r.angle_off * ANG, grown = 0.0;   // log2 of the squared norm's growth since the last
    for (int l = 0; l < r.p; ++l) {
        if (grown >= RESCALE_BITS) {
            const int h = (int)(grown * 0.5);
            grown -= 2.0 * h;
            ang[ANG * l + 3] = ldexp(1.0, -h);
        }
        const double c = ang[ANG * l + 1], s = ang[ANG * l + 2];
        grown -= (double)r.n * log2(fmax(c * c, s * s));
    }
}

// C(x) = sum_(i,j) w_ij [x_i != x_j] for one graph
__global__ __launch_bounds__(256) void maxcut_diag_kernel(double *__restrict__ out, u64 N, int ne,
                                                         const int *__restrict__ ei, const int *__restrict__ ej,
                                                         const double *__restrict__ w) {
    const u64 x = (u64)blockIdx.x * 256 + threadIdx.x;
    if (x >= N) return;
    double acc = 0.0;
    for (int k = 0; k < ne; ++k)
        if (((x >> ei[k]) ^ (x >> ej[k])) & 1) acc += w[k];
    out[x] = acc;
}

// info[2 g] = the largest |C| of graph g, infinity if any is not finite; info[2 g + 1] = 0 if C(x) = C(~x) for every x, else
// not 0.  Cleared first; workgroups of one graph join through integer maxima (a double that is not negative orders like its
// bits).  Up to 256 workgroups per graph, each at least INFO_RUN pairs: a handle for one graph of 20, 22 and 24
// qubits takes 0.19, 0.45 and 0.75 ms to make and destroy, 0.34, 1.17 and 4.6 with one workgroup per graph.
constexpr u64 INFO_RUN = 4096;
__global__ __launch_bounds__(256) void diag_info_kernel(const QaoaGraph *__restrict__ graphs, const double *__restrict__ diag,
                                                        u64 *__restrict__ info) {
    __shared__ double red[256];
    __shared__ int differ;
    const QaoaGraph g = graphs[blockIdx.x];
    const double *C = diag + g.diag_off;
    const u64 N = (u64)1 << g.n;
    if ((u64)blockIdx.y * 256 >= N / 2) return;
    double m = 0.0;
    bool diff = false;
    if (threadIdx.x == 0) differ = 0;
    __syncthreads();
#pragma unroll 4
    for (u64 x = (u64)blockIdx.y * 256 + threadIdx.x; x < N / 2; x += 256 * (u64)gridDim.y) {
        const double a = C[x], b = C[N - 1 - x], h = fmax(fabs(a), fabs(b));
        diff |= !(a == b);
        m = fmax(m, fabs(a) <= 1.7976931348623157e308 && fabs(b) <= 1.7976931348623157e308 ? h : __builtin_huge_val());
    }
    if (diff) differ = 1;
    red[threadIdx.x] = m;
    __syncthreads();
    for (int h = 128; h; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicMax((unsigned long long *)info + 2 * blockIdx.x, (unsigned long long)__double_as_longlong(red[0]));
        if (differ) atomicMax((unsigned long long *)info + 2 * blockIdx.x + 1, 1ull);
    }
}

template <int LT, int THREADS>
int launch_qaoa(hipStream_t st, const QaoaArgs &a, int grid) {
    reset_counter<<<1, 64, 0, st>>>(a.counter);
    ORK_LAUNCH_CHECK();
    qaoa_persistent<LT, THREADS><<<grid, THREADS, 0, st>>>(a);
    ORK_LAUNCH_CHECK();
    return 0;
}

}  // namespace

// ---- C ABI (used by the host module ork_qaoa.c) ----------------------------------------------
extern "C" int ork_qaoa_launch(void *stream, int lt, int threads, int grid, const void *evals, const int *order,
                               const int *nevals, const void *graphs, const double *angles, const double *diag,
                               void *states, uint64_t slot_elems, double *out, unsigned *counter) {
    QaoaArgs a;
    a.evals = (const QaoaEval *)evals;
    a.order = order;
    a.nevals = nevals;
    a.graphs = (const QaoaGraph *)graphs;
    a.angles = angles;
    a.diag = diag;
    a.states = (double2 *)states;
    a.slot_elems = slot_elems;
    a.out = out;
    a.counter = counter;
    hipStream_t st = (hipStream_t)stream;
#define ORK_QCASE(L, TH) if (lt == L && threads == TH) return launch_qaoa<L, TH>(st, a, grid);
    ORK_QCASE(10, 256) ORK_QCASE(10, 512) ORK_QCASE(10, 1024)
    ORK_QCASE(11, 256) ORK_QCASE(11, 512) ORK_QCASE(11, 1024)
    ORK_QCASE(12, 512) ORK_QCASE(12, 1024)
    ORK_QCASE(13, 512) ORK_QCASE(13, 1024)
#undef ORK_QCASE
    return (int)hipErrorInvalidValue;
}

// recs: `count` QaoaRec on the device, all of one form (sym), sorted by index bits, then by layers, both descending; n and p:
// their index bits and layers on the host; the states of more than 12 bits have their tiles in `states`, one partial sum per
// tile in `part`; deep: their layers' scalings are not all 1
extern "C" int ork_qaoa_sweeps(void *stream, int sym, int deep, const void *recs, const int *n, const int *p, int count,
                               const double *angles, const double *diag, void *states, double *part, double *out) {
    hipStream_t st = (hipStream_t)stream;
    const QaoaRec *r = (const QaoaRec *)recs;
    int large = 0, pmax = 0;
    while (large < count && n[large] > RT_BITS) {
        if (n[large] > 2 * RT_BITS) return (int)hipErrorInvalidValue;
        if (p[large] > pmax) pmax = p[large];
        ++large;
    }
    if (count > large) {
        auto *kernel = sym ? (deep ? qaoa_one_tile<1, 1> : qaoa_one_tile<1, 0>)
                           : (deep ? qaoa_one_tile<0, 1> : qaoa_one_tile<0, 0>);
        kernel<<<count - large, RT_THREADS, 0, st>>>(r + large, angles, diag, out);
        ORK_LAUNCH_CHECK();
    }
    for (int k = 0; k <= pmax && large; ++k) {
        SweepArgs A;
        A.recs = r;
        A.angles = angles;
        A.diag = diag;
        A.states = (double2 *)states;
        A.part = part;
        A.k = k;
        A.nclass = 0;
        unsigned blocks = 0;
        for (int i = 0; i < large;) {
            int m = 0, j = i;
            for (; j < large && n[j] == n[i]; ++j) m += p[j] >= k;   // the first m of the class
            if (m) {
                A.first[A.nclass] = blocks;
                A.rec[A.nclass] = i;
                A.n[A.nclass++] = n[i];
                blocks += (unsigned)m << (n[i] - RT_BITS);
            }
            i = j;
        }
        A.first[A.nclass] = blocks;
        auto *kernel = sym ? (deep ? qaoa_sweep<1, 1> : qaoa_sweep<1, 0>) : (deep ? qaoa_sweep<0, 1> : qaoa_sweep<0, 0>);
        kernel<<<blocks, RT_THREADS, 0, st>>>(A);
        ORK_LAUNCH_CHECK();
    }
    if (large) {
        qaoa_finish<<<large, 256, 0, st>>>(r, angles, part, out);
        ORK_LAUNCH_CHECK();
    }
    return 0;
}

extern "C" int ork_qaoa_stage(void *stream, const double *gb, uint64_t rows, double *angles, const void *recs, int nrecs,
                              void *recs_dst) {
    static_assert(sizeof(QaoaRec) % sizeof(u64) == 0, "copied in words");
    const u64 words = (u64)nrecs * (sizeof(QaoaRec) / sizeof(u64)), n = rows > words ? rows : words;
    stage_kernel<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(gb, rows, angles, (const u64 *)recs, words,
                                                                              (u64 *)recs_dst);
    ORK_LAUNCH_CHECK();
    return 0;
}

// recs_dev: `count` staged records; where n p < 768 for all of them the state's squared norm stays below 2^768 and no
// scaling is needed
extern "C" int ork_qaoa_rescale(void *stream, const void *recs_dev, int count, double *angles) {
    rescale_kernel<<<(unsigned)(count + 63) / 64, 64, 0, (hipStream_t)stream>>>((const QaoaRec *)recs_dev, count, angles);
    ORK_LAUNCH_CHECK();
    return 0;
}

// info: 2 words per graph, all 0; nmax: the largest graph's qubits
extern "C" int ork_qaoa_diag_info(void *stream, int ngraphs, int nmax, const void *graphs, const double *diag, uint64_t *info) {
    const u64 runs = ((u64)1 << nmax) / 2 / INFO_RUN;
    diag_info_kernel<<<dim3(ngraphs, (unsigned)(runs < 1 ? 1 : runs > 256 ? 256 : runs)), 256, 0, (hipStream_t)stream>>>(
        (const QaoaGraph *)graphs, diag, (u64 *)info);
    ORK_LAUNCH_CHECK();
    return 0;
}

extern "C" int ork_qaoa_occupancy(int lt, int threads, int *blocks_per_cu) {
    hipError_t e = hipErrorInvalidValue;
    if (lt == RT_BITS && threads == RT_THREADS)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, qaoa_sweep<0, 0>, RT_THREADS, 0);
#define ORK_QOCC(L, TH) \
    if (lt == L && threads == TH) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, qaoa_persistent<L, TH>, TH, 0);
    ORK_QOCC(10, 256) ORK_QOCC(10, 512) ORK_QOCC(10, 1024)
    ORK_QOCC(11, 256) ORK_QOCC(11, 512) ORK_QOCC(11, 1024)
    ORK_QOCC(12, 512) ORK_QOCC(12, 1024)
    ORK_QOCC(13, 512) ORK_QOCC(13, 1024)
#undef ORK_QOCC
    return (int)e;
}

extern "C" int ork_maxcut_diag(void *stream, double *out, int n, int ne, const int *ei, const int *ej,
                               const double *w) {
    const u64 N = (u64)1 << n;
    maxcut_diag_kernel<<<(unsigned)((N + 255) / 256), 256, 0, (hipStream_t)stream>>>(out, N, ne, ei, ej, w);
    ORK_LAUNCH_CHECK();
    return 0;
}
