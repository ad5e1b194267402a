// k_tile.hpp -- a tile of 2^12 complex128 amplitudes in the registers of a workgroup of 256 threads.
//
// Every thread holds 16 amplitudes, in one of three layouts:
//   layout 0: e = u | t << 4                          (register index u = tile bits 0-3)
//   layout 1: e = (t & 15) | u << 4 | (t >> 4) << 8   (bits 4-7)
//   layout 2: e = t | u << 8                          (bits 8-11)
// Gates on the four qubits of the register index need no exchange.  A change of layout moves the real parts, then the
// imaginary parts, through one padded array of 2^12 doubles (34 KB: four workgroups per CU), written and read without
// bank conflicts (one spare slot per 16).
#pragma once
#include "k_common.hpp"

constexpr int RT_BITS = 12, RT_THREADS = 256;
constexpr unsigned RT_SIZE = 1u << RT_BITS;
constexpr int RT_SLOTS = 4096 + 256;   // doubles of LDS that change_layout needs

// the thread's 16 amplitudes: two arrays, so that either half can change layout by itself
struct Amps {
    double re[16], im[16];
};
// tile element of register u: lay_base + u * lay_step; its slot in LDS: lay_slot + u * lay_slot_step (one spare slot per 16
// elements; in layout 0 the 16 elements of a thread are one such group)
template <int LAY> __device__ __forceinline__ int lay_base(int t) {
    return LAY == 0 ? t << 4 : LAY == 1 ? (t & 15) | (t >> 4) << 8 : t;
}
template <int LAY> __device__ __forceinline__ int lay_slot(int t) {
    const int e = lay_base<LAY>(t);
    return e + (e >> 4);
}
constexpr int lay_step(int lay) { return lay == 0 ? 1 : lay == 1 ? 16 : 256; }
constexpr int lay_slot_step(int lay) { return lay == 0 ? 1 : lay == 1 ? 17 : 272; }

template <int FROM, int TO>
__device__ __forceinline__ void change_layout(Amps &v, double *lds) {
    constexpr int ws = lay_slot_step(FROM), rs = lay_slot_step(TO);
    double *w = lds + lay_slot<FROM>(threadIdx.x);
    const double *r = lds + lay_slot<TO>(threadIdx.x);
#pragma unroll
    for (int u = 0; u < 16; ++u) w[u * ws] = v.re[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) v.re[u] = r[u * rs];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) w[u * ws] = v.im[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) v.im[u] = r[u * rs];
    __syncthreads();
}

// a change of layout and, on its way, I - i u X on the qubits whose X flips the tile bits of `mask`: each thread reads its
// new elements and those at the flipped places
template <int FROM, int TO>
__device__ __forceinline__ void change_layout_flip(Amps &v, double *lds, unsigned mask, double u) {
    constexpr int ws = lay_slot_step(FROM), rs = lay_slot_step(TO);
    constexpr unsigned RB = 15u * lay_step(TO);   // tile bits of the register index
    __builtin_amdgcn_sched_barrier(0);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid) : : "memory");
    const unsigned far = (unsigned)lay_base<TO>(tid) ^ (mask & (RT_SIZE - 1) & ~RB), fu = (mask & RB) / lay_step(TO);
    double *w = lds + lay_slot<FROM>(tid);
    const double *r = lds + lay_slot<TO>(tid);
    // the flipped places' addresses are formed at each use: kept they spill
    const auto flipped = [&](int k) {
        unsigned x = far + (far >> 4);
        asm volatile("" : "+v"(x));
        return lds[x + ((unsigned)k ^ fu) * rs];
    };
    double pre[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) w[k * ws] = v.re[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        v.re[k] = r[k * rs];
        pre[k] = flipped(k);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) w[k * ws] = v.im[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        v.re[k] = fma(u, flipped(k), v.re[k]);
        v.im[k] = fma(-u, pre[k], r[k * rs]);
    }
    __syncthreads();
}
