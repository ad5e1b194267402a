// k_reduce.hpp -- sums over a whole launch: one partial sum per workgroup, stored in pinned host memory and added there
// after the stream has been waited for, in an order that depends on their number only.
//
// An expectation value on few qubits is latency: with a second launch for the last sum and a copy of its 8 B into the
// caller's pageable memory it took 25 to 31 us on 10 to 16 qubits, most of it in the copy; this way 12 to 14.  (A last
// workgroup that finds itself by a ticket and adds the partial sums costs 30 ns per workgroup, one after the other across
// the XCDs: 4 us more at 256 workgroups, 60 at 2048.)
#pragma once
#include "k_common.hpp"

constexpr int RED_THREADS = 256;
constexpr int RED_BLOCKS = 2048;   // room for partial sums; their count depends only on the size and shape

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// block-wide sum of NV values; result valid in thread 0
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV]) {
    __shared__ double red[NV][RED_THREADS / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        v[i] = wave_sum(v[i]);
        if (lane == 0) red[i][wv] = v[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double s = 0.0;
            for (int w = 0; w < RED_THREADS / 64; ++w) s += red[i][w];
            v[i] = s;
        }
    }
}

// the workgroup's share into its slot of `part` (NV per workgroup, host memory)
template <int NV>
__device__ __forceinline__ void put_partial(double (&v)[NV], double *part) {
    block_sum<NV>(v);
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i)
            __hip_atomic_store(part + NV * blockIdx.x + i, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[0..NV) = sums of nblk partials, added like a workgroup would: 256 strided sums, then halves of 64
template <int NV>
inline void add_partials(const double *part, int nblk, double *out) {
    for (int i = 0; i < NV; ++i) {
        double v[RED_THREADS], s = 0.0;
        for (int t = 0; t < RED_THREADS; ++t) v[t] = 0.0;
        for (int b = 0; b < nblk; ++b) v[b % RED_THREADS] += part[NV * b + i];
        for (int w = 0; w < RED_THREADS; w += 64) {
            for (int off = 32; off > 0; off >>= 1)
                for (int l = 0; l < off; ++l) v[w + l] += v[w + l + off];
            s += v[w];
        }
        out[i] = s;
    }
}
