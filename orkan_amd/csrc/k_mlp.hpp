// k_mlp.hpp -- shared by the surrogate's kernels: bf16 and MFMA vector types, GELU and its derivative, and the
// arguments of the fused GEMM epilogues.
#pragma once
#include "k_common.hpp"

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {

enum { EPI_F32 = 0, EPI_BIAS_GELU = 1, EPI_GELU_BWD = 2 };

// erf(x) by Abramowitz & Stegun, Handbook of Mathematical Functions, 7.1.26 (Hastings):
// 1 - (a1 t + ... + a5 t^5) exp(-x^2), t = 1 / (1 + p |x|), |error| <= 1.5e-7, far below the
// bf16 rounding of the activations it feeds; branch-free, unlike a piecewise erff, which
// dominated the GEMM epilogue.
__device__ __forceinline__ float erf_as(float x) {
    const float ax = fabsf(x);
    // hardware reciprocal (1 ulp): the approximation's own error is 1.5e-7
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, ax, 1.0f));
    const float poly =
        t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
    return copysignf(1.0f - poly * __expf(-ax * ax), x);
}
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erf_as(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
    const float cdf = 0.5f * (1.0f + erf_as(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * __expf(-0.5f * x * x);
    return cdf + x * pdf;
}

struct EpiArgs {
    float *c32;          // EPI_F32: fp32 C, ldc
    int ldc;
    const float *bias;   // EPI_BIAS_GELU: bias[N]
    float *pre;          // EPI_BIAS_GELU: pre-activation out (fp32, ldc); EPI_GELU_BWD: pre-activation in
    bf16 *act;           // EPI_BIAS_GELU: gelu(pre) out (bf16, ldc); EPI_GELU_BWD: dPre out (bf16, ldc)
    bf16 *actT;          // act transposed, [N][ldt], or null
    long ldt;
};

// rows row0 .. row0 + 3 of one column: what a lane holds of an MFMA tile per four accumulators, one 8 B store of the
// transposed copy
template <int EPI>
__device__ __forceinline__ void epilogue4(const EpiArgs &ep, long row0, long col, float bias, const float (&v)[4]) {
    bf16x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const long at = (row0 + j) * ep.ldc + col;
        if constexpr (EPI == EPI_F32) {
            ep.c32[at] = v[j];
        } else if constexpr (EPI == EPI_BIAS_GELU) {
            const float z = v[j] + bias;
            if (ep.pre) ep.pre[at] = z;
            o[j] = (bf16)gelu(z);
            ep.act[at] = o[j];
        } else {
            o[j] = (bf16)(v[j] * gelu_grad(ep.pre[at]));
            ep.act[at] = o[j];
        }
    }
    if constexpr (EPI != EPI_F32)
        if (ep.actT) *(bf16x4 *)(ep.actT + col * ep.ldt + row0) = o;
}

}  // namespace
