// k_screen.hip -- the screening forward of the surrogate in one kernel: a workgroup takes 64 candidates through every
// layer, the activations staying in LDS, and writes 64 predictions.
//
// Layer by layer through memory, 10^6 candidates of a 512-wide network wrote and read 1 GB of bf16 activations per
// layer, and each layer's GEMM ended in an epilogue (bias + GELU: two transcendental and 15 plain instructions per
// value) that no matrix work covered.  Here a 64 x H tile of bf16 activations (64 KB for H = 512) is rewritten in place
// by each layer; two workgroups fit a CU, so one's GELU runs while the other's waves feed the matrix cores, and memory
// sees the angles, the predictions and, from L2, the weights (1 MB per 64 candidates for two layers of 512).
//
// The products run transposed, D[n][m] = W[n] . act[m]: a lane then holds four consecutive columns n of one candidate
// m, one 8 B LDS store.  Weight fragments come straight from global memory, packed so that a wave reads 1 KB runs, four
// K steps ahead (across the layers' ends too, under the GELU); activation fragments come from LDS rows whose 16 B chunks
// are XOR-swizzled by the row.  Every value sees the same operations in the same order as in the layer kernels, the
// MFMA chain over K included, so predictions keep their bits.
//
// Measured on 1,000,003 candidates, 128 -> 512 -> 512 -> 512 -> 1: 1.53 ms, 690 TFLOP/s, against 3.1 ms layer by layer
// (GEMMs 74 us per 65536 rows and layer, layer 1 45 us, head 13 us).  Bound by the matrix work and the GELUs together:
// with the GELUs left out the kernel takes 1.13 ms, with the weight loads left out as well 0.95; 1536 GELUs per candidate,
// 6 per thread of the workgroup, add up to 1 ms of vector issue.  Wave priorities and a staggered start of a CU's two workgroups changed
// nothing (1.53-1.57 ms).
#include "k_mlp.hpp"

namespace {

constexpr int SC_ROWS = 64, SC_THREADS = 256, SC_MAX = 3, SC_NA = 8;

struct ScreenArgs {
    const float *angles;            // [ncand][8]
    long ncand;
    const float *u;                 // [H] the graph features' share of layer 1
    const bf16 *wa;                 // [8][H] layer-1 rows of the angles
    const bf16 *wpk[SC_MAX];        // packed weights of the layers after the first
    const float *bias[SC_MAX + 1];  // per layer [H]
    int nl;
    const float *w_out;             // [H]
    float b_out;
    float *y;
};

template <int H>
__global__ __launch_bounds__(SC_THREADS, 2) void screen_kernel(ScreenArgs a) {
    constexpr int CPR = H / 8;               // 16 B chunks per row
    constexpr int NT = H / 4 / 32;           // 32-column tiles per wave
    constexpr int KS = H / 16;               // K steps
    constexpr int PF = 4;                    // weight steps in flight
    __shared__ __attribute__((aligned(16))) bf16 act[SC_ROWS * H];
    __shared__ float ang[SC_ROWS][SC_NA];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, lhi = lane >> 5;
    const long r0 = (long)blockIdx.x * SC_ROWS;

    // packed fragment (tile t, step s): 64 lanes x 8 values at ((t KS + s) 64 + lane) 8
    const auto frag = [&](const bf16 *w, int j, int s) {
        return *(const bf16x8 *)(w + (((long)(wave * NT + j) * KS + s) * 64 + lane) * 8);
    };
    bf16x8 w[PF][NT];
    const auto prefetch = [&](const bf16 *p) {
#pragma unroll
        for (int s = 0; s < PF; ++s)
#pragma unroll
            for (int j = 0; j < NT; ++j) w[s][j] = frag(p, j, s);
    };
    if (a.nl > 1) prefetch(a.wpk[0]);

    // ---- layer 1: pre = (u + sum_k bf16(angle_k) W[k]) + b, 8 columns per thread, rows one after the other ----
    for (int i = tid; i < SC_ROWS * SC_NA; i += SC_THREADS) {
        const long at = r0 * SC_NA + i;
        ang[i / SC_NA][i % SC_NA] = at < a.ncand * SC_NA ? (float)(bf16)a.angles[at] : 0.0f;
    }
    __syncthreads();
    {
        constexpr int GROUPS = SC_THREADS / CPR;     // rows in flight: 4 (H = 512), 8, 16
        const int c = tid % CPR, g = tid / CPR, j = c * 8;
        float uu[8], bb[8];
        bf16x8 wk[SC_NA];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            uu[t] = a.u[j + t];
            bb[t] = a.bias[0][j + t];
        }
#pragma unroll
        for (int k = 0; k < SC_NA; ++k) wk[k] = *(const bf16x8 *)(a.wa + (long)k * H + j);
#pragma unroll 1
        for (int r = g; r < SC_ROWS; r += GROUPS) {
            float z[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) z[t] = uu[t];
#pragma unroll
            for (int k = 0; k < SC_NA; ++k) {
                const float ak = ang[r][k];
#pragma unroll
                for (int t = 0; t < 8; ++t) z[t] = fmaf(ak, (float)wk[k][t], z[t]);
            }
            bf16x8 o;
#pragma unroll
            for (int t = 0; t < 8; ++t) o[t] = (bf16)gelu(z[t] + bb[t]);
            *(bf16x8 *)(act + r * H + (c ^ (r & 7)) * 8) = o;
        }
    }
    __syncthreads();

    // ---- the other layers ----
    const int sw = l32 & 7;     // rows l32 and l32 + 32 swizzle alike
    for (int l = 1; l < a.nl; ++l) {
        const bf16 *wp = a.wpk[l - 1];
        f32x16 acc[NT][2];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;
#pragma unroll 1
        for (int s0 = 0; s0 < KS; s0 += PF) {
#pragma unroll
            for (int s = 0; s < PF; ++s) {
                const int ch = (2 * (s0 + s) + lhi) ^ sw;
                const bf16x8 m0 = *(const bf16x8 *)(act + l32 * H + ch * 8);
                const bf16x8 m1 = *(const bf16x8 *)(act + (l32 + 32) * H + ch * 8);
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    acc[j][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s][j], m0, acc[j][0], 0, 0, 0);
                    acc[j][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s][j], m1, acc[j][1], 0, 0, 0);
                }
                // this step's registers take the step PF further on (in the last round: the last step again)
                const int sn = s0 + PF + s < KS ? s0 + PF + s : KS - 1;
#pragma unroll
                for (int j = 0; j < NT; ++j) w[s][j] = frag(wp, j, sn);
            }
        }
        if (l + 1 < a.nl) prefetch(a.wpk[l]);
        __syncthreads();        // every wave has read the old activations
        const float *__restrict__ bias = a.bias[l];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // lane: candidate m = l32 (+ 32), columns n0 .. n0 + 3
                const int n0 = (wave * NT + j) * 32 + 8 * q + 4 * lhi;
                const float4 b = *(const float4 *)(bias + n0);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    bf16x4 o;
                    o[0] = (bf16)gelu(acc[j][i][4 * q] + b.x);
                    o[1] = (bf16)gelu(acc[j][i][4 * q + 1] + b.y);
                    o[2] = (bf16)gelu(acc[j][i][4 * q + 2] + b.z);
                    o[3] = (bf16)gelu(acc[j][i][4 * q + 3] + b.w);
                    *(bf16x4 *)(act + (l32 + 32 * i) * H + (((n0 >> 3) ^ sw) * 8) + (n0 & 7)) = o;
                }
            }
        __syncthreads();
    }

    // ---- head: one wave per row, lane k owns columns 8 k .. 8 k + 7 ----
    float4 w0 = {0.0f, 0.0f, 0.0f, 0.0f}, w1 = w0;
    if (lane < CPR) {
        w0 = *(const float4 *)(a.w_out + lane * 8);
        w1 = *(const float4 *)(a.w_out + lane * 8 + 4);
    }
#pragma unroll 4
    for (int rr = 0; rr < SC_ROWS / 4; ++rr) {
        const int r = wave * (SC_ROWS / 4) + rr;
        float s = 0.0f;
        if (lane < CPR) {
            const bf16x8 h = *(const bf16x8 *)(act + r * H + (lane ^ (r & 7)) * 8);
            float t = (float)h[1] * w0.y;
            t = fmaf(w0.x, (float)h[0], t);
            t = fmaf(w0.z, (float)h[2], t);
            t = fmaf(w0.w, (float)h[3], t);
            t = fmaf(w1.x, (float)h[4], t);
            t = fmaf(w1.y, (float)h[5], t);
            t = fmaf(w1.z, (float)h[6], t);
            t = fmaf(w1.w, (float)h[7], t);
            s += t;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if (lane == 0 && r0 + r < a.ncand) a.y[r0 + r] = s + a.b_out;
    }
}

// Per call: the graph features' share of layer 1, u[j] = sum_k bf16(gf[k]) W[k][j] (k ascending), and the later layers'
// weights [N][K] in fragment order (lane l of tile t, step s: row 32 t + l % 32, columns 16 s + 8 (l / 32) .. + 7).
struct PrepArgs {
    const float *gf;
    int ng;
    const bf16 *w0;             // [K][H] layer-1 weights
    float *u;
    const bf16 *wt[SC_MAX];     // [H][H], K-contiguous
    bf16 *wpk[SC_MAX];
    int H, ublocks;
};

__global__ __launch_bounds__(64) void screen_prepare_kernel(PrepArgs p) {
    if ((int)blockIdx.x < p.ublocks) {
        const int j = blockIdx.x * 64 + threadIdx.x;
        float s = 0.0f;
#pragma unroll 24
        for (int k = 0; k < p.ng; ++k) s = fmaf((float)(bf16)p.gf[k], (float)p.w0[(long)k * p.H + j], s);
        p.u[j] = s;
        return;
    }
    const int KS = p.H / 16, per = p.H / 32 * KS;      // fragments per layer
    const int f = (int)blockIdx.x - p.ublocks, l = f / per, t = f % per / KS, s = f % KS, lane = threadIdx.x;
    const bf16x8 v = *(const bf16x8 *)(p.wt[l] + (long)(t * 32 + (lane & 31)) * p.H + s * 16 + (lane >> 5) * 8);
    *(bf16x8 *)(p.wpk[l] + ((long)(f % per) * 64 + lane) * 8) = v;
}

}  // namespace

// shapes the fused forward takes: 8 angles, a hidden width of 128, 256 or 512
extern "C" int ork_mlp_screen_ok(int na, int hidden, int nl) {
    return na == SC_NA && (hidden == 128 || hidden == 256 || hidden == 512) && nl >= 1 && nl <= SC_MAX + 1;
}

// gf: ng graph features (device); w0: layer-1 bf16 [ng + 8][H]; wt[l]: bf16 [H][H] of layer l + 1 (K-contiguous); wpk: (nl -
// 1) x H x H bf16 scratch; u: H floats scratch; y: ncand predictions
extern "C" int ork_mlp_screen(void *stream, const float *gf, int ng, const void *w0, const void *const *wt, void *wpk,
                              float *u, const float *const *bias, int nl, int H, const float *w_out, float b_out,
                              const float *angles, long ncand, float *y) {
    if (!ork_mlp_screen_ok(SC_NA, H, nl) || ng <= 0 || ncand < 0) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    PrepArgs p{};
    ScreenArgs a{};
    p.gf = gf;
    p.ng = ng;
    p.w0 = (const bf16 *)w0;
    p.u = u;
    p.H = H;
    p.ublocks = H / 64;
    for (int l = 0; l + 1 < nl; ++l) {
        p.wt[l] = (const bf16 *)wt[l];
        p.wpk[l] = (bf16 *)wpk + (long)l * H * H;
        a.wpk[l] = p.wpk[l];
    }
    screen_prepare_kernel<<<p.ublocks + (nl - 1) * (H / 32) * (H / 16), 64, 0, st>>>(p);
    ORK_LAUNCH_CHECK();
    for (int l = 0; l < nl; ++l) a.bias[l] = bias[l];
    a.u = u;
    a.wa = (const bf16 *)w0 + (long)ng * H;
    a.nl = nl;
    a.w_out = w_out;
    a.b_out = b_out;
    const long most = 1L << 30;     // candidates per launch
    for (long r = 0; r < ncand; r += most) {
        a.angles = angles + r * SC_NA;
        a.ncand = ncand - r < most ? ncand - r : most;
        a.y = y + r;
        const unsigned grid = (unsigned)((a.ncand + SC_ROWS - 1) / SC_ROWS);
        if (H == 512) screen_kernel<512><<<grid, SC_THREADS, 0, st>>>(a);
        else if (H == 256) screen_kernel<256><<<grid, SC_THREADS, 0, st>>>(a);
        else screen_kernel<128><<<grid, SC_THREADS, 0, st>>>(a);
        ORK_LAUNCH_CHECK();
    }
    return 0;
}
