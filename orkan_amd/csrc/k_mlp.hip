// k_mlp.hip -- BF16 MFMA kernels of the QAOA energy surrogate (an MLP
// 128 -> 512 -> 512 -> 512 -> 1 with GELU): forward, backward and Adam.
//
// The GEMM is C[M x N] = A[M x K] * B[N x K]^T with both operands K-contiguous
// bf16 and fp32 accumulation on v_mfma_f32_32x32x16_bf16 (gfx950).  A 256-thread
// workgroup computes a 128 x 128 tile (2 x 2 waves, each 64 x 64 = 2 x 2 MFMA
// tiles) over K steps of 32, staged through double-buffered LDS.  The epilogue
// is fused: bias + GELU (forward), GELU' (backward), or plain fp32 (weight
// gradients).  Shapes must be multiples of the tile (M, N of 128, K of 32);
// the host pads the batch.
//
// No reference counterpart: this is the learned screening stage on top of the
// simulator.
#include "k_mlp.hpp"

namespace {

constexpr int BM = 128, BN = 128, BK = 32;
constexpr int KP = BK + 8;            // padded LDS row (bf16 elements)
constexpr int GT = 256;               // threads per GEMM workgroup

template <int EPI>
__global__ __launch_bounds__(GT) void gemm_nt_kernel(const bf16 *__restrict__ A, int lda, const bf16 *__restrict__ B,
                                                     int ldb, int K, EpiArgs ep) {
    __shared__ __attribute__((aligned(16))) bf16 As[2][BM * KP];
    __shared__ __attribute__((aligned(16))) bf16 Bs[2][BN * KP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const long m0 = (long)blockIdx.y * BM, n0 = (long)blockIdx.x * BN;
    // global -> register staging: each thread moves 16 bf16 of A and 16 of B per K step
    const int lr = tid >> 1, lk = (tid & 1) * 16;
    const bf16 *ga = A + (m0 + lr) * (long)lda + lk;
    const bf16 *gb = B + (n0 + lr) * (long)ldb + lk;
    uint4 ra0, ra1, rb0, rb1;
#define GEMM_GLOAD(k0)                                  \
    do {                                                \
        ra0 = *(const uint4 *)(ga + (k0));              \
        ra1 = *(const uint4 *)(ga + (k0) + 8);          \
        rb0 = *(const uint4 *)(gb + (k0));              \
        rb1 = *(const uint4 *)(gb + (k0) + 8);          \
    } while (0)
#define GEMM_SSTORE(buf)                                         \
    do {                                                         \
        *(uint4 *)(&As[(buf)][lr * KP + lk]) = ra0;              \
        *(uint4 *)(&As[(buf)][lr * KP + lk + 8]) = ra1;          \
        *(uint4 *)(&Bs[(buf)][lr * KP + lk]) = rb0;              \
        *(uint4 *)(&Bs[(buf)][lr * KP + lk + 8]) = rb1;          \
    } while (0)
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int KT = K / BK;
    GEMM_GLOAD(0);
    GEMM_SSTORE(0);
    __syncthreads();
    const int l32 = lane & 31, lhi = lane >> 5;
    for (int kt = 0; kt < KT; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < KT) GEMM_GLOAD((kt + 1) * BK);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int kk = s * 16 + lhi * 8;
            bf16x8 av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) av[i] = *(const bf16x8 *)(&As[buf][(wm * 64 + i * 32 + l32) * KP + kk]);
#pragma unroll
            for (int j = 0; j < 2; ++j) bv[j] = *(const bf16x8 *)(&Bs[buf][(wn * 64 + j * 32 + l32) * KP + kk]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < KT) GEMM_SSTORE(buf ^ 1);
        __syncthreads();
    }
#undef GEMM_GLOAD
#undef GEMM_SSTORE
    // epilogue: lane holds C[row][col] with col = l32, row = 8 (r / 4) + 4 lhi + (r % 4)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const long col = n0 + wn * 64 + j * 32 + l32;
            const float bias = EPI == EPI_BIAS_GELU ? ep.bias[col] : 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                epilogue4<EPI>(ep, m0 + wm * 64 + i * 32 + 8 * q + 4 * lhi, col, bias,
                               {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]});
        }
}

// ---- 256 x 256 tile variant: 8 waves of 128 x 64 (4 x 2 MFMA tiles each), K steps of 64 ------
// Each operand fragment read from LDS feeds two or four MFMAs; 128 accumulator registers per
// lane leave room for the staging registers without spills, and the 2 waves per SIMD plus the
// 64-deep K step (2048 MFMA cycles per SIMD between barriers) cover the global-load latency of
// the next step.  Used when M, N are multiples of 256 and K of 64.
constexpr int BM2 = 256, BN2 = 256, BK2 = 64, KP2 = BK2 + 8, GT2 = 512;

template <int EPI>
__global__ __launch_bounds__(GT2) void gemm_nt_big_kernel(const bf16 *__restrict__ A, int lda,
                                                          const bf16 *__restrict__ B, int ldb, int K, EpiArgs ep) {
    extern __shared__ __attribute__((aligned(16))) bf16 smem[];
    bf16 *As = smem;                          // [2][BM2 * KP2]
    bf16 *Bs = smem + 2 * BM2 * KP2;          // [2][BN2 * KP2]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;  // 2 x 4 waves: 128 rows x 64 columns each
    const long m0 = (long)blockIdx.y * BM2, n0 = (long)blockIdx.x * BN2;
    // staging: 8 lanes cover the 128 B of one row's K step, a wave 8 rows (fully used cache
    // lines); each thread moves 16 B of rows lr, lr + 64, lr + 128, lr + 192 of A and of B
    const int lr = tid >> 3, lk = (tid & 7) * 8;
    const bf16 *ga = A + (m0 + lr) * (long)lda + lk;
    const bf16 *gb = B + (n0 + lr) * (long)ldb + lk;
    const long sa = 64 * (long)lda, sb = 64 * (long)ldb;
    uint4 ra0, ra1, ra2, ra3, rb0, rb1, rb2, rb3;
#define BIG_GLOAD(k0)                                                                            \
    do {                                                                                         \
        ra0 = *(const uint4 *)(ga + (k0));          ra1 = *(const uint4 *)(ga + sa + (k0));      \
        ra2 = *(const uint4 *)(ga + 2 * sa + (k0)); ra3 = *(const uint4 *)(ga + 3 * sa + (k0));  \
        rb0 = *(const uint4 *)(gb + (k0));          rb1 = *(const uint4 *)(gb + sb + (k0));      \
        rb2 = *(const uint4 *)(gb + 2 * sb + (k0)); rb3 = *(const uint4 *)(gb + 3 * sb + (k0));  \
    } while (0)
#define BIG_SSTORE(buf)                                                                  \
    do {                                                                                 \
        bf16 *pa = As + (buf) * BM2 * KP2 + lr * KP2 + lk;                               \
        bf16 *pb = Bs + (buf) * BN2 * KP2 + lr * KP2 + lk;                               \
        *(uint4 *)(pa) = ra0; *(uint4 *)(pa + 64 * KP2) = ra1;                           \
        *(uint4 *)(pa + 128 * KP2) = ra2; *(uint4 *)(pa + 192 * KP2) = ra3;              \
        *(uint4 *)(pb) = rb0; *(uint4 *)(pb + 64 * KP2) = rb1;                           \
        *(uint4 *)(pb + 128 * KP2) = rb2; *(uint4 *)(pb + 192 * KP2) = rb3;              \
    } while (0)
    f32x16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const int KT = K / BK2;
    BIG_GLOAD(0);
    BIG_SSTORE(0);
    __syncthreads();
    const int l32 = lane & 31, lhi = lane >> 5;
    for (int kt = 0; kt < KT; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < KT) BIG_GLOAD((kt + 1) * BK2);
        const bf16 *as = As + buf * BM2 * KP2 + (wm * 128 + l32) * KP2;
        const bf16 *bs = Bs + buf * BN2 * KP2 + (wn * 64 + l32) * KP2;
#pragma unroll
        for (int s = 0; s < BK2 / 16; ++s) {
            const int kk = s * 16 + lhi * 8;
            bf16x8 av[4], bv[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = *(const bf16x8 *)(as + i * 32 * KP2 + kk);
#pragma unroll
            for (int j = 0; j < 2; ++j) bv[j] = *(const bf16x8 *)(bs + j * 32 * KP2 + kk);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < KT) BIG_SSTORE(buf ^ 1);
        __syncthreads();
    }
#undef BIG_GLOAD
#undef BIG_SSTORE
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const long col = n0 + wn * 64 + j * 32 + l32;
            const float bias = EPI == EPI_BIAS_GELU ? ep.bias[col] : 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                epilogue4<EPI>(ep, m0 + wm * 128 + i * 32 + 8 * q + 4 * lhi, col, bias,
                               {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]});
        }
}
constexpr int BIG_LDS = 2 * (BM2 + BN2) * KP2 * (int)sizeof(bf16);

// ---- 256 x 256 tile, operands streamed into LDS by DMA (global_load_lds), four stages ----------
// Same waves and MFMA tiles as gemm_nt_big_kernel, but K steps of 32 move from global memory
// straight into LDS (no staging registers), three steps ahead of the one being multiplied.  Each
// stage is its own __shared__ array, so the compiler's wait tracking keeps the DMA into one stage
// from blocking reads of another.  A stage row is 64 B (32 bf16); its four 16 B chunks are stored
// XOR-swizzled (position p holds K chunk p ^ ((row >> 2) & 3)), which keeps the 16 rows an MFMA
// operand read touches in distinct banks without padding (a DMA instruction writes 64 contiguous
// 16 B slots, one per lane).
constexpr int BK3 = 32, GT3 = 512;
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 2) & 3); }

template <int EPI>
__global__ __launch_bounds__(GT3) void gemm_nt_dma_kernel(const bf16 *__restrict__ A, int lda,
                                                          const bf16 *__restrict__ B, int ldb, int K, EpiArgs ep) {
    __shared__ __attribute__((aligned(16))) bf16 sa0[BM2 * BK3], sa1[BM2 * BK3], sa2[BM2 * BK3], sa3[BM2 * BK3];
    __shared__ __attribute__((aligned(16))) bf16 sb0[BN2 * BK3], sb1[BN2 * BK3], sb2[BN2 * BK3], sb3[BN2 * BK3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    const long m0 = (long)blockIdx.y * BM2, n0 = (long)blockIdx.x * BN2;
    // DMA: wave w fills rows [32 w, 32 w + 32) of the A and B stage, 16 rows (1 KB) per instruction;
    // lane l lands in row 32 w + 16 i + l / 4 at chunk position l % 4
    const int drow = wave * 32 + (lane >> 2), dp = lane & 3;
    const bf16 *ga0 = A + (m0 + drow) * (long)lda + swz(drow, dp) * 8;
    const bf16 *ga1 = A + (m0 + drow + 16) * (long)lda + swz(drow + 16, dp) * 8;
    const bf16 *gb0 = B + (n0 + drow) * (long)ldb + swz(drow, dp) * 8;
    const bf16 *gb1 = B + (n0 + drow + 16) * (long)ldb + swz(drow + 16, dp) * 8;
    const int dst0 = wave * 32 * BK3, dst1 = (wave * 32 + 16) * BK3;
#define DMA(SA, SB, k0)                                                                         \
    do {                                                                                        \
        __builtin_amdgcn_global_load_lds((const void *)(ga0 + (k0)), (lds_void *)((SA) + dst0), 16, 0, 0); \
        __builtin_amdgcn_global_load_lds((const void *)(ga1 + (k0)), (lds_void *)((SA) + dst1), 16, 0, 0); \
        __builtin_amdgcn_global_load_lds((const void *)(gb0 + (k0)), (lds_void *)((SB) + dst0), 16, 0, 0); \
        __builtin_amdgcn_global_load_lds((const void *)(gb1 + (k0)), (lds_void *)((SB) + dst1), 16, 0, 0); \
    } while (0)
    f32x16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    const int KT = K / BK3;
    const int l32 = lane & 31, lhi = lane >> 5;
    int ra[4], rb[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = wm * 128 + i * 32 + l32;
#pragma unroll
    for (int j = 0; j < 2; ++j) rb[j] = wn * 64 + j * 32 + l32;
#define MMA(SA, SB)                                                                                    \
    do {                                                                                               \
        _Pragma("unroll") for (int s = 0; s < BK3 / 16; ++s) {                                         \
            const int c = 2 * s + lhi;                                                                 \
            bf16x8 av[4], bv[2];                                                                       \
            _Pragma("unroll") for (int i = 0; i < 4; ++i)                                              \
                av[i] = *(const bf16x8 *)((SA) + ra[i] * BK3 + swz(ra[i], c) * 8);                     \
            _Pragma("unroll") for (int j = 0; j < 2; ++j)                                              \
                bv[j] = *(const bf16x8 *)((SB) + rb[j] * BK3 + swz(rb[j], c) * 8);                     \
            _Pragma("unroll") for (int i = 0; i < 4; ++i)                                              \
                _Pragma("unroll") for (int j = 0; j < 2; ++j)                                          \
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i], bv[j], acc[i][j], 0, 0, 0); \
        }                                                                                              \
    } while (0)
    // stage kc sits in (CA, CB).  Every step issues one stage of DMA (past the end of K it reloads
    // the last stage into the slot nobody reads again), so at step kc the stages kc + 1 and kc + 2
    // are the only later ones in flight: wait until this wave has at most those 8 instructions
    // outstanding, barrier (every wave's DMA of stage kc landed and every wave is done with stage
    // kc - 1: its LDS reads fed MFMAs issued before the barrier, and the scheduling barrier keeps
    // them there), refill the slot of stage kc - 1 with stage kc + 3, multiply stage kc.
    // s_waitcnt immediate: vmcnt in bits 3:0, expcnt 6:4 = 7 and lgkmcnt 11:8 = 15 (no wait).  The
    // acquire fence (LDS only) keeps the stage reads below the barrier without the vmcnt(0) that a
    // release fence adds for DMA still in flight.
#define STEP(CA, CB, NA, NB, kc)                                                                       \
    do {                                                                                               \
        __builtin_amdgcn_s_waitcnt(0x0F70 | 8);                                                        \
        __builtin_amdgcn_s_barrier();                                                                  \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");                                \
        DMA(NA, NB, ((kc) + 3 < KT ? (kc) + 3 : KT - 1) * BK3);                                        \
        MMA(CA, CB);                                                                                   \
        __builtin_amdgcn_sched_barrier(0);                                                             \
    } while (0)
    // K is a multiple of 4 BK3 (the host checks), so the loop body runs whole
    DMA(sa0, sb0, 0);
    DMA(sa1, sb1, BK3);
    DMA(sa2, sb2, 2 * BK3);
    for (int kt = 0; kt < KT; kt += 4) {
        STEP(sa0, sb0, sa3, sb3, kt);
        STEP(sa1, sb1, sa0, sb0, kt + 1);
        STEP(sa2, sb2, sa1, sb1, kt + 2);
        STEP(sa3, sb3, sa2, sb2, kt + 3);
    }
    // no DMA may still be writing this workgroup's LDS when it ends
    __builtin_amdgcn_s_waitcnt(0x0F70);
#undef STEP
#undef MMA
#undef DMA
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const long col = n0 + wn * 64 + j * 32 + l32;
            const float bias = EPI == EPI_BIAS_GELU ? ep.bias[col] : 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                epilogue4<EPI>(ep, m0 + wm * 128 + i * 32 + 8 * q + 4 * lhi, col, bias,
                               {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]});
        }
}


// ---- small kernels -----------------------------------------------------------------------------
// y[m] = sum_k h[m][k] w[k] + b   (one wave per row); optional loss gradient and
// per-row squared error (target given)
__global__ __launch_bounds__(256) void head_forward_kernel(const bf16 *__restrict__ h, const float *__restrict__ w, float b,
                                                          int M, int K, float *__restrict__ y,
                                                          const float *__restrict__ target, float *__restrict__ dy,
                                                          float *__restrict__ sqerr, int valid, float scale) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= M) return;
    float s = 0.0f;
    if (K % 8 == 0 && ((uintptr_t)h & 15) == 0 && ((uintptr_t)w & 15) == 0) {
        // 16 B per lane: one load instruction covers 512 activations of the row
        for (int k = lane * 8; k < K; k += 512) {
            const bf16x8 hv = *(const bf16x8 *)(h + (long)row * K + k);
            const float4 w0 = *(const float4 *)(w + k), w1 = *(const float4 *)(w + k + 4);
            s += (float)hv[0] * w0.x + (float)hv[1] * w0.y + (float)hv[2] * w0.z + (float)hv[3] * w0.w +
                 (float)hv[4] * w1.x + (float)hv[5] * w1.y + (float)hv[6] * w1.z + (float)hv[7] * w1.w;
        }
    } else {
        for (int k = lane; k < K; k += 64) s += (float)h[(long)row * K + k] * w[k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0 && (target || row < valid)) {   // forward only: no writes past the valid rows
        const float v = s + b;
        y[row] = v;
        if (target) {
            const float e = (row < valid) ? (v - target[row]) : 0.0f;
            dy[row] = 2.0f * e * scale;
            sqerr[row] = e * e;
        }
    }
}

// X[r] = [gf (ng floats), angles[r0 + r] (na floats)] as fp32 rows of width ng + na
// ---- first layer for screening ------------------------------------------------------------
// Every candidate row of one graph shares the ng graph features, so their share
// of layer 1 is computed once: u[j] = sum_{k<ng} bf16(gf[k]) W[k][j].  A row's
// pre-activation is then (u[j] + sum_k bf16(a[r][k]) W[ng+k][j]) + b[j]: the same
// bf16 products as the GEMM over the assembled row, summed in fp32 in another
// order.  W is the bf16 [K][N] copy of the layer.
__global__ void first_layer_graph_kernel(const float *__restrict__ gf, int ng, const bf16 *__restrict__ w, int N,
                                         float *__restrict__ u) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= N) return;
    float s = 0.0f;
    for (int k = 0; k < ng; ++k) s += (float)(bf16)gf[k] * (float)w[(long)k * N + j];
    u[j] = s;
}

// act[r][j] = gelu(pre) for rows [0, rows) of the chunk starting at candidate r0,
// zero for the padding rows [rows, Mp); four consecutive columns per thread
// (one 8-byte weight load per angle, one 8-byte store).  NA > 0 fixes the angle
// count at compile time so that all loads of a row issue together.
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
template <int NA>
__global__ void first_layer_rows_kernel(const float *__restrict__ angles, int na_rt, long r0, int rows, int Mp,
                                        const float *__restrict__ u, const bf16 *__restrict__ wa,
                                        const float *__restrict__ bias, int N, bf16 *__restrict__ act) {
    const int na = NA > 0 ? NA : na_rt;
    // 8 outputs per thread: 16 B weight loads and one 16 B store
    const unsigned nq = (unsigned)(N >> 3);
    const unsigned total = (unsigned)Mp * nq;
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < total; i += gridDim.x * 256u) {
        const unsigned r = i / nq;
        const int j = (int)(i - r * nq) * 8;
        bf16x8 out;
        if ((int)r < rows) {
            const float4 u0 = *(const float4 *)(u + j), u1 = *(const float4 *)(u + j + 4);
            float z[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
            const float *a = angles + (r0 + (long)r) * na;
#pragma unroll 8
            for (int k = 0; k < na; ++k) {
                const float ak = (float)(bf16)a[k];
                const bf16x8 w = *(const bf16x8 *)(wa + (long)k * N + j);
#pragma unroll
                for (int t = 0; t < 8; ++t) z[t] += ak * (float)w[t];
            }
            const float4 b0 = *(const float4 *)(bias + j), b1 = *(const float4 *)(bias + j + 4);
            const float bb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
            for (int t = 0; t < 8; ++t) out[t] = (bf16)gelu(z[t] + bb[t]);
        } else {
#pragma unroll
            for (int t = 0; t < 8; ++t) out[t] = (bf16)0.0f;
        }
        *(bf16x8 *)(act + (long)r * N + j) = out;
    }
}

// ---- top-k selection (radix select on order-preserving float keys) ---------------------------
__device__ __forceinline__ unsigned fkey(float f) {
    const unsigned u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

struct TopkState {
    unsigned prefix, mask;   // bits of the k-th largest key fixed so far
    long need;               // elements still to take among those matching the prefix
    unsigned hist[256];
    unsigned n_gt, n_eq;     // compaction counters
};

__global__ __launch_bounds__(256) void topk_hist_kernel(const float *__restrict__ y, long n, TopkState *st, int shift) {
    __shared__ unsigned h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const unsigned prefix = st->prefix, mask = st->mask;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const unsigned key = fkey(y[i]);
        if ((key & mask) == prefix) atomicAdd(&h[(key >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&st->hist[threadIdx.x], h[threadIdx.x]);
}

// the k-th largest key has the digit where the running count, from the largest digit down, reaches `need`: an inclusive
// scan over the bins in descending order, one bin per thread (2.5 us; one thread walking the 256 bins took 9)
__global__ __launch_bounds__(256) void topk_select_kernel(TopkState *st, int shift) {
    __shared__ long scan[256];
    const int t = threadIdx.x;
    const long cnt = st->hist[255 - t], need = st->need;
    scan[t] = cnt;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const long v = t >= off ? scan[t - off] : 0;
        __syncthreads();
        scan[t] += v;
        __syncthreads();
    }
    st->hist[255 - t] = 0;
    if (scan[t] >= need && scan[t] - cnt < need) {   // one thread: the counts add up to at least `need`
        st->need = need - (scan[t] - cnt);
        st->prefix |= (unsigned)(255 - t) << shift;
        st->mask |= 255u << shift;
    }
}

__global__ void topk_init_kernel(TopkState *st, long k) {
    if (threadIdx.x != 0) return;
    st->prefix = 0;
    st->mask = 0;
    st->need = k;
    st->n_gt = 0;
    st->n_eq = 0;
    for (int b = 0; b < 256; ++b) st->hist[b] = 0;
}

// keys above the threshold all go out; `need` of the keys equal to it (in the
// order the atomics hand out slots -- ties are re-ordered by index on the host)
__global__ __launch_bounds__(256) void topk_compact_kernel(const float *__restrict__ y, long n, TopkState *st,
                                                          int k, int *__restrict__ out) {
    const unsigned T = st->prefix;
    const long need = st->need;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        const unsigned key = fkey(y[i]);
        if (key > T) {
            const unsigned s = atomicAdd(&st->n_gt, 1u);
            if (s < (unsigned)k) out[s] = (int)i;
        } else if (key == T) {
            const unsigned s = atomicAdd(&st->n_eq, 1u);
            if ((long)s < need) out[k - 1 - s] = (int)i;
        }
    }
}

unsigned g1(long n) {
    long g = (n + 255) / 256;
    if (g > 65536) g = 65536;
    if (g < 1) g = 1;
    return (unsigned)g;
}

}  // namespace

// ---- C ABI ------------------------------------------------------------------------------------
constexpr int kGemmVariant = 2;
static int g_gemm_big = kGemmVariant;   // 256 x 256 tiles where the shape allows: 1 register-staged, 2 DMA-staged
extern "C" void ork_mlp_gemm_reset(void) { g_gemm_big = kGemmVariant; }

extern "C" int ork_mlp_gemm_select(int variant) {
    if (variant < 0 || variant > 2) return (int)hipErrorInvalidValue;
    g_gemm_big = variant;
    return 0;
}

extern "C" int ork_mlp_gemm_mid(void *stream, int epi, const void *A, int lda, const void *B, int ldb, int M, int N,
                                int K, float *c32, int ldc, const float *bias, float *pre, void *act, void *actT,
                                long ldt);

// epi: 0 fp32 C, 1 bias+GELU, 2 GELU backward; actT: the bf16 result transposed as well ([N][ldt]), or null
extern "C" int ork_mlp_gemm(void *stream, int epi, const void *A, int lda, const void *B, int ldb, int M, int N, int K,
                            float *c32, int ldc, const float *bias, float *pre, void *act, void *actT, long ldt) {
    if (M % BM || N % BN || K % BK || M <= 0 || N <= 0 || K <= 0 || ldt % 4 || ((uintptr_t)actT & 7))
        return (int)hipErrorInvalidValue;
    EpiArgs ep{c32, ldc, bias, pre, (bf16 *)act, (bf16 *)actT, ldt};
    hipStream_t st = (hipStream_t)stream;
    const bf16 *a = (const bf16 *)A, *b = (const bf16 *)B;
    // the DMA moves 16 B per lane: rows of both operands must start on 16 B boundaries
    const bool aligned16 = lda % 8 == 0 && ldb % 8 == 0 && ((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0;
    if (g_gemm_big == 2 && aligned16 && M % BM2 == 0 && N % BN2 == 0 && K % (4 * BK3) == 0 &&
        (long)(M / BM2) * (N / BN2) >= 256) {
        dim3 grid3(N / BN2, M / BM2);
        switch (epi) {
        case EPI_F32: gemm_nt_dma_kernel<EPI_F32><<<grid3, GT3, 0, st>>>(a, lda, b, ldb, K, ep); break;
        case EPI_BIAS_GELU: gemm_nt_dma_kernel<EPI_BIAS_GELU><<<grid3, GT3, 0, st>>>(a, lda, b, ldb, K, ep); break;
        case EPI_GELU_BWD: gemm_nt_dma_kernel<EPI_GELU_BWD><<<grid3, GT3, 0, st>>>(a, lda, b, ldb, K, ep); break;
        default: return (int)hipErrorInvalidValue;
        }
        ORK_LAUNCH_CHECK();
        return 0;
    }
    if (g_gemm_big == 1 && M % BM2 == 0 && N % BN2 == 0 && K % BK2 == 0) {
        dim3 grid2(N / BN2, M / BM2);
        switch (epi) {
        case EPI_F32: gemm_nt_big_kernel<EPI_F32><<<grid2, GT2, BIG_LDS, st>>>(a, lda, b, ldb, K, ep); break;
        case EPI_BIAS_GELU: gemm_nt_big_kernel<EPI_BIAS_GELU><<<grid2, GT2, BIG_LDS, st>>>(a, lda, b, ldb, K, ep); break;
        case EPI_GELU_BWD: gemm_nt_big_kernel<EPI_GELU_BWD><<<grid2, GT2, BIG_LDS, st>>>(a, lda, b, ldb, K, ep); break;
        default: return (int)hipErrorInvalidValue;
        }
        ORK_LAUNCH_CHECK();
        return 0;
    }
    // Up to one 128 x 64 tile per CU: those, twice the workgroups of 128 x 128 and the operands by DMA.  A second round of
    // them costs more than the better reuse of 128 x 128 saves.  Three forward layers from 128 to H, H and H wide with
    // 128 x 64, 128 x 128 and (where it divides) 256 x 256 tiles, at `tiles` of 128 x 128:
    //   H 512, tiles 128: 46 us, 64, 108    188: 66.7, 65.6, -    316: 87, 75, -    768: 149, 102, 123    2044: 357, 213, -
    //   H 128, tiles 128: 46 us, 58, -    192: 61.2, 59.3, -    512: 104, 82, -
    //   H 1024, tiles 128: 55 us, 79, 124    256: 81.9, 82.9, 126    1024: -, 172, 130    2040: 461, 275, -
    if (g_gemm_big == 2 && aligned16 && (long)(M / BM) * (N / BN) <= 128)
        return ork_mlp_gemm_mid(stream, epi, A, lda, B, ldb, M, N, K, c32, ldc, bias, pre, act, actT, ldt);
    dim3 grid(N / BN, M / BM);
    switch (epi) {
    case EPI_F32: gemm_nt_kernel<EPI_F32><<<grid, GT, 0, st>>>(a, lda, b, ldb, K, ep); break;
    case EPI_BIAS_GELU: gemm_nt_kernel<EPI_BIAS_GELU><<<grid, GT, 0, st>>>(a, lda, b, ldb, K, ep); break;
    case EPI_GELU_BWD: gemm_nt_kernel<EPI_GELU_BWD><<<grid, GT, 0, st>>>(a, lda, b, ldb, K, ep); break;
    default: return (int)hipErrorInvalidValue;
    }
    ORK_LAUNCH_CHECK();
    return 0;
}

extern "C" int ork_mlp_head_forward(void *stream, const void *h, const float *w, float b, int M, int K, float *y,
                                    const float *target, float *dy, float *sqerr, int valid, float scale) {
    head_forward_kernel<<<(M + 3) / 4, 256, 0, (hipStream_t)stream>>>((const bf16 *)h, w, b, M, K, y, target, dy,
                                                                      sqerr, valid, scale);
    ORK_LAUNCH_CHECK();
    return 0;
}

extern "C" int ork_mlp_first_layer_graph(void *stream, const float *gf, int ng, const void *w, int N, float *u) {
    first_layer_graph_kernel<<<(N + 255) / 256, 256, 0, (hipStream_t)stream>>>(gf, ng, (const bf16 *)w, N, u);
    ORK_LAUNCH_CHECK();
    return 0;
}

extern "C" int ork_mlp_first_layer_rows(void *stream, const float *angles, int na, long r0, int rows, int Mp,
                                        const float *u, const void *wa, const float *bias, int N, void *act) {
    if (N % 8 || (long)Mp * (N / 8) >= (1L << 32)) return (int)hipErrorInvalidValue;
    const unsigned grid = g1((long)Mp * (N / 8));
    if (na == 8)
        first_layer_rows_kernel<8><<<grid, 256, 0, (hipStream_t)stream>>>(angles, na, r0, rows, Mp, u,
                                                                         (const bf16 *)wa, bias, N, (bf16 *)act);
    else
        first_layer_rows_kernel<0><<<grid, 256, 0, (hipStream_t)stream>>>(angles, na, r0, rows, Mp, u,
                                                                         (const bf16 *)wa, bias, N, (bf16 *)act);
    ORK_LAUNCH_CHECK();
    return 0;
}

// indices of the k largest of y_dev[0..n) into idx_dev[0..k) (unordered); st_dev: scratch of
// ork_topk_state_bytes() bytes
extern "C" unsigned long ork_topk_state_bytes(void) { return sizeof(TopkState); }

__global__ void gather_f32_kernel(const float *__restrict__ y, const int *__restrict__ idx, float *__restrict__ out,
                                  int k) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < k) out[i] = y[idx[i]];
}

extern "C" int ork_topk(void *stream, const float *y, long n, int k, int *idx, float *vals, void *st_dev) {
    if (k <= 0 || (long)k > n) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    TopkState *ts = (TopkState *)st_dev;
    long g = (n + 255) / 256;
    if (g > 2048) g = 2048;
    topk_init_kernel<<<1, 64, 0, st>>>(ts, k);
    ORK_LAUNCH_CHECK();
    for (int shift = 24; shift >= 0; shift -= 8) {
        topk_hist_kernel<<<(unsigned)g, 256, 0, st>>>(y, n, ts, shift);
        ORK_LAUNCH_CHECK();
        topk_select_kernel<<<1, 256, 0, st>>>(ts, shift);
        ORK_LAUNCH_CHECK();
    }
    topk_compact_kernel<<<(unsigned)g, 256, 0, st>>>(y, n, ts, k, idx);
    ORK_LAUNCH_CHECK();
    gather_f32_kernel<<<(k + 255) / 256, 256, 0, st>>>(y, idx, vals, k);
    ORK_LAUNCH_CHECK();
    return 0;
}
