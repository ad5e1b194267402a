// k_train.hip -- the surrogate's training step at its own sizes: a batch of a few thousand rows through layers a few
// hundred wide.  Each product of the step is a fraction of a chip's work, so the kernels here are shaped for enough
// workgroups and few launches: a GEMM on 128 x 64 tiles whose epilogue also writes the transposed operand the weight
// gradients need, every layer's weight gradient in one launch, and one launch each for all column sums and for Adam.
//
// Every sum keeps a fixed order (the MFMA chain over K, then slices, chunks or lanes in ascending order), so results
// do not depend on the grid.
//
// Measured on batches of 4096 rows through 128 -> 512 -> 512 -> 512 -> 1: 118 us of kernels per step (350 us when each
// layer and operand had a launch of its own).
#include "k_mlp.hpp"

namespace {

// ---- GEMM C[M x N] = A[M x K] B[N x K]^T on 128 x 64 tiles -----------------------------------------
// For products with too few 256 x 256 tiles to fill the chip (4096 x 512 x 512 has 32 of them for 256 CUs, and 256
// tiles of this size).  Four waves of 64 x 32; K steps of 64 move by DMA (global_load_lds) into four LDS stages, three
// steps ahead: at these K (128 to 512) nearly the whole operand panel is in flight at once, and a step's latency is
// paid once, not once per step.  Each stage is its own __shared__ array (the compiler's wait tracking is per array).
// A stage row is 128 B, its eight 16 B chunks XOR-swizzled by the row (position p holds chunk p ^ (row & 7)), so the
// 8 lanes of an LDS read phase touch distinct banks.
// Batch 4096, hidden 512: 10.7 us per forward layer, 13.7 us per backward one (28 us each on 256 x 256 tiles); what is
// left is latency: the first DMA, and an epilogue of 16-20 MB (fp32 pre-activations, both bf16 copies).
constexpr int MM = 128, MN = 64, MK = 64, MT = 256;
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ int swz8(int row, int chunk) { return chunk ^ (row & 7); }

template <int EPI>
__global__ __launch_bounds__(MT) void gemm_nt_mid_kernel(const bf16 *__restrict__ A, int lda,
                                                         const bf16 *__restrict__ B, int ldb, int K, EpiArgs ep, int ntn) {
    __shared__ __attribute__((aligned(16))) bf16 sa0[MM * MK], sa1[MM * MK], sa2[MM * MK], sa3[MM * MK];
    __shared__ __attribute__((aligned(16))) bf16 sb0[MN * MK], sb1[MN * MK], sb2[MN * MK], sb3[MN * MK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    // workgroups go round-robin over the 8 XCDs: give each XCD a contiguous run of row panels with all their columns,
    // so that an A panel is fetched into one XCD's L2 only
    unsigned t = blockIdx.x;
    if ((gridDim.x & 7) == 0) t = (t & 7) * (gridDim.x >> 3) + (t >> 3);
    const long m0 = (long)(t / (unsigned)ntn) * MM, n0 = (long)(t % (unsigned)ntn) * MN;
    // DMA: one instruction fills 8 rows (64 lanes x 16 B); wave w fills A rows 32 w .. + 31 and B rows 16 w .. + 15.
    // Lane l lands in row l / 8 of the 8 at chunk position l % 8, which holds chunk (l % 8) ^ (row & 7).
    const int drow = lane >> 3, dchunk = swz8(drow, lane & 7);
    const bf16 *ga[4], *gb[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) ga[i] = A + (m0 + wave * 32 + i * 8 + drow) * (long)lda;
#pragma unroll
    for (int i = 0; i < 2; ++i) gb[i] = B + (n0 + wave * 16 + i * 8 + drow) * (long)ldb;
    const int KT = (K + MK - 1) / MK;
    // K is a multiple of 32: in a half last step the lanes of the missing half load the half that is there again
#define DMA(SA, SB, kc)                                                                                             \
    do {                                                                                                            \
        int k_ = (kc) * MK + dchunk * 8;                                                                            \
        if (k_ >= K) k_ -= 32;                                                                                      \
        _Pragma("unroll") for (int i = 0; i < 4; ++i) __builtin_amdgcn_global_load_lds(                             \
            (const void *)(ga[i] + k_), (lds_void *)((SA) + (wave * 32 + i * 8) * MK), 16, 0, 0);                   \
        _Pragma("unroll") for (int i = 0; i < 2; ++i) __builtin_amdgcn_global_load_lds(                             \
            (const void *)(gb[i] + k_), (lds_void *)((SB) + (wave * 16 + i * 8) * MK), 16, 0, 0);                   \
    } while (0)
    f32x16 acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    const int l32 = lane & 31, lhi = lane >> 5;
    const int ra0 = wm * 64 + l32, rb0 = wn * 32 + l32;
    const int swza = ra0 & 7, swzb = rb0 & 7;   // rows ra0 and ra0 + 32 swizzle alike
#define MMA(SA, SB, kc)                                                                                             \
    do {                                                                                                            \
        const int ns_ = (kc) * MK + MK <= K ? 4 : 2;                                                                \
        _Pragma("unroll") for (int s = 0; s < 4; ++s) {                                                             \
            if (s >= ns_) break;                                                                                    \
            const int c = 2 * s + lhi;                                                                              \
            const bf16x8 a0 = *(const bf16x8 *)((SA) + ra0 * MK + (c ^ swza) * 8);                                  \
            const bf16x8 a1 = *(const bf16x8 *)((SA) + (ra0 + 32) * MK + (c ^ swza) * 8);                           \
            const bf16x8 b0 = *(const bf16x8 *)((SB) + rb0 * MK + (c ^ swzb) * 8);                                  \
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc[0], 0, 0, 0);                              \
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b0, acc[1], 0, 0, 0);                              \
        }                                                                                                           \
    } while (0)
    // Every step issues one stage of 6 DMA instructions (past the end of K it loads the last step again, into the slot
    // nobody reads any more), so when step kc starts, stages kc + 1 and kc + 2 are the only later ones in flight: wait
    // until this wave has at most those 12 outstanding, barrier (every wave's part of stage kc has landed, every wave
    // is done with stage kc - 1), refill the slot of stage kc - 1, multiply stage kc.  The acquire fence (LDS only)
    // keeps the stage's reads below the barrier.
#define STEP(CA, CB, NA, NB, kc)                                                                                    \
    do {                                                                                                            \
        __builtin_amdgcn_s_waitcnt(0x0F70 | 12);                                                                    \
        __builtin_amdgcn_s_barrier();                                                                               \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");                                             \
        DMA(NA, NB, ((kc) + 3 < KT ? (kc) + 3 : KT - 1));                                                           \
        MMA(CA, CB, kc);                                                                                            \
        __builtin_amdgcn_sched_barrier(0);                                                                          \
    } while (0)
    DMA(sa0, sb0, 0);
    DMA(sa1, sb1, (1 < KT ? 1 : KT - 1));
    DMA(sa2, sb2, (2 < KT ? 2 : KT - 1));
    for (int kt = 0; kt < KT; kt += 4) {
        STEP(sa0, sb0, sa3, sb3, kt);
        if (kt + 1 >= KT) break;
        STEP(sa1, sb1, sa0, sb0, kt + 1);
        if (kt + 2 >= KT) break;
        STEP(sa2, sb2, sa1, sb1, kt + 2);
        if (kt + 3 >= KT) break;
        STEP(sa3, sb3, sa2, sb2, kt + 3);
    }
    // no DMA may still be writing this workgroup's LDS when it ends
    __builtin_amdgcn_s_waitcnt(0x0F70);
#undef STEP
#undef MMA
#undef DMA
    // lane holds C[row][col] with col = l32, row = 8 (r / 4) + 4 lhi + (r % 4)
    const long col = n0 + wn * 32 + l32;
    const float bias = EPI == EPI_BIAS_GELU ? ep.bias[col] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            epilogue4<EPI>(ep, m0 + wm * 64 + i * 32 + 8 * q + 4 * lhi, col, bias,
                           {acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]});
}

// ---- operand preparation ------------------------------------------------------------------------
// Rows m_first .. of x (fp32 [rows][K]) -> bf16 x16 [M][K] and its transpose x16t [K][ldt]; rows at and past `rows` are
// zero.  One 64 x 32 tile per workgroup through LDS.  x may be pinned host memory: a host batch is then read over PCIe
// once, by this kernel, chunk after chunk behind the host's copies into that memory, and its targets (tgt_src, `rows` of
// them, may be null) come along.  Bound by PCIe there: 16 B per lane,
// every load of a thread in flight; 0.5 MB in 14.5 us, 36 GB/s, against 87 us for 2 MB through hipMemcpy.
__global__ __launch_bounds__(256) void stage_input_kernel(const float *__restrict__ x, int m_first, int rows, int K,
                                                          bf16 *__restrict__ x16, bf16 *__restrict__ x16t, long ldt,
                                                          const float *__restrict__ tgt_src, float *__restrict__ tgt) {
    __shared__ bf16 tile[32][64 + 2];
    const int m0 = m_first + blockIdx.x * 64, k0 = blockIdx.y * 32;
    if (tgt_src && blockIdx.y == 0 && threadIdx.x < 64 && m0 + (int)threadIdx.x < rows)
        tgt[m0 + threadIdx.x] = tgt_src[m0 + threadIdx.x];
    float4 f[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = threadIdx.x + u * 256, m = m0 + (e >> 3);
        f[u] = *(const float4 *)(x + (long)(m < rows ? m : rows - 1) * K + k0 + (e & 7) * 4);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = threadIdx.x + u * 256, m = e >> 3, k = (e & 7) * 4;
        const bool in = m0 + m < rows;
        const bf16x4 v = {(bf16)(in ? f[u].x : 0.0f), (bf16)(in ? f[u].y : 0.0f), (bf16)(in ? f[u].z : 0.0f),
                          (bf16)(in ? f[u].w : 0.0f)};
        *(bf16x4 *)(x16 + (long)(m0 + m) * K + k0 + k) = v;
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[k + j][m] = v[j];
    }
    __syncthreads();
    if (x16t)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int e = threadIdx.x + u * 256, k = e >> 6, m = e & 63;
            x16t[(long)(k0 + k) * ldt + m0 + m] = tile[k][m];
        }
}

// Arrays one after the other into pinned host memory, 4096 floats per workgroup: one launch and one wait for all the
// parameters of a network, where a copy into pageable memory waits for each array.
constexpr int PACK_MAX = 2 * 4 + 1;
struct PackArgs {
    const float *src[PACK_MAX];
    int first[PACK_MAX + 1];   // in float4
    int count;
};
__global__ __launch_bounds__(256) void pack_kernel(PackArgs a, float4 *__restrict__ dst) {
    float4 f[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int x = min((int)blockIdx.x * 1024 + u * 256 + (int)threadIdx.x, a.first[a.count] - 1);
        int i = 0;
#pragma unroll
        for (int j = 1; j < PACK_MAX; ++j) i += j < a.count && x >= a.first[j];
        f[u] = ((const float4 *)a.src[i])[x - a.first[i]];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int x = (int)blockIdx.x * 1024 + u * 256 + (int)threadIdx.x;
        if (x < a.first[a.count]) dst[x] = f[u];
    }
}

// dPre of the last hidden layer, dpre[m][k] = dy[m] w[k] gelu'(pre[m][k]) (bf16), and its transpose
__global__ __launch_bounds__(256) void head_backward_t_kernel(const float *__restrict__ dy, const float *__restrict__ w,
                                                              const float *__restrict__ pre, int K,
                                                              bf16 *__restrict__ dpre, bf16 *__restrict__ dpret,
                                                              long ldt) {
    __shared__ bf16 tile[32][64 + 2];
    const int m0 = blockIdx.x * 64, k0 = blockIdx.y * 32;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int e = threadIdx.x + u * 256, m = e >> 5, k = e & 31;
        const long at = (long)(m0 + m) * K + k0 + k;
        const bf16 v = (bf16)(dy[m0 + m] * w[k0 + k] * gelu_grad(pre[at]));
        dpre[at] = v;
        tile[k][m] = v;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int e = threadIdx.x + u * 256, k = e >> 6, m = e & 63;
        dpret[(long)(k0 + k) * ldt + m0 + m] = tile[k][m];
    }
}

// ---- weight gradients of every layer, one launch ------------------------------------------------------
// dW_l [K_l][N] = X_l^T dP_l: a contraction over the batch with only K_l x N outputs.  The batch is cut into `slices`
// of at least 128 rows, each slice one MFMA chain, and the slices are added in ascending order in fp32.  A workgroup
// owns one 64 x 64 tile of one layer (a 32 x 32 quadrant per wave) and walks the whole batch, so the slices' sum stays
// in registers and no partial product goes through memory (33 MB written and read again per 512 x 512 layer with a
// workgroup per slice); the 144 tiles of a 128 -> 512 -> 512 -> 512 network run side by side.  Operands come by DMA in
// steps of 64 rows, four LDS stages, as in the GEMM above.
// Batch 4096 of that network: 26.6 us (21 us per layer with a workgroup per slice; 53 us for 32 x 32 tiles that read
// their operands straight from L2, 300 MB of them).
constexpr int DW_T = 64, DW_MAX = 4;
struct DwArgs {
    const bf16 *xt[DW_MAX], *dt[DW_MAX];   // [K_l][ldt], [N][ldt]
    float *g[DW_MAX];                      // [K_l][N]
    int first[DW_MAX];                     // first tile of each layer
    int slices[DW_MAX];
    int N, rows;                           // rows: the padded batch
    long ldt;
};

__global__ __launch_bounds__(256) void weight_grads_kernel(DwArgs a) {
    __shared__ __attribute__((aligned(16))) bf16 sa0[DW_T * MK], sa1[DW_T * MK], sa2[DW_T * MK], sa3[DW_T * MK];
    __shared__ __attribute__((aligned(16))) bf16 sb0[DW_T * MK], sb1[DW_T * MK], sb2[DW_T * MK], sb3[DW_T * MK];
    unsigned t = blockIdx.x;
    if ((gridDim.x & 7) == 0) t = (t & 7) * (gridDim.x >> 3) + (t >> 3);   // an XCD: neighbouring tiles
    int l = 0;
#pragma unroll
    for (int i = 1; i < DW_MAX; ++i) l += (int)t >= a.first[i];
    const int tile = (int)t - a.first[l], ntn = a.N / DW_T;
    const int k0 = tile / ntn * DW_T, n0 = tile % ntn * DW_T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, lhi = lane >> 5;
    const int wm = wave >> 1, wn = wave & 1;
    const int drow = lane >> 3, dchunk = swz8(drow, lane & 7);
    const bf16 *ga[2], *gb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        ga[i] = a.xt[l] + (long)(k0 + wave * 16 + i * 8 + drow) * a.ldt + dchunk * 8;
        gb[i] = a.dt[l] + (long)(n0 + wave * 16 + i * 8 + drow) * a.ldt + dchunk * 8;
    }
    const int KT = a.rows / MK;                        // even: rows is a multiple of 128
    const int per = KT / a.slices[l];                  // steps per slice, even
#define DMA(SA, SB, kc)                                                                                             \
    do {                                                                                                            \
        _Pragma("unroll") for (int i = 0; i < 2; ++i) {                                                             \
            __builtin_amdgcn_global_load_lds((const void *)(ga[i] + (long)(kc) * MK),                               \
                                             (lds_void *)((SA) + (wave * 16 + i * 8) * MK), 16, 0, 0);              \
            __builtin_amdgcn_global_load_lds((const void *)(gb[i] + (long)(kc) * MK),                               \
                                             (lds_void *)((SB) + (wave * 16 + i * 8) * MK), 16, 0, 0);              \
        }                                                                                                           \
    } while (0)
    f32x16 acc, sum;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = sum[r] = 0.0f;
    const int ra0 = wm * 32 + l32, rb0 = wn * 32 + l32, sw = l32 & 7;
    // as in the GEMM: 4 DMA instructions per step, two later steps in flight
#define STEP(CA, CB, NA, NB, kc)                                                                                    \
    do {                                                                                                            \
        __builtin_amdgcn_s_waitcnt(0x0F70 | 8);                                                                     \
        __builtin_amdgcn_s_barrier();                                                                               \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");                                             \
        DMA(NA, NB, ((kc) + 3 < KT ? (kc) + 3 : KT - 1));                                                           \
        _Pragma("unroll") for (int s = 0; s < 4; ++s) {                                                             \
            const int c = (2 * s + lhi) ^ sw;                                                                       \
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8 *)((CA) + ra0 * MK + c * 8),               \
                                                          *(const bf16x8 *)((CB) + rb0 * MK + c * 8), acc, 0, 0, 0); \
        }                                                                                                           \
        __builtin_amdgcn_sched_barrier(0);                                                                          \
        if (++in == per) {                                                                                          \
            in = 0;                                                                                                 \
            _Pragma("unroll") for (int r = 0; r < 16; ++r) {                                                        \
                sum[r] += acc[r];                                                                                   \
                acc[r] = 0.0f;                                                                                      \
            }                                                                                                       \
        }                                                                                                           \
    } while (0)
    int in = 0;
    DMA(sa0, sb0, 0);
    DMA(sa1, sb1, 1);
    DMA(sa2, sb2, (2 < KT ? 2 : KT - 1));
    for (int kt = 0; kt < KT; kt += 4) {
        STEP(sa0, sb0, sa3, sb3, kt);
        STEP(sa1, sb1, sa0, sb0, kt + 1);
        if (kt + 2 >= KT) break;
        STEP(sa2, sb2, sa1, sb1, kt + 2);
        STEP(sa3, sb3, sa2, sb2, kt + 3);
    }
    // no DMA may still be writing this workgroup's LDS when it ends
    __builtin_amdgcn_s_waitcnt(0x0F70);
#undef STEP
#undef DMA
#pragma unroll
    for (int r = 0; r < 16; ++r)
        a.g[l][(long)(k0 + wm * 32 + 8 * (r >> 2) + 4 * lhi + (r & 3)) * a.N + n0 + wn * 32 + l32] = sum[r];
}

// ---- column sums: the bias gradients of every layer and the head's weight gradient -------------------
// out_i[k] = sum_m a_i[m][k] (s_i ? s_i[m] : 1).  Stage 1: 64 row chunks, 8 columns per thread, four row subgroups of a
// chunk added through LDS in a fixed order; stage 2 adds the chunks in ascending order and, in one more row of
// workgroups, the two scalar sums of the step (squared errors, d loss / d b_out).
constexpr int CS_CHUNKS = 64, CS_MAX = DW_MAX + 1;
struct ColsumArgs {
    const bf16 *a[CS_MAX];
    const float *s[CS_MAX];
    float *out[CS_MAX];
    int count, M, K;
    float *part;             // count x 64 x K
    const float *v[2];       // scalar sums over M
    float *vout;
};

__global__ __launch_bounds__(256) void colsums_part_kernel(ColsumArgs c) {
    __shared__ float red[4][512];
    const int i = blockIdx.z;
    const bf16 *__restrict__ a = c.a[i];
    const float *__restrict__ s = c.s[i];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int k0 = blockIdx.x * 512 + tx * 8;
    const int rows = (c.M + CS_CHUNKS - 1) / CS_CHUNKS;
    const int m0 = blockIdx.y * rows, m1 = min(c.M, m0 + rows);
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (k0 < c.K)
#pragma unroll 4
        for (int m = m0 + ty; m < m1; m += 4) {
            const bf16x8 v = *(const bf16x8 *)(a + (long)m * c.K + k0);
            const float sc = s ? s[m] : 1.0f;
#pragma unroll
            for (int t = 0; t < 8; ++t) acc[t] += (float)v[t] * sc;
        }
#pragma unroll
    for (int t = 0; t < 8; ++t) red[ty][tx * 8 + t] = acc[t];
    __syncthreads();
    if (ty == 0 && k0 < c.K)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int x = tx * 8 + t;
            c.part[((long)i * CS_CHUNKS + blockIdx.y) * c.K + k0 + t] = ((red[0][x] + red[1][x]) + red[2][x]) + red[3][x];
        }
}

__global__ __launch_bounds__(256) void colsums_finish_kernel(ColsumArgs c) {
    __shared__ float red[4];
    const int i = blockIdx.y;
    if (i < c.count) {
        const int k = blockIdx.x * 256 + threadIdx.x;
        if (k >= c.K) return;
        const float *__restrict__ p = c.part + (long)i * CS_CHUNKS * c.K + k;
        float acc = 0.0f;
#pragma unroll 32
        for (int j = 0; j < CS_CHUNKS; ++j) acc += p[(long)j * c.K];
        c.out[i][k] = acc;
        return;
    }
    for (int w = blockIdx.x; w < 2; w += gridDim.x) {
        const float *__restrict__ v = c.v[w];
        float acc = 0.0f;
#pragma unroll 8
        for (int j = threadIdx.x; j < c.M; j += 256) acc += v[j];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0)   // pinned host memory
            __hip_atomic_store(c.vout + w, red[0] + red[1] + red[2] + red[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __syncthreads();
    }
}

// ---- Adam on every parameter array, one launch --------------------------------------------------
// fp32 master weights; the bf16 copies [K][N] and [N][K] are rewritten.  A weight matrix goes by 32 x 32 tiles, the
// transposed copy through LDS (written element by element it took one 2 B store per weight, 2 KB apart); a vector goes
// by runs of 1024.
constexpr int ADAM_MAX = 2 * DW_MAX + 1;
struct AdamArgs {
    float *w[ADAM_MAX], *m[ADAM_MAX], *v[ADAM_MAX];
    const float *g[ADAM_MAX];      // null: no step, only the bf16 copies, and the moments cleared
    bf16 *wb[ADAM_MAX], *wtb[ADAM_MAX];
    int rows[ADAM_MAX], cols[ADAM_MAX], first[ADAM_MAX + 1];
    int count;
    float lr, b1, b2, eps, c1, c2;
};

__global__ __launch_bounds__(256) void adam_all_kernel(AdamArgs a) {
    __shared__ bf16 tile[32][32 + 2];
    int i = 0;
#pragma unroll
    for (int j = 1; j < ADAM_MAX; ++j) i += j < a.count && (int)blockIdx.x >= a.first[j];
    const int t = (int)blockIdx.x - a.first[i], N = a.cols[i];
    const bool matrix = a.wb[i] != nullptr;
    const int ntn = N >> 5, r0 = matrix ? t / ntn * 32 : 0, c0 = matrix ? t % ntn * 32 : t * 1024;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = threadIdx.x + u * 256;
        const int r = matrix ? e >> 5 : 0, c = matrix ? e & 31 : e;
        if (!matrix && c0 + c >= N) continue;
        const long at = (long)(r0 + r) * N + c0 + c;
        float mi = 0.0f, vi = 0.0f, wi = a.w[i][at];
        if (a.g[i]) {
            const float gi = a.g[i][at];
            // products fused explicitly, so that the rounding does not depend on what the compiler contracts
            mi = fmaf(1.0f - a.b1, gi, a.b1 * a.m[i][at]);
            vi = fmaf(gi, (1.0f - a.b2) * gi, a.b2 * a.v[i][at]);
            wi -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
            a.w[i][at] = wi;
        }
        a.m[i][at] = mi;
        a.v[i][at] = vi;
        if (matrix) {
            a.wb[i][at] = (bf16)wi;
            tile[c][r] = (bf16)wi;
        }
    }
    if (!matrix) return;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = threadIdx.x + u * 256, c = e >> 5, r = e & 31;
        a.wtb[i][(long)(c0 + c) * a.rows[i] + r0 + r] = tile[c][r];
    }
}

}  // namespace

// ---- C ABI ------------------------------------------------------------------------------------
// epi: 0 fp32 C, 1 bias + GELU, 2 GELU backward; actT: the bf16 result transposed as well ([N][ldt]), or null
extern "C" int ork_mlp_gemm_mid(void *stream, int epi, const void *A, int lda, const void *B, int ldb, int M, int N,
                                int K, float *c32, int ldc, const float *bias, float *pre, void *act, void *actT,
                                long ldt) {
    // the DMA and the fragment reads move 16 B: rows of both operands start on 16 B boundaries
    if (M % MM || N % MN || K % 32 || M <= 0 || N <= 0 || K <= 0 || lda % 8 || ldb % 8 || ((uintptr_t)A & 15) ||
        ((uintptr_t)B & 15) || ldt % 4)
        return (int)hipErrorInvalidValue;
    const EpiArgs ep{c32, ldc, bias, pre, (bf16 *)act, (bf16 *)actT, ldt};
    const long tiles = (long)(M / MM) * (N / MN);
    if (tiles >= (1L << 31)) return (int)hipErrorInvalidValue;
    hipStream_t st = (hipStream_t)stream;
    const bf16 *a = (const bf16 *)A, *b = (const bf16 *)B;
    switch (epi) {
    case EPI_F32: gemm_nt_mid_kernel<EPI_F32><<<(unsigned)tiles, MT, 0, st>>>(a, lda, b, ldb, K, ep, N / MN); break;
    case EPI_BIAS_GELU: gemm_nt_mid_kernel<EPI_BIAS_GELU><<<(unsigned)tiles, MT, 0, st>>>(a, lda, b, ldb, K, ep, N / MN); break;
    case EPI_GELU_BWD: gemm_nt_mid_kernel<EPI_GELU_BWD><<<(unsigned)tiles, MT, 0, st>>>(a, lda, b, ldb, K, ep, N / MN); break;
    default: return (int)hipErrorInvalidValue;
    }
    ORK_LAUNCH_CHECK();
    return 0;
}

// rows m0 .. m1 - 1 of x fp32 [rows][K] -> x16 [M][K] and x16t [K][ldt] (null: not needed); m0 and m1 multiples of 64, K
// of 32; x on a 16 B boundary, device or pinned host memory.  tgt_src: `rows` targets to copy to tgt, or null.
extern "C" int ork_mlp_stage_input(void *stream, const float *x, int m0, int m1, int rows, int K, void *x16, void *x16t,
                                   long ldt, const float *tgt_src, float *tgt) {
    if (m0 % 64 || m1 % 64 || K % 32 || m0 < 0 || m1 <= m0 || rows <= 0 || K <= 0 || ((uintptr_t)x & 15))
        return (int)hipErrorInvalidValue;
    stage_input_kernel<<<dim3((m1 - m0) / 64, K / 32), 256, 0, (hipStream_t)stream>>>(
        x, m0, rows, K, (bf16 *)x16, (bf16 *)x16t, ldt, tgt_src, tgt);
    ORK_LAUNCH_CHECK();
    return 0;
}

// dst = the arrays src[i] of len[i] floats (multiples of 4) one after the other; dst and every src on 16 B boundaries
extern "C" int ork_mlp_pack(void *stream, int count, const float *const *src, const int *len, float *dst) {
    if (count < 1 || count > PACK_MAX) return (int)hipErrorInvalidValue;
    PackArgs a{};
    long total = 0;
    for (int i = 0; i < count; ++i) {
        if (len[i] <= 0 || len[i] % 4) return (int)hipErrorInvalidValue;
        a.src[i] = src[i];
        a.first[i] = (int)total;
        total += len[i] / 4;
    }
    if (total > (1 << 28)) return (int)hipErrorInvalidValue;
    a.first[count] = (int)total;
    a.count = count;
    pack_kernel<<<(unsigned)((total + 1023) / 1024), 256, 0, (hipStream_t)stream>>>(a, (float4 *)dst);
    ORK_LAUNCH_CHECK();
    return 0;
}

extern "C" int ork_mlp_head_backward_t(void *stream, const float *dy, const float *w, const float *pre, int M, int K,
                                       void *dpre, void *dpret, long ldt) {
    if (M % 64 || K % 32 || M <= 0 || K <= 0) return (int)hipErrorInvalidValue;
    head_backward_t_kernel<<<dim3(M / 64, K / 32), 256, 0, (hipStream_t)stream>>>(dy, w, pre, K, (bf16 *)dpre,
                                                                                (bf16 *)dpret, ldt);
    ORK_LAUNCH_CHECK();
    return 0;
}

// g[l] [K[l]][N] = xt[l] dt[l]^T for l < nl; rows: the padded batch, a multiple of 128; slices: at most max_slices
extern "C" int ork_mlp_weight_grads(void *stream, int nl, const void *const *xt, const void *const *dt, float *const *g,
                                    const int *K, int N, int rows, long ldt, int max_slices) {
    if (nl < 1 || nl > DW_MAX || N % 128 || rows % 128 || rows <= 0 || ldt % 8) return (int)hipErrorInvalidValue;
    DwArgs a{};
    a.N = N;
    a.rows = rows;
    a.ldt = ldt;
    int total = 0;
    for (int l = 0; l < DW_MAX; ++l) {
        a.first[l] = l < nl ? total : 0x7fffffff;
        if (l >= nl) continue;
        if (K[l] % 128) return (int)hipErrorInvalidValue;
        a.xt[l] = (const bf16 *)xt[l];
        a.dt[l] = (const bf16 *)dt[l];
        a.g[l] = g[l];
        // up to max_slices slices of at least 128 rows while 128 x 128 tiles times slices stay below 512: the slicing
        // fixes the order of the sum
        const int tiles = (K[l] / 128) * (N / 128);
        int slices = 1;
        while (slices < max_slices && tiles * slices < 512 && rows % (slices * 2 * 128) == 0) slices *= 2;
        a.slices[l] = slices;
        total += (K[l] / DW_T) * (N / DW_T);
    }
    weight_grads_kernel<<<total, 256, 0, (hipStream_t)stream>>>(a);
    ORK_LAUNCH_CHECK();
    return 0;
}

// out[i][k] = sum_m a[i][m][k] (s[i] ? s[i][m] : 1), i < count; vout[0..1] = sums of v0 and v1 over M (device or pinned host
// memory); part: count x 64 x K floats
extern "C" int ork_mlp_colsums(void *stream, int count, const void *const *a, const float *const *s, float *const *out,
                               int M, int K, float *part, const float *v0, const float *v1, float *vout) {
    if (count < 1 || count > CS_MAX || K % 8 || K <= 0 || M <= 0) return (int)hipErrorInvalidValue;
    ColsumArgs c{};
    for (int i = 0; i < count; ++i) {
        c.a[i] = (const bf16 *)a[i];
        c.s[i] = s[i];
        c.out[i] = out[i];
    }
    c.count = count;
    c.M = M;
    c.K = K;
    c.part = part;
    c.v[0] = v0;
    c.v[1] = v1;
    c.vout = vout;
    colsums_part_kernel<<<dim3((K + 511) / 512, CS_CHUNKS, count), 256, 0, (hipStream_t)stream>>>(c);
    ORK_LAUNCH_CHECK();
    colsums_finish_kernel<<<dim3((K + 255) / 256, count + 1), 256, 0, (hipStream_t)stream>>>(c);
    ORK_LAUNCH_CHECK();
    return 0;
}

// one Adam step on `count` arrays of rows[i] x cols[i]; with wb and wtb (rows and cols multiples of 32) the bf16 copies
// are written, else the array is a vector (rows 1); g[i] null: the copies only, and the moments cleared
extern "C" int ork_mlp_adam_all(void *stream, int count, float *const *w, const float *const *g, float *const *m,
                                float *const *v, void *const *wb, void *const *wtb, const int *rows, const int *cols,
                                float lr, float b1, float b2, float eps, float c1, float c2) {
    if (count < 1 || count > ADAM_MAX) return (int)hipErrorInvalidValue;
    AdamArgs a{};
    int total = 0;
    for (int i = 0; i < count; ++i) {
        if (wb[i] ? (rows[i] % 32 || cols[i] % 32 || !wtb[i]) : rows[i] != 1) return (int)hipErrorInvalidValue;
        a.w[i] = w[i];
        a.g[i] = g[i];
        a.m[i] = m[i];
        a.v[i] = v[i];
        a.wb[i] = (bf16 *)wb[i];
        a.wtb[i] = (bf16 *)wtb[i];
        a.rows[i] = rows[i];
        a.cols[i] = cols[i];
        a.first[i] = total;
        total += wb[i] ? (rows[i] / 32) * (cols[i] / 32) : (cols[i] + 1023) / 1024;
    }
    a.count = count;
    a.lr = lr;
    a.b1 = b1;
    a.b2 = b2;
    a.eps = eps;
    a.c1 = c1;
    a.c2 = c2;
    adam_all_kernel<<<total, 256, 0, (hipStream_t)stream>>>(a);
    ORK_LAUNCH_CHECK();
    return 0;
}
