/*
 * Newton initial-guess network: a 16 -> 256 -> 256 -> 256 -> 1 MLP with SiLU,
 * BF16 weights and activations on the matrix cores (v_mfma_f32_32x32x16
 * bf16, FP32 accumulate), FP32 master weights and Adam for training.
 *
 * On matrix-core tiles lane l feeds rows/cols l % 32 and the k octet
 * (l / 32) * 8 .. +7 of every 16-deep step, and receives C rows
 * (v / 4) * 8 + (l / 32) * 4 + v % 4, column l % 32, v = 0..15.
 *
 * Layer-by-layer inference is k_gemm_bf16 per layer.  A training step is
 * three launches: k_train_rows (forward and backward of a tile of rows),
 * k_train_dw (weight gradients and the parts of the column sums) and
 * k_train_apply (the column sums, and Adam).  At 4000 rows they take 24.5,
 * 14.5 and 5.1 us; as 24 launches, a layer's product, SiLU derivative and
 * column sums each their own and the weight gradients 64 waves that waited
 * for every load, a step was 471 us.
 *
 * Inference inside the transient uses k_guess_net instead: one kernel from
 * the feature rows to the nodes' starting values, with the weights held in
 * registers and the activations in LDS.  It issues the same matrix-core
 * steps in the same order and the same element-wise code, so its outputs
 * equal the layer-by-layer path's bit for bit.
 */
#include <algorithm>
#include "ngmi_internal.h"
#include "mlp_types.h"
#include "guess_types.h"

namespace ngmi {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma16(bf16x8 a, bf16x8 b, f32x16 acc)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}

/*
 * One hidden layer: Cb[i][j] = hidden_out(bias[j] + sum_k A[i][k] B[j][k]),
 * grid: (N/32, tiles) wavefronts of 64 lanes, each a 32 x 32 tile; M, N
 * multiples of 32, K a multiple of 16.  Row tiles are visited grid-stride,
 * so with Mdev (a device row count below M) the launch can be sized to the
 * machine and the work follows the rows actually present.
 */
__global__ void __launch_bounds__(64)
k_gemm_bf16(const unsigned short *__restrict__ A, const unsigned short *__restrict__ B,
            const float *__restrict__ bias, unsigned short *__restrict__ Cb, int M, int N, int K,
            const int *__restrict__ Mdev)
{
    const int l = threadIdx.x;
    const int j0 = blockIdx.x * 32;
    if (Mdev) M = min(M, *Mdev);
    const int r = l & 31, kq = (l >> 5) * 8;
    for (int i0 = blockIdx.y * 32; i0 < M; i0 += gridDim.y * 32) {
        /* the accumulator starts from the bias (the column is the lane's,
         * the same for all 16 values) */
        const float acc0 = bias[j0 + r];
        f32x16 acc;
#pragma unroll
        for (int v = 0; v < 16; v++) acc[v] = acc0;
        const unsigned short *pa = A + (int64_t)(i0 + r) * K;
        const unsigned short *pb = B + (int64_t)(j0 + r) * K;
        for (int k0 = 0; k0 < K; k0 += 16)
            acc = mfma16(*reinterpret_cast<const bf16x8 *>(pa + k0 + kq),
                         *reinterpret_cast<const bf16x8 *>(pb + k0 + kq), acc);
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int i = i0 + (v >> 2) * 8 + (l >> 5) * 4 + (v & 3);
            if (i < M) Cb[(int64_t)i * N + j0 + r] = hidden_out(acc[v]);
        }
    }
}

__global__ void k_f32_to_bf16(const float *__restrict__ x, unsigned short *__restrict__ y, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

/* output layer (256 -> 1) forward: y[i] = b + the in-order sum of the
 * blocks' dot products over MLP_HEAD_BLOCK hidden units, each accumulated
 * in order with FMA (k_guess_net sums the same way).  K is a multiple of
 * MLP_HEAD_BLOCK. */
__global__ void k_head(const unsigned short *__restrict__ H, const unsigned short *__restrict__ w,
                       const float *__restrict__ b, float *__restrict__ y, int M, int K,
                       const int *__restrict__ Mdev)
{
    if (Mdev) M = min(M, *Mdev);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < M; i += gridDim.x * blockDim.x) {
        float s = b[0];
        for (int k0 = 0; k0 < K; k0 += MLP_HEAD_BLOCK) {
            float p = 0.0f;
            for (int k = k0; k < k0 + MLP_HEAD_BLOCK; k++) p = fmaf(bf2f(H[(int64_t)i * K + k]), bf2f(w[k]), p);
            s += p;
        }
        y[i] = s;
    }
}

/* ---------------- fused inference for the transient ---------------- */

constexpr int GN_THREADS = 512;                 /* 8 waves: wave w owns hidden units 32w .. 32w + 31 */
constexpr int GN_XLD = MLP_IN_PAD + 8;          /* LDS row strides in elements, padded by 16 bytes */
constexpr int GN_HLD = MLP_HID + 8;
constexpr int GN_HEAD_BLOCKS = MLP_HID / MLP_HEAD_BLOCK;
static_assert(GN_THREADS == 32 * MLP_IN, "the input tile is packed one element per thread");
static_assert(GN_THREADS / 64 * 32 == MLP_HID, "one wave per 32 hidden units");

/* one hidden layer for a tile of 32 rows: A (32 x 16 STEPS, BF16, LDS) times
 * this wave's register-resident weight octets, written to out (LDS) as
 * BF16 activations of columns col0 .. col0 + 31.  The matrix-core steps and
 * the epilogue are those of k_gemm_bf16 (the accumulator starts at the
 * bias). */
template <int STEPS>
__device__ __forceinline__ void gn_layer(const unsigned short *A, int lda, const bf16x8 (&w)[STEPS], float bias,
                                         unsigned short *out, int col0, int l)
{
    const unsigned short *pa = A + (l & 31) * lda + (l >> 5) * 8;
    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = bias;
#pragma unroll
    for (int s = 0; s < STEPS; s++) acc = mfma16(*reinterpret_cast<const bf16x8 *>(pa + 16 * s), w[s], acc);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int i = (v >> 2) * 8 + (l >> 5) * 4 + (v & 3);
        out[i * GN_HLD + col0 + (l & 31)] = hidden_out(acc[v]);
    }
}

/*
 * Feature rows -> network -> starting values, one launch.  count[0] holds
 * the number of rows (at most maxRows), count[1] is a finish counter: the
 * last workgroup to finish clears both, so the next pass's features kernel
 * starts from zero without a separate launch.  Without count the rows are
 * maxRows and no counter is touched.  Each workgroup loads the
 * BF16 weights once into registers (8 + 64 + 64 VGPRs a lane) and walks
 * tiles of 32 rows grid-stride; per tile the packed input and the hidden
 * activations stay in LDS.  Row r's node value x[dest[r]] becomes
 * guess_value(base[r], y) (and yout[r] = y when yout is set); rows_total,
 * when set, accumulates the rows processed.
 */
__global__ void __launch_bounds__(GN_THREADS)
k_guess_net(const float *__restrict__ X, const unsigned short *__restrict__ wb, const float *__restrict__ wf,
            int *count, int maxRows, const int64_t *__restrict__ dest, const double2 *__restrict__ base,
            double *__restrict__ x, float *__restrict__ yout, unsigned long long *rows_total)
{
    __shared__ __align__(16) unsigned short xs[32 * GN_XLD];
    __shared__ __align__(16) unsigned short ha[32 * GN_HLD];
    __shared__ __align__(16) unsigned short hb[32 * GN_HLD];
    __shared__ float w4s[MLP_HID];
    __shared__ float ps[32][GN_HEAD_BLOCKS + 1];
    const int tid = threadIdx.x, l = tid & 63, col0 = (tid >> 6) * 32;
    const int M = count ? min(count[0], maxRows) : maxRows;
    if ((int64_t)blockIdx.x * 32 < M) {
        const int j = col0 + (l & 31), kh = (l >> 5) * 8;
        bf16x8 w1[MLP_IN_PAD / 16], w2[MLP_HID / 16], w3[MLP_HID / 16];
        const unsigned short *p1 = wb + MLP_OFF_W1 + (int64_t)j * MLP_IN_PAD + kh;
        const unsigned short *p2 = wb + MLP_OFF_W2 + (int64_t)j * MLP_HID + kh;
        const unsigned short *p3 = wb + MLP_OFF_W3 + (int64_t)j * MLP_HID + kh;
#pragma unroll
        for (int s = 0; s < MLP_IN_PAD / 16; s++) w1[s] = *reinterpret_cast<const bf16x8 *>(p1 + 16 * s);
#pragma unroll
        for (int s = 0; s < MLP_HID / 16; s++) {
            w2[s] = *reinterpret_cast<const bf16x8 *>(p2 + 16 * s);
            w3[s] = *reinterpret_cast<const bf16x8 *>(p3 + 16 * s);
        }
        const float b1 = wf[MLP_OFF_B1 + j], b2 = wf[MLP_OFF_B2 + j], b3 = wf[MLP_OFF_B3 + j];
        const float b4 = wf[MLP_OFF_B4];
        for (int e = tid; e < MLP_HID; e += GN_THREADS) w4s[e] = bf2f(wb[MLP_OFF_W4 + e]);
        for (int e = tid; e < 32 * GN_XLD; e += GN_THREADS) xs[e] = 0;   /* the zero columns stay */
        __syncthreads();
        /* this thread's input element (row tid / 16, feature tid % 16) of
         * the tile, loaded one tile ahead so its latency hides behind the
         * previous tile's layers */
        const int rr = tid >> 4, cc = tid & 15;
        const int64_t step = (int64_t)gridDim.x * 32;
        int64_t i0 = (int64_t)blockIdx.x * 32;
        float xin = i0 + rr < M ? X[(i0 + rr) * MLP_IN + cc] : 0.0f;
        for (; i0 < M; i0 += step) {
            xs[rr * GN_XLD + cc] = f2bf(xin);
            xin = i0 + step + rr < M ? X[(i0 + step + rr) * MLP_IN + cc] : 0.0f;
            /* the apply's operands, loaded now for use after the layers */
            const bool mine = tid < 32 && i0 + tid < M;
            const int64_t d_row = (mine && x) ? dest[i0 + tid] : 0;
            const double2 b_row = (mine && x) ? base[i0 + tid] : make_double2(0.0, 0.0);
            __syncthreads();
            gn_layer(xs, GN_XLD, w1, b1, ha, col0, l);
            __syncthreads();
            gn_layer(ha, GN_HLD, w2, b2, hb, col0, l);
            __syncthreads();
            gn_layer(hb, GN_HLD, w3, b3, ha, col0, l);
            __syncthreads();
            if (tid < 32 * GN_HEAD_BLOCKS) {
                const int rr = tid / GN_HEAD_BLOCKS, cb = tid % GN_HEAD_BLOCKS;
                const uint4 *h = reinterpret_cast<const uint4 *>(ha + rr * GN_HLD + cb * MLP_HEAD_BLOCK);
                const float *w4 = w4s + cb * MLP_HEAD_BLOCK;
                float p = 0.0f;
#pragma unroll
                for (int q = 0; q < MLP_HEAD_BLOCK / 8; q++) {
                    const uint4 u = h[q];
                    const unsigned int wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        p = fmaf(bf2f((unsigned short)(wd[e] & 0xffffu)), w4[8 * q + 2 * e], p);
                        p = fmaf(bf2f((unsigned short)(wd[e] >> 16)), w4[8 * q + 2 * e + 1], p);
                    }
                }
                ps[rr][cb] = p;
            }
            __syncthreads();
            if (mine) {
                float y = b4;
#pragma unroll
                for (int cb = 0; cb < GN_HEAD_BLOCKS; cb++) y += ps[tid][cb];
                if (yout) yout[i0 + tid] = y;
                if (x) x[d_row] = guess_value(b_row, y);
            }
        }
    }
    if (!count) return;
    __syncthreads();   /* every wave has read count[0] */
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(reinterpret_cast<unsigned int *>(count + 1), 1u) == gridDim.x - 1) {
            if (rows_total) atomicAdd(rows_total, (unsigned long long)M);
            count[0] = 0;
            count[1] = 0;
        }
    }
}

/* ---------------- training ---------------- */

/* The operands of the weight gradients, whose matrix-core steps run along
 * the rows: element (row, column) of a matrix of C columns at
 * ((row / 8) * C + column) * 8 + row % 8, so that a lane's octet of rows is
 * one 16-byte load and 32 lanes' are 512 consecutive bytes. */
__device__ __forceinline__ int64_t oct_at(int64_t row, int C, int col) { return ((row >> 3) * C + col) * 8 + (row & 7); }

/* 32 x 32 tile of A (32 rows, BF16, LDS) times this wave's weights, k in
 * order, from acc on */
template <int STEPS>
__device__ __forceinline__ f32x16 tr_product(const unsigned short *A, int lda, const bf16x8 (&w)[STEPS], f32x16 acc,
                                             int l)
{
    const unsigned short *pa = A + (l & 31) * lda + (l >> 5) * 8;
#pragma unroll
    for (int s = 0; s < STEPS; s++) acc = mfma16(*reinterpret_cast<const bf16x8 *>(pa + 16 * s), w[s], acc);
    return acc;
}

template <int STEPS>
__device__ __forceinline__ void tr_weights(bf16x8 (&w)[STEPS], const unsigned short *__restrict__ W, int ldw, int j, int l)
{
    const unsigned short *p = W + (int64_t)j * ldw + (l >> 5) * 8;
#pragma unroll
    for (int s = 0; s < STEPS; s++) w[s] = *reinterpret_cast<const bf16x8 *>(p + 16 * s);
}

/* this wave's tile, rounded to BF16: rows to LDS (the next product's
 * operand) and, in octets of rows, to memory */
__device__ __forceinline__ void tr_put(const unsigned short (&h)[16], unsigned short *lds, unsigned short *__restrict__ oct,
                                       int64_t i0, int j, int l)
{
#pragma unroll
    for (int v = 0; v < 16; v++) lds[((v >> 2) * 8 + (l >> 5) * 4 + (v & 3)) * GN_HLD + j] = h[v];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint2 u = make_uint2(h[4 * q] | (unsigned)h[4 * q + 1] << 16, h[4 * q + 2] | (unsigned)h[4 * q + 3] << 16);
        *reinterpret_cast<uint2 *>(oct + oct_at(i0 + 8 * q + 4 * (l >> 5), MLP_HID, j)) = u;
    }
}

/* this wave's tile of pre-activation gradients, FP32 by rows (the column
 * sums' operand) */
__device__ __forceinline__ void tr_rows(const float (&g)[16], float *__restrict__ out, int64_t i0, int j, int l)
{
    float *p = out + (i0 + (l >> 5) * 4) * MLP_HID + j;
#pragma unroll
    for (int v = 0; v < 16; v++) p[((v >> 2) * 8 + (v & 3)) * MLP_HID] = g[v];
}

/* dH times the derivative of SiLU at z */
__device__ __forceinline__ float silu_back(float dh, float z)
{
    const float s = 1.0f / (1.0f + __expf(-z));
    return dh * (s * (1.0f + z * (1.0f - s)));
}

/*
 * Forward and backward of 32 rows a workgroup: the rows' gradients need
 * nothing of the other rows, so pre-activations stay in registers (the wave
 * that forms a layer's columns also forms their gradients) and activations
 * and gradients go from layer to layer through LDS.  Out come y and dy, the
 * weight gradients' operands in octets of rows, and by rows the operands of
 * the column sums (h3, and the gradients in FP32).  The matrix-core steps and
 * the element-wise code are those of the inference kernels; rows from M on
 * have zero gradients.  wbt: W2 and W3 transposed, so that both directions
 * load octets.  Each layer's weights load during the layer before.  Bound by
 * that chain of seven barriers and by 530 KB of weights from L2 for every
 * workgroup: 24.5 us at 4000 rows, where 125 workgroups leave half of the
 * CUs idle.
 */
__global__ void __launch_bounds__(GN_THREADS)
k_train_rows(const float *__restrict__ X, const float *__restrict__ target, int M, TrainBufs B)
{
    __shared__ __align__(16) unsigned short xs[32 * GN_XLD];
    __shared__ __align__(16) unsigned short ha[32 * GN_HLD];
    __shared__ __align__(16) unsigned short hb[32 * GN_HLD];
    __shared__ float w4s[MLP_HID];
    __shared__ float ps[32][GN_HEAD_BLOCKS + 1];
    __shared__ float dys[32];
    const int tid = threadIdx.x, l = tid & 63, j = (tid >> 6) * 32 + (l & 31), r4 = (l >> 5) * 4;
    const int64_t i0 = (int64_t)blockIdx.x * 32;
    const unsigned short *__restrict__ wb = B.wb, *__restrict__ wbt = B.wbt;
    const float *__restrict__ wf = B.w;
    bf16x8 wa[MLP_HID / 16], wc[MLP_HID / 16], w1[MLP_IN_PAD / 16];
    {
        const int rr = tid >> 4, cc = tid & 15;
        const unsigned short v = f2bf(i0 + rr < M ? X[(i0 + rr) * MLP_IN + cc] : 0.0f);
        xs[rr * GN_XLD + cc] = v;
        xs[rr * GN_XLD + MLP_IN + cc] = 0;
        B.x[oct_at(i0 + rr, MLP_IN_PAD, cc)] = v;
        B.x[oct_at(i0 + rr, MLP_IN_PAD, MLP_IN + cc)] = 0;
    }
    if (tid < MLP_HID) w4s[tid] = bf2f(wb[MLP_OFF_W4 + tid]);
    tr_weights(w1, wb + MLP_OFF_W1, MLP_IN_PAD, j, l);
    tr_weights(wa, wb + MLP_OFF_W2, MLP_HID, j, l);
    const float b1 = wf[MLP_OFF_B1 + j], b2 = wf[MLP_OFF_B2 + j], b3 = wf[MLP_OFF_B3 + j], b4 = wf[MLP_OFF_B4];
    const float tg = tid < 32 && i0 + tid < M ? target[i0 + tid] : 0.0f;
    f32x16 z1, z2, z3;
    unsigned short h[16];
#pragma unroll
    for (int v = 0; v < 16; v++) z1[v] = b1;
    __syncthreads();
    z1 = tr_product(xs, GN_XLD, w1, z1, l);
#pragma unroll
    for (int v = 0; v < 16; v++) h[v] = hidden_out(z1[v]);
    tr_put(h, ha, B.h1, i0, j, l);
    tr_weights(wc, wb + MLP_OFF_W3, MLP_HID, j, l);
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 16; v++) z2[v] = b2;
    z2 = tr_product(ha, GN_HLD, wa, z2, l);
#pragma unroll
    for (int v = 0; v < 16; v++) h[v] = hidden_out(z2[v]);
    tr_put(h, hb, B.h2, i0, j, l);
    tr_weights(wa, wbt + MLP_SZ_W2, MLP_HID, j, l);   /* W3 transposed */
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 16; v++) z3[v] = b3;
    z3 = tr_product(hb, GN_HLD, wc, z3, l);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        h[v] = hidden_out(z3[v]);
        const int i = (v >> 2) * 8 + r4 + (v & 3);
        ha[i * GN_HLD + j] = h[v];
        B.h3[(i0 + i) * MLP_HID + j] = h[v];
    }
    __syncthreads();
    if (tid < 32 * GN_HEAD_BLOCKS) {
        const int rr = tid / GN_HEAD_BLOCKS, cb = tid % GN_HEAD_BLOCKS;
        const unsigned short *hr = ha + rr * GN_HLD + cb * MLP_HEAD_BLOCK;
        float p = 0.0f;
#pragma unroll
        for (int e = 0; e < MLP_HEAD_BLOCK; e++) p = fmaf(bf2f(hr[e]), w4s[cb * MLP_HEAD_BLOCK + e], p);
        ps[rr][cb] = p;
    }
    __syncthreads();
    if (tid < 32) {
        float y = b4, dy = 0.0f;
#pragma unroll
        for (int cb = 0; cb < GN_HEAD_BLOCKS; cb++) y += ps[tid][cb];
        if (i0 + tid < M) {
            B.y[i0 + tid] = y;
            dy = 2.0f * (y - tg) / (float)M;
        }
        dys[tid] = B.dy[i0 + tid] = dy;
    }
    __syncthreads();
    float g[16];
    {
        const float w4 = w4s[j];
#pragma unroll
        for (int v = 0; v < 16; v++) {
            g[v] = silu_back(dys[(v >> 2) * 8 + r4 + (v & 3)] * w4, z3[v]);
            h[v] = f2bf(g[v]);
        }
    }
    tr_rows(g, B.df3, i0, j, l);
    tr_put(h, hb, B.dz3, i0, j, l);
    tr_weights(wc, wbt, MLP_HID, j, l);               /* W2 transposed */
    __syncthreads();
    z3 = tr_product(hb, GN_HLD, wa, f32x16{}, l);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        g[v] = silu_back(z3[v], z2[v]);
        h[v] = f2bf(g[v]);
    }
    tr_put(h, ha, B.dz2, i0, j, l);
    tr_rows(g, B.df2, i0, j, l);
    __syncthreads();
    z3 = tr_product(ha, GN_HLD, wc, f32x16{}, l);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        g[v] = silu_back(z3[v], z1[v]);
        h[v] = f2bf(g[v]);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint2 u = make_uint2(h[4 * q] | (unsigned)h[4 * q + 1] << 16, h[4 * q + 2] | (unsigned)h[4 * q + 3] << 16);
        *reinterpret_cast<uint2 *>(B.dz1 + oct_at(i0 + 8 * q + r4, MLP_HID, j)) = u;
    }
    tr_rows(g, B.df1, i0, j, l);
}

/* dW[o][i] = sum_m dZ[m][o] Hin[m][i], a 32 x 32 tile a wave, all rows in
 * one chain of matrix-core steps: the order of the sum is part of the result
 * (parts added up afterwards give other last bits, which Adam's g / |g| turns
 * into other weights).  The chain is 32 cycles a step, 3.4 us of 4000 rows;
 * the loads are what takes longer, so a batch of DW_STEPS is in flight while
 * the one before it is multiplied. */
constexpr int DW_STEPS = 16;

struct DwBatch {
    bf16x8 a[DW_STEPS], b[DW_STEPS];
};

__device__ __forceinline__ void dw_load(DwBatch &t, const unsigned short *pa, const unsigned short *pb, int kin, int m,
                                        int rows)
{
#pragma unroll
    for (int q = 0; q < DW_STEPS; q++) {
        const int64_t mm = min(m + 16 * q, rows - 16);
        t.a[q] = *reinterpret_cast<const bf16x8 *>(pa + mm * MLP_HID);
        t.b[q] = *reinterpret_cast<const bf16x8 *>(pb + mm * kin);
    }
}

__device__ __forceinline__ void dw_tile(const unsigned short *__restrict__ dz, const unsigned short *__restrict__ hin,
                                        int kin, int o0, int c0, int rows, float *__restrict__ out, int l)
{
    const int r = l & 31, half = l >> 5;
    const unsigned short *pa = dz + ((int64_t)half * MLP_HID + o0 + r) * 8;
    const unsigned short *pb = hin + ((int64_t)half * kin + c0 + r) * 8;
    f32x16 acc = {};
    constexpr int BR = 16 * DW_STEPS;
    DwBatch t, u;
    dw_load(t, pa, pb, kin, 0, rows);
    int m = 0;
    for (; m + 2 * BR <= rows; m += 2 * BR) {
        dw_load(u, pa, pb, kin, m + BR, rows);
#pragma unroll
        for (int q = 0; q < DW_STEPS; q++) acc = mfma16(t.a[q], t.b[q], acc);
        dw_load(t, pa, pb, kin, m + 2 * BR, rows);
#pragma unroll
        for (int q = 0; q < DW_STEPS; q++) acc = mfma16(u.a[q], u.b[q], acc);
    }
    /* under two batches are left, the first in t */
    if (m + BR < rows) dw_load(u, pa, pb, kin, m + BR, rows);
#pragma unroll
    for (int q = 0; q < DW_STEPS; q++)
        if (m + 16 * q < rows) acc = mfma16(t.a[q], t.b[q], acc);
    m += BR;
#pragma unroll
    for (int q = 0; q < DW_STEPS; q++)
        if (m + 16 * q < rows) acc = mfma16(u.a[q], u.b[q], acc);
#pragma unroll
    for (int v = 0; v < 16; v++)
        out[(int64_t)(o0 + (v >> 2) * 8 + half * 4 + (v & 3)) * kin + c0 + r] = acc[v];
}

/* the sums of rows [i0, i1) of a column of x (times wt), four row lanes whose
 * sums are added in order; the product is rounded before it is added */
template <class X>
__device__ __forceinline__ float col_part(int i0, int i1, X x)
{
#pragma clang fp contract(off)
    constexpr int U = 8;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int i = i0;
    for (; i + 4 * U <= i1; i += 4 * U) {
        float t[4 * U];
#pragma unroll
        for (int q = 0; q < 4 * U; q++) t[q] = x(i + q);
#pragma unroll
        for (int q = 0; q < 4 * U; q++) s[q & 3] += t[q];
    }
    for (; i < i1; i += 4)
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (i + q < i1) s[q] += x(i + q);
    return ((s[0] + s[1]) + s[2]) + s[3];
}

/* The weight gradients, a tile a workgroup of one wavefront, and beside them
 * the column sums (bias gradients of the FP32 gradients, w4's and b4's), a
 * part of the rows and 64 columns a workgroup, parts in cols.  14.5 us at
 * 4000 rows. */
constexpr int DW_W2 = (MLP_HID / 32) * (MLP_HID / 32), DW_TILES = 2 * DW_W2 + MLP_HID / 32;

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_train_dw(TrainBufs B, int rows, int parts, int chunk)
{
    const int l = threadIdx.x;
    int t = blockIdx.x;
    if (t < DW_TILES) {
        const int o0 = (t & 7) * 32, c0 = (t >> 3 & 7) * 32;
        if (t < DW_W2) dw_tile(B.dz2, B.h1, MLP_HID, o0, c0, rows, B.g + MLP_OFF_W2, l);
        else if (t < 2 * DW_W2) dw_tile(B.dz3, B.h2, MLP_HID, o0, c0, rows, B.g + MLP_OFF_W3, l);
        else dw_tile(B.dz1, B.x, MLP_IN_PAD, o0, 0, rows, B.g + MLP_OFF_W1, l);
        return;
    }
    t -= DW_TILES;
    const int p = t % parts, i0 = p * chunk, i1 = min(rows, i0 + chunk);
    t /= parts;
    const int k = t >> 2, j = (t & 3) * 64 + l;   /* vector, column */
    float *out = B.cols + (int64_t)p * TR_PART;
    if (k < 3) {
        const float *__restrict__ f = (k == 0 ? B.df1 : k == 1 ? B.df2 : B.df3) + j;
        out[k * MLP_HID + j] = col_part(i0, i1, [&](int i) { return f[(int64_t)i * MLP_HID]; });
    } else if (k == 3) {
        const float *__restrict__ dy = B.dy;
        const unsigned short *__restrict__ h = B.h3 + j;
        out[3 * MLP_HID + j] = col_part(i0, i1, [&](int i) {
#pragma clang fp contract(off)
            return dy[i] * bf2f(h[(int64_t)i * MLP_HID]);
        });
    } else if (l == 0) {
        const float *__restrict__ dy = B.dy;
        out[4 * MLP_HID] = col_part(i0, i1, [&](int i) { return dy[i]; });
    }
}

/* Adam on an FP32 master weight */
__device__ __forceinline__ float adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v, float gi,
                                      const AdamStep &A)
{
    const float mi = A.b1 * *m + (1.0f - A.b1) * gi;
    const float vi = A.b2 * *v + (1.0f - A.b2) * gi * gi;
    *m = mi;
    *v = vi;
    return *w = *w - A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
}

/* The column sums from their parts, in order, and with lr > 0 an Adam step on
 * all gradients, refreshing the BF16 copies.  A workgroup takes 256 of the
 * column-summed parameters, or 16 x 16 weights (the transposed copy written
 * through LDS); the weights' are launched only with lr > 0.  5.1 us. */
constexpr int TR_TILES_W1 = (int)(MLP_SZ_W1 / 256), TR_TILES_W2 = (int)(MLP_SZ_W2 / 256);
constexpr int TR_WG_COLS = (TR_COLS + 255) / 256;
__global__ void __launch_bounds__(256)
k_train_apply(TrainBufs B, int parts, AdamStep A)
{
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    int b = blockIdx.x;
    if (b < TR_WG_COLS) {
        const int c = b * 256 + tid;
        if (c >= TR_COLS) return;
        float s = 0.0f;
#pragma unroll 16
        for (int p = 0; p < parts; p++) s += B.cols[(int64_t)p * TR_PART + c];
        const int k = c / MLP_HID;
        const int64_t i = (k == 0 ? MLP_OFF_B1 : k == 1 ? MLP_OFF_B2 : k == 2 ? MLP_OFF_B3 : k == 3 ? MLP_OFF_W4 : MLP_OFF_B4) +
                          c % MLP_HID;
        B.g[i] = s;
        if (A.lr > 0) B.wb[i] = f2bf(adam(B.w + i, B.m + i, B.v + i, s, A));
        return;
    }
    b -= TR_WG_COLS;
    __shared__ unsigned short T[16][17];
    int kin = MLP_IN_PAD;
    int64_t off = MLP_OFF_W1, toff = -1;
    if (b >= TR_TILES_W1) {
        b -= TR_TILES_W1;
        const bool w3 = b >= TR_TILES_W2;
        kin = MLP_HID;
        off = w3 ? MLP_OFF_W3 : MLP_OFF_W2;
        toff = w3 ? MLP_SZ_W2 : 0;
        if (w3) b -= TR_TILES_W2;
    }
    const int o0 = b / (kin / 16) * 16, c0 = b % (kin / 16) * 16;
    const int64_t i = off + (int64_t)(o0 + ty) * kin + c0 + tx;
    const unsigned short nb = f2bf(adam(B.w + i, B.m + i, B.v + i, B.g[i], A));
    B.wb[i] = nb;
    if (toff < 0) return;
    T[ty][tx] = nb;
    __syncthreads();
    B.wbt[toff + (int64_t)(c0 + ty) * MLP_HID + o0 + tx] = T[tx][ty];
}

/* W2 and W3 of wb transposed into wbt */
__global__ void k_train_transpose(const unsigned short *__restrict__ wb, unsigned short *__restrict__ wbt)
{
    const int o = blockIdx.x, i = threadIdx.x;
    wbt[(int64_t)i * MLP_HID + o] = wb[MLP_OFF_W2 + (int64_t)o * MLP_HID + i];
    wbt[MLP_SZ_W2 + (int64_t)i * MLP_HID + o] = wb[MLP_OFF_W3 + (int64_t)o * MLP_HID + i];
}

int launch_train_step(const TrainBufs &B, const float *X, const float *target, int M, const AdamStep &A, hipStream_t s)
{
    const int rows = (M + 31) / 32 * 32, parts = train_parts(rows), chunk = (rows + parts - 1) / parts;
    hipLaunchKernelGGL(k_train_rows, dim3((unsigned)(rows / 32)), dim3(GN_THREADS), 0, s, X, target, M, B);
    NGMI_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_train_dw, dim3((unsigned)(DW_TILES + (4 * 4 + 1) * parts)), dim3(64), 0, s, B, rows, parts, chunk);
    NGMI_HIP(hipGetLastError());
    const unsigned apply = TR_WG_COLS + (A.lr > 0 ? TR_TILES_W1 + 2 * TR_TILES_W2 : 0);
    hipLaunchKernelGGL(k_train_apply, dim3(apply), dim3(256), 0, s, B, parts, A);
    NGMI_HIP(hipGetLastError());
    return NGMI_OK;
}

/* The same network with the weights streamed from L2 per tile instead of
 * held in registers: 4 waves, wave w owning hidden units 64w .. 64w + 63 as
 * two 32-column groups, each group's weights for one layer loaded just
 * before its matrix-core steps.  About 100 VGPRs a lane, so a workgroup
 * fits where one BSIM4 workgroup of the other stream's half finished
 * instead of needing a whole compute unit.  Every output column takes the
 * same matrix-core steps in the same order as in k_guess_net, so both give
 * the same values bit for bit. */
constexpr int GL_THREADS = 256;
static_assert(GL_THREADS / 64 * 64 == MLP_HID, "one wave per 64 hidden units");
static_assert(GL_THREADS == 32 * GN_HEAD_BLOCKS, "one head partial per thread");

template <int STEPS>
__device__ __forceinline__ void gl_layer(const unsigned short *A, int lda, const unsigned short *__restrict__ W,
                                         int ldw, const float *__restrict__ bias, unsigned short *out, int col0,
                                         int l)
{
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const int j = col0 + 32 * g + (l & 31);
        const unsigned short *pw = W + (int64_t)j * ldw + (l >> 5) * 8;
        bf16x8 w[STEPS];
#pragma unroll
        for (int q = 0; q < STEPS; q++) w[q] = *reinterpret_cast<const bf16x8 *>(pw + 16 * q);
        gn_layer(A, lda, w, bias[j], out, col0 + 32 * g, l);
    }
}

__global__ void __launch_bounds__(GL_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_guess_net_lite(const float *__restrict__ X, const unsigned short *__restrict__ wb, const float *__restrict__ wf,
                 int *count, int maxRows, const int64_t *__restrict__ dest, const double2 *__restrict__ base,
                 double *__restrict__ x, float *__restrict__ yout, unsigned long long *rows_total)
{
    __shared__ __align__(16) unsigned short xs[32 * GN_XLD];
    __shared__ __align__(16) unsigned short ha[32 * GN_HLD];
    __shared__ __align__(16) unsigned short hb[32 * GN_HLD];
    __shared__ float w4s[MLP_HID];
    __shared__ float ps[32][GN_HEAD_BLOCKS + 1];
    const int tid = threadIdx.x, l = tid & 63, col0 = (tid >> 6) * 64;
    const int M = count ? min(count[0], maxRows) : maxRows;
    if ((int64_t)blockIdx.x * 32 < M) {
        const float b4 = wf[MLP_OFF_B4];
        for (int e = tid; e < MLP_HID; e += GL_THREADS) w4s[e] = bf2f(wb[MLP_OFF_W4 + e]);
        for (int e = tid; e < 32 * GN_XLD; e += GL_THREADS) xs[e] = 0;   /* the zero columns stay */
        __syncthreads();
        /* this thread's two input elements (rows rr and rr + 16, feature
         * cc), loaded one tile ahead */
        const int rr = tid >> 4, cc = tid & 15;
        const int64_t step = (int64_t)gridDim.x * 32;
        int64_t i0 = (int64_t)blockIdx.x * 32;
        float xa = i0 + rr < M ? X[(i0 + rr) * MLP_IN + cc] : 0.0f;
        float xb = i0 + rr + 16 < M ? X[(i0 + rr + 16) * MLP_IN + cc] : 0.0f;
        for (; i0 < M; i0 += step) {
            xs[rr * GN_XLD + cc] = f2bf(xa);
            xs[(rr + 16) * GN_XLD + cc] = f2bf(xb);
            xa = i0 + step + rr < M ? X[(i0 + step + rr) * MLP_IN + cc] : 0.0f;
            xb = i0 + step + rr + 16 < M ? X[(i0 + step + rr + 16) * MLP_IN + cc] : 0.0f;
            const bool mine = tid < 32 && i0 + tid < M;
            const int64_t d_row = (mine && x) ? dest[i0 + tid] : 0;
            const double2 b_row = (mine && x) ? base[i0 + tid] : make_double2(0.0, 0.0);
            /* the weight pointers made opaque per tile, so the compiler does
             * not hoist every layer's weights out of the loop into registers */
            const unsigned short *wt = wb;
            const float *ft = wf;
            asm volatile("" : "+s"(wt), "+s"(ft));
            __syncthreads();
            gl_layer<MLP_IN_PAD / 16>(xs, GN_XLD, wt + MLP_OFF_W1, MLP_IN_PAD, ft + MLP_OFF_B1, ha, col0, l);
            __syncthreads();
            gl_layer<MLP_HID / 16>(ha, GN_HLD, wt + MLP_OFF_W2, MLP_HID, ft + MLP_OFF_B2, hb, col0, l);
            __syncthreads();
            gl_layer<MLP_HID / 16>(hb, GN_HLD, wt + MLP_OFF_W3, MLP_HID, ft + MLP_OFF_B3, ha, col0, l);
            __syncthreads();
            {
                const int hr = tid / GN_HEAD_BLOCKS, cb = tid % GN_HEAD_BLOCKS;
                const uint4 *h = reinterpret_cast<const uint4 *>(ha + hr * GN_HLD + cb * MLP_HEAD_BLOCK);
                const float *w4 = w4s + cb * MLP_HEAD_BLOCK;
                float p = 0.0f;
#pragma unroll
                for (int q = 0; q < MLP_HEAD_BLOCK / 8; q++) {
                    const uint4 u = h[q];
                    const unsigned int wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        p = fmaf(bf2f((unsigned short)(wd[e] & 0xffffu)), w4[8 * q + 2 * e], p);
                        p = fmaf(bf2f((unsigned short)(wd[e] >> 16)), w4[8 * q + 2 * e + 1], p);
                    }
                }
                ps[hr][cb] = p;
            }
            __syncthreads();
            if (mine) {
                float y = b4;
#pragma unroll
                for (int cb = 0; cb < GN_HEAD_BLOCKS; cb++) y += ps[tid][cb];
                if (yout) yout[i0 + tid] = y;
                if (x) x[d_row] = guess_value(b_row, y);
            }
        }
    }
    if (!count) return;
    __syncthreads();   /* every wave has read count[0] */
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(reinterpret_cast<unsigned int *>(count + 1), 1u) == gridDim.x - 1) {
            if (rows_total) atomicAdd(rows_total, (unsigned long long)M);
            count[0] = 0;
            count[1] = 0;
        }
    }
}

int launch_guess_net(const unsigned short *wb, const float *wf, const float *X, int *count, int maxRows,
                     const int64_t *dest, const double2 *base, double *x, float *yout,
                     unsigned long long *rows_total, hipStream_t s)
{
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        NGMI_HIP(hipGetDevice(&dev));
        NGMI_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        if (cus <= 0) cus = 256;
    }
    /* guess_grid workgroups (each holds a whole compute unit's registers),
     * 0 = one per compute unit: 64 leave the other compute units to the
     * BSIM4 kernel of the other stream's half (measured 0.933x plain
     * against 0.923x with all 256) */
    const int tiles = std::max(1, (maxRows + 31) / 32);
    const int want = tune_get(TUNE_GUESS_GRID);
    if (tune_get(TUNE_GUESS_FUSED) == 2) {
        /* streamed weights: guess_grid small workgroups (0 = one per
         * compute unit) */
        const int grid = std::min(tiles, want > 0 ? want : cus);
        hipLaunchKernelGGL(k_guess_net_lite, dim3((unsigned)grid), dim3(GL_THREADS), 0, s, X, wb, wf, count,
                           maxRows, dest, base, x, yout, rows_total);
        NGMI_HIP(hipGetLastError());
        return NGMI_OK;
    }
    const int grid = std::min(tiles, want > 0 ? want : cus);
    hipLaunchKernelGGL(k_guess_net, dim3((unsigned)grid), dim3(GN_THREADS), 0, s, X, wb, wf, count, maxRows,
                       dest, base, x, yout, rows_total);
    NGMI_HIP(hipGetLastError());
    return NGMI_OK;
}

int launch_gemm_bf16(const unsigned short *A, const unsigned short *B, const float *bias, unsigned short *Cb, int M,
                     int N, int K, hipStream_t s, const int *Mdev)
{
    if (M % 32 || N % 32 || K % 16) {
        set_error("gemm shape %d x %d x %d not a multiple of 32 x 32 x 16", M, N, K);
        return NGMI_E_PARMVAL;
    }
    /* with a device row count the grid is sized to the machine (8 XCDs x
     * 32 CUs x a few waves per tile column) and strides over the tiles */
    const int tiles = Mdev ? std::min(M / 32, 2048) : M / 32;
    hipLaunchKernelGGL(k_gemm_bf16, dim3(N / 32, tiles), dim3(64), 0, s, A, B, bias, Cb, M, N, K, Mdev);
    NGMI_HIP(hipGetLastError());
    return NGMI_OK;
}

}  // namespace ngmi
