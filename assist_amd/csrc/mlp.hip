// Learned IAS15 start: a multilayer perceptron that maps a system's state to the step size
// IAS15 settles on and a warm start for its b coefficients, with its forward pass, backward
// pass and Adam update written here as HIP kernels for gfx950.
//
// Network: 16 inputs (10 used) -> 128 -> 128 -> 128 (tanh) -> 32 outputs (22 used).  Weights
// are kept as an FP32 master copy for the optimizer and BF16 copies for the matrix cores; every
// product runs on v_mfma_f32_16x16x16_bf16 (BF16 operands, FP32 accumulation).  Activations and
// gradients are held in FP32 and rounded to BF16 (nearest even) where they enter a product.
//
// MFMA 16x16x16 BF16 operand layout (one wave): lane l holds A[l % 16][4 (l / 16) + j] and
// B[4 (l / 16) + j][l % 16] for j = 0..3, and receives C[4 (l / 16) + j][l % 16].
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <vector>

#include "../../include/assist.h"

namespace assist_gpu {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// Parameter layout: layer by layer, W[in][out] row-major, then b[out].  The BF16 copy is kept twice,
// in this layout (p16, the operand of the backward products, which reduce over the outputs) and with
// every W transposed to [out][in] (p16t, the operand of the forward products, which reduce over the
// inputs), so that a lane's four consecutive operand elements are one 8-byte read in either direction.
constexpr int kIn = ASSIST_MLP_IN, kHid = ASSIST_MLP_HIDDEN, kOut = ASSIST_MLP_OUT;
constexpr int kOff1 = 0, kOff2 = kOff1 + kIn * kHid + kHid, kOff3 = kOff2 + kHid * kHid + kHid,
              kOff4 = kOff3 + kHid * kHid + kHid, kNumParams = kOff4 + kHid * kOut + kOut;
__device__ __forceinline__ int transposed_pos(int i) {
    const int off = i < kOff2 ? kOff1 : (i < kOff3 ? kOff2 : (i < kOff4 ? kOff3 : kOff4));
    const int K = i < kOff2 ? kIn : kHid, N = i < kOff4 ? kHid : kOut;
    const int e = i - off;
    return e < K * N ? off + (e % N) * K + e / N : i;
}

// Adam (Kingma & Ba 2015) with bias correction; refreshes the BF16 copies of the weights.
__global__ void adam_kernel(float* p, uint16_t* p16, uint16_t* p16t, const float* g, float* m, float* v, int n,
                            float lr, float b1, float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    const uint16_t h = f2bf(pi);
    p16[i] = h;
    p16t[transposed_pos(i)] = h;
}

__global__ void to_bf16_kernel(const float* p, uint16_t* p16, uint16_t* p16t, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint16_t h = f2bf(p[i]);
    p16[i] = h;
    p16t[transposed_pos(i)] = h;
}

// ---- prediction: the four layers fused in one kernel ----------------------------------------
// The forward pass keeps no activations: each wave takes 16 rows at a time
// through all four layers, with the BF16 weights staged once per workgroup in LDS (transposed,
// [out][in], so that a lane's four consecutive inputs of one output are one 8-byte read) and the
// 16 x 128 activation tile in the wave's own LDS area, through which the MFMA result layout
// (four rows of one column per lane) becomes the next operand layout (four columns of one row).
// (LDS rows are padded by 4 elements, 8 bytes: the 16 lanes that read one operand slice then
// fall in distinct banks instead of all in one)
constexpr int kPad = 4;
constexpr int kPW1 = 0, kPW2 = kPW1 + kHid * (kIn + kPad), kPW3 = kPW2 + kHid * (kHid + kPad),
              kPW4 = kPW3 + kHid * (kHid + kPad);
constexpr int kPWords = kPW4 + kOut * (kHid + kPad);  // BF16 weights in LDS
constexpr int kPBias = 3 * kHid + kOut;                 // FP32 biases in LDS
constexpr int kPWaves = 16;  // four waves per SIMD share one copy of the weights
constexpr int kPTileRow = kHid + kPad;
constexpr size_t kPLdsBytes = (size_t)kPWords * 2 + (size_t)kPBias * 4 + (size_t)kPWaves * 16 * kPTileRow * 2;

struct PredictArgs {
    const uint16_t* p16t; // BF16 parameters, weights as [out][in]
    const float* p;       // FP32 parameters (the biases are read from here)
    const float* X;       // [M][16]
    float* Y;             // [M][32]
    int M;
};

// One layer of a 16-row tile: out = act(A W + b) for K = KC * 16 inputs and NT * 16 outputs.
// a[KC]: this lane's operand fragments (row l % 16, inputs 16 kc + 4 (l / 16) + 0..3).
template <int KC, int NT, bool Last>
__device__ __forceinline__ void predict_layer(const bf16x4 (&a)[KC], const uint16_t* Wt, const float* bias,
                                              uint16_t* tile, float* Y, int row0, int M) {
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, q = (lane >> 4) << 2;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        const uint16_t* w = Wt + (size_t)(nt * 16 + r) * (KC * 16 + kPad) + q;
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
            const bf16x4 b = *(const bf16x4*)(w + kc * 16);
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[kc], b, acc, 0, 0, 0);
        }
        const int col = nt * 16 + r;
        const float bc = bias[col];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float v = acc[j] + bc;
            if constexpr (Last) {
                const int row = row0 + q + j;
                if (row < M) Y[(size_t)row * kOut + col] = v;
            } else {
                tile[(q + j) * kPTileRow + col] = f2bf(tanhf(v));
            }
        }
    }
}

__global__ void __launch_bounds__(64 * kPWaves) mlp_predict_kernel(PredictArgs g) {
    extern __shared__ __align__(16) unsigned char s_pred[];
    uint16_t* const sw = (uint16_t*)s_pred;
    float* const sb = (float*)(s_pred + (size_t)kPWords * 2);
    uint16_t* const tiles = (uint16_t*)(s_pred + (size_t)kPWords * 2 + (size_t)kPBias * 4);
    // stage the weights ([out][in]) and the biases
    {
        const int dims[5] = {kIn, kHid, kHid, kHid, kOut};
        const int dst[4] = {kPW1, kPW2, kPW3, kPW4};
        size_t src = 0;
        int boff = 0;
        for (int l = 0; l < 4; l++) {
            const int K = dims[l], N = dims[l + 1];
            for (int i = threadIdx.x * 4; i < K * N; i += blockDim.x * 4) {
                const int n = i / K, k = i - n * K;  // (K is a multiple of 4)
                *(bf16x4*)(sw + dst[l] + n * (K + kPad) + k) = *(const bf16x4*)(g.p16t + src + i);
            }
            src += (size_t)K * N;
            for (int i = threadIdx.x; i < N; i += blockDim.x) sb[boff + i] = g.p[src + i];
            src += N;
            boff += N;
        }
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, q = (lane >> 4) << 2;
    uint16_t* const tile = tiles + (size_t)wave * 16 * kPTileRow;
    const int ntiles = (g.M + 15) >> 4;
    for (int t = blockIdx.x * kPWaves + wave; t < ntiles; t += gridDim.x * kPWaves) {
        const int row0 = t << 4;
        bf16x4 a1[1];
        {
            const int row = row0 + r;
#pragma unroll
            for (int j = 0; j < 4; j++) a1[0][j] = (short)(row < g.M ? f2bf(g.X[(size_t)row * kIn + q + j]) : 0);
        }
        predict_layer<1, kHid / 16, false>(a1, sw + kPW1, sb, tile, nullptr, row0, g.M);
        bf16x4 a[kHid / 16];
        // (LDS operations of one wave complete in order; the fence keeps the compiler's order)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int kc = 0; kc < kHid / 16; kc++) a[kc] = *(const bf16x4*)(tile + r * kPTileRow + kc * 16 + q);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        predict_layer<kHid / 16, kHid / 16, false>(a, sw + kPW2, sb + kHid, tile, nullptr, row0, g.M);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int kc = 0; kc < kHid / 16; kc++) a[kc] = *(const bf16x4*)(tile + r * kPTileRow + kc * 16 + q);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        predict_layer<kHid / 16, kHid / 16, false>(a, sw + kPW3, sb + 2 * kHid, tile, nullptr, row0, g.M);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int kc = 0; kc < kHid / 16; kc++) a[kc] = *(const bf16x4*)(tile + r * kPTileRow + kc * 16 + q);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        predict_layer<kHid / 16, kOut / 16, true>(a, sw + kPW4, sb + 3 * kHid, tile, g.Y, row0, g.M);
    }
}

// ---- training: loss and gradients of a batch in one kernel ------------------------------------
// A workgroup of 8 waves takes 32 rows at a time through the forward pass, the loss and the backward
// pass without leaving the CU: four waves share a 16-row tile and own a quarter of every layer's
// outputs, and the tanh outputs (FP32) stay in their registers until the backward pass needs them.
// Operands change layout through LDS, where each layer's inputs and gradients lie twice: row-major
// (the operand of the products that reduce over inputs or outputs) and transposed with 4 consecutive
// rows per lane (the operand of the weight gradients, which reduce over the rows; the MFMA result
// layout writes it directly).  The weight gradients are 152 tiles of 16 x 16, 19 per wave,
// accumulated in registers over all rows of the workgroup and written once, to the workgroup's own
// slice of a partial-sum buffer that reduce_grad_kernel adds up (no atomics: the sums do not depend
// on the order in which workgroups finish).
// What bounds it: 8192 rows need 2 GFLOP of matrix work, under 2 us of the matrix cores; a workgroup's
// time is its serial chain of 8 layer products (tanh, LDS round trips and barriers, weight fragments
// from L2) and the write of its 157 KB slice.  32 rows per workgroup put 8192 rows on all 256 CUs:
// 39 us for the kernel and 9 us for the sums, against 59 and 6 us with 64 rows (half the CUs) and
// 780 us in 21 launches with one GEMM launch per product, whose weight gradients (one wave per tile,
// 1024 rows each) took 590 us.
constexpr int kTWaves = 8, kTRows = 32;
constexpr int kTSplit = kTWaves / (kTRows / 16);  // waves that share a 16-row tile
constexpr int kTNt = kHid / 16 / kTSplit;         // tiles of 16 outputs a wave owns in a hidden layer
constexpr int kTRow = kHid + kPad;   // elements per row of the row-major tile
constexpr int kTCol = kTRows + kPad; // elements per column of the transposed tiles
constexpr int kTBias = 3 * kHid + kOut;
constexpr int kPartStride = kNumParams + 4;  // a workgroup's gradients, then its loss
constexpr int kTMaxBlocks = 256;

struct TrainArgs {
    const uint16_t* p16;   // BF16 parameters, weights as [in][out]
    const uint16_t* p16t;  // weights as [out][in]
    const float* p;
    const float* X;        // [M][16]
    const float* T;        // [M][32]
    const float* w;        // [32]
    float* part;           // [gridDim.x][kPartStride]
    int M;
};

// Operand fragments of NT tiles of 16 output columns, from W stored with the reduction contiguous.
template <int KC, int NT>
__device__ __forceinline__ void load_frags(const uint16_t* W, int col0, bf16x4 (&b)[NT][KC]) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = (lane >> 4) << 2;
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int kc = 0; kc < KC; kc++)
            b[nt][kc] = *(const bf16x4*)(W + (size_t)(col0 + nt * 16 + r) * (KC * 16) + kc * 16 + q);
}
// acc = A B over KC slices of 16, A from the row-major tile (rows row0..row0+15).
template <int KC, int NT>
__device__ __forceinline__ void tile_product(const uint16_t* tile, int row0, const bf16x4 (&b)[NT][KC], f32x4 (&acc)[NT]) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = (lane >> 4) << 2;
    bf16x4 a[KC];
#pragma unroll
    for (int kc = 0; kc < KC; kc++) a[kc] = *(const bf16x4*)(tile + (row0 + r) * kTRow + kc * 16 + q);
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < KC; kc++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[kc], b[nt][kc], acc[nt], 0, 0, 0);
}
// acc[i] += In^T D for the 16 inputs at in0 and the 16-column tiles out0 + 16 i, over the rows.
template <int NT>
__device__ __forceinline__ void weight_grad(const uint16_t* inT, int in0, const uint16_t* dT, int out0, f32x4 (&acc)[NT]) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = (lane >> 4) << 2;
#pragma unroll
    for (int kc = 0; kc < kTRows / 16; kc++) {
        const bf16x4 a = *(const bf16x4*)(inT + (in0 + r) * kTCol + kc * 16 + q);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const bf16x4 b = *(const bf16x4*)(dT + (out0 + nt * 16 + r) * kTCol + kc * 16 + q);
            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[nt], 0, 0, 0);
        }
    }
}
// A wave's columns col0.. of its 16-row tile: to the row-major tile and / or transposed.
template <int NT>
__device__ __forceinline__ void put_rows(uint16_t* tile, int row0, int col0, const f32x4 (&v)[NT]) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = (lane >> 4) << 2;
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int j = 0; j < 4; j++) tile[(row0 + q + j) * kTRow + col0 + nt * 16 + r] = f2bf(v[nt][j]);
}
template <int NT>
__device__ __forceinline__ void put_cols(uint16_t* tileT, int row0, int col0, const f32x4 (&v)[NT]) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = (lane >> 4) << 2;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        bf16x4 h;
#pragma unroll
        for (int j = 0; j < 4; j++) h[j] = (short)f2bf(v[nt][j]);
        *(bf16x4*)(tileT + (col0 + nt * 16 + r) * kTCol + row0 + q) = h;
    }
}
// Gradient through tanh from its output H, and this lane's share of the bias gradients.
__device__ __forceinline__ void tanh_grad(f32x4 (&d)[kTNt], const f32x4 (&H)[kTNt], float (&db)[kTNt]) {
#pragma unroll
    for (int nt = 0; nt < kTNt; nt++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            d[nt][j] *= 1.f - H[nt][j] * H[nt][j];
            db[nt] += d[nt][j];
        }
}
__device__ __forceinline__ void tanh_layer(f32x4 (&H)[kTNt], const float* bias, int col0) {
    const int r = threadIdx.x & 15;
#pragma unroll
    for (int nt = 0; nt < kTNt; nt++) {
        const float bc = bias[col0 + nt * 16 + r];
#pragma unroll
        for (int j = 0; j < 4; j++) H[nt][j] = tanhf(H[nt][j] + bc);
    }
}

__global__ void __launch_bounds__(64 * kTWaves) mlp_train_kernel(TrainArgs args) {
    __shared__ __align__(16) uint16_t s_tile[kTRows * kTRow];
    __shared__ __align__(16) uint16_t s_inT[kHid * kTCol], s_dT[kHid * kTCol], s_xT[kIn * kTCol];
    __shared__ float s_loss[kTWaves];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, q = (lane >> 4) << 2;
    const int row0 = wave / kTSplit * 16, share = wave % kTSplit, col0 = share * kTNt * 16;
    const bool outs = share < kOut / 16;  // this wave owns a tile of the output layer
    f32x4 gw1[1] = {}, gw2[8] = {}, gw3[8] = {}, gw4[2] = {};
    float db1[kTNt] = {}, db2[kTNt] = {}, db3[kTNt] = {}, db4 = 0.f, loss = 0.f;
    TrainArgs g = args;
    for (int base = blockIdx.x * kTRows; base < args.M; base += gridDim.x * kTRows) {
        // (opaque per trip: the weight fragments are the same for every 32 rows, and hoisted out of
        // the loop they would not fit the registers)
        int zero = 0;
        asm volatile("" : "+s"(zero));
        g.p16 = args.p16 + zero;
        g.p16t = args.p16t + zero;
        g.p = args.p + zero;
        f32x4 H1[kTNt], H2[kTNt], H3[kTNt];
        {
            const int row = base + row0 + r;
            bf16x4 a;
#pragma unroll
            for (int j = 0; j < 4; j++) a[j] = (short)(row < g.M ? f2bf(g.X[(size_t)row * kIn + q + j]) : 0);
            bf16x4 b[kTNt][1];
            load_frags<1, kTNt>(g.p16t + kOff1, col0, b);
            if (share == 0) {
#pragma unroll
                for (int j = 0; j < 4; j++) s_xT[(q + j) * kTCol + row0 + r] = (uint16_t)a[j];
            }
#pragma unroll
            for (int nt = 0; nt < kTNt; nt++)
                H1[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[nt][0], (f32x4{0.f, 0.f, 0.f, 0.f}), 0, 0, 0);
        }
        tanh_layer(H1, g.p + kOff1 + kIn * kHid, col0);
        put_rows(s_tile, row0, col0, H1);
        {
            bf16x4 b[kTNt][8];
            load_frags<8, kTNt>(g.p16t + kOff2, col0, b);
            __syncthreads();
            tile_product<8, kTNt>(s_tile, row0, b, H2);
        }
        tanh_layer(H2, g.p + kOff2 + kHid * kHid, col0);
        __syncthreads();
        put_rows(s_tile, row0, col0, H2);
        {
            bf16x4 b[kTNt][8];
            load_frags<8, kTNt>(g.p16t + kOff3, col0, b);
            __syncthreads();
            tile_product<8, kTNt>(s_tile, row0, b, H3);
        }
        tanh_layer(H3, g.p + kOff3 + kHid * kHid, col0);
        __syncthreads();
        put_rows(s_tile, row0, col0, H3);
        put_cols(s_inT, row0, col0, H3);
        // output layer and loss: dY = 2 w (Y - T) / M (0 past the batch)
        f32x4 dY[1] = {};
        __syncthreads();
        if (outs) {
            bf16x4 b[1][8];
            load_frags<8, 1>(g.p16t + kOff4, share * 16, b);
            tile_product<8, 1>(s_tile, row0, b, dY);
            const int col = share * 16 + r;
            const float bc = g.p[kOff4 + kHid * kOut + col], wc = g.w[col];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = base + row0 + q + j;
                float d = 0.f;
                if (row < g.M) d = (dY[0][j] + bc) - g.T[(size_t)row * kOut + col];
                loss += wc * d * d;
                dY[0][j] = 2.f * wc * d / (float)g.M;
                db4 += dY[0][j];
            }
        }
        __syncthreads();
        // backward: the layers' gradients with respect to their pre-activations replace the tile
        f32x4 D[kTNt];
        if (outs) {
            put_rows(s_tile, row0, share * 16, dY);
            put_cols(s_dT, row0, share * 16, dY);
        }
        {
            bf16x4 b[kTNt][2];
            load_frags<2, kTNt>(g.p16 + kOff4, col0, b);
            __syncthreads();
            tile_product<2, kTNt>(s_tile, row0, b, D);
        }
        weight_grad<2>(s_inT, wave * 16, s_dT, 0, gw4);
        tanh_grad(D, H3, db3);
        __syncthreads();
        put_rows(s_tile, row0, col0, D);
        put_cols(s_dT, row0, col0, D);
        put_cols(s_inT, row0, col0, H2);
        {
            bf16x4 b[kTNt][8];
            load_frags<8, kTNt>(g.p16 + kOff3, col0, b);
            __syncthreads();
            tile_product<8, kTNt>(s_tile, row0, b, D);
        }
        weight_grad<8>(s_inT, wave * 16, s_dT, 0, gw3);
        tanh_grad(D, H2, db2);
        __syncthreads();
        put_rows(s_tile, row0, col0, D);
        put_cols(s_dT, row0, col0, D);
        put_cols(s_inT, row0, col0, H1);
        {
            bf16x4 b[kTNt][8];
            load_frags<8, kTNt>(g.p16 + kOff2, col0, b);
            __syncthreads();
            tile_product<8, kTNt>(s_tile, row0, b, D);
        }
        weight_grad<8>(s_inT, wave * 16, s_dT, 0, gw2);
        tanh_grad(D, H1, db1);
        __syncthreads();
        put_cols(s_dT, row0, col0, D);
        __syncthreads();
        weight_grad<1>(s_xT, 0, s_dT, wave * 16, gw1);
        __syncthreads();
    }
    // this workgroup's sums
    float* const out = args.part + (size_t)blockIdx.x * kPartStride;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        out[kOff1 + (q + j) * kHid + wave * 16 + r] = gw1[0][j];
        const int in = wave * 16 + q + j;
#pragma unroll
        for (int nt = 0; nt < 8; nt++) {
            out[kOff2 + in * kHid + nt * 16 + r] = gw2[nt][j];
            out[kOff3 + in * kHid + nt * 16 + r] = gw3[nt][j];
        }
#pragma unroll
        for (int nt = 0; nt < 2; nt++) out[kOff4 + in * kOut + nt * 16 + r] = gw4[nt][j];
    }
    // bias gradients: over a tile's rows by lane exchange, over the two tiles through LDS
    float* const s_db = (float*)s_inT;  // [kTRows / 16][kTBias]
    auto put_bias = [&](float v, int at) {
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (lane < 16) s_db[wave / kTSplit * kTBias + at + r] = v;
    };
#pragma unroll
    for (int nt = 0; nt < kTNt; nt++) {
        put_bias(db1[nt], col0 + nt * 16);
        put_bias(db2[nt], kHid + col0 + nt * 16);
        put_bias(db3[nt], 2 * kHid + col0 + nt * 16);
    }
    if (outs) put_bias(db4, 3 * kHid + share * 16);
    for (int m = 32; m >= 1; m >>= 1) loss += __shfl_xor(loss, m, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();
    for (int i = threadIdx.x; i < kTBias; i += blockDim.x) {
        const int l = i >> 7, c = i & 127;
        const int at = l == 0 ? kOff2 - kHid : (l == 1 ? kOff3 - kHid : (l == 2 ? kOff4 - kHid : kNumParams - kOut));
        float v = s_db[i];
        for (int k = 1; k < kTRows / 16; k++) v += s_db[k * kTBias + i];
        out[at + c] = v;
    }
    if (threadIdx.x == 0) {
        float t = 0.f;
        for (int k = 0; k < kTWaves; k++) t += s_loss[k];
        out[kNumParams] = t;
    }
}

// Gradients and loss from the workgroups' sums: 64 groups of four parameters per block, each
// summed by four waves that take every fourth workgroup's slice (the slices stream from L2; one
// thread per group alone would leave the loads of up to 256 slices in a chain).
__global__ void __launch_bounds__(256) reduce_grad_kernel(const float* __restrict__ part, int nblocks, int M, float* grad,
                                                          float* loss) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = (blockIdx.x * 64 + lane) * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (e < kPartStride) {
#pragma unroll 8
        for (int b = wave; b < nblocks; b += 4) s += *(const f32x4*)(part + (size_t)b * kPartStride + e);
    }
    __shared__ f32x4 acc[4][64];
    acc[wave][lane] = s;
    __syncthreads();
    if (wave != 0) return;
    s = (acc[0][lane] + acc[1][lane]) + (acc[2][lane] + acc[3][lane]);
    if (e < kNumParams) *(f32x4*)(grad + e) = s;
    else if (e == kNumParams) *loss = s[0] / (float)M;
}

}  // namespace assist_gpu

using namespace assist_gpu;

// ------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------
namespace {

constexpr int kLayers = 4;
constexpr int kDims[kLayers + 1] = {ASSIST_MLP_IN, ASSIST_MLP_HIDDEN, ASSIST_MLP_HIDDEN, ASSIST_MLP_HIDDEN, ASSIST_MLP_OUT};

size_t w_off(int l) {
    size_t o = 0;
    for (int i = 0; i < l; i++) o += (size_t)kDims[i] * kDims[i + 1] + kDims[i + 1];
    return o;
}

bool ok(hipError_t e, const char* what) {
    if (e == hipSuccess) return true;
    fprintf(stderr, "(ASSIST) HIP error in %s: %s\n", what, hipGetErrorString(e));
    return false;
}

unsigned grid1(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

struct assist_mlp {
    int device = 0;
    int max_batch = 0;
    float* p = nullptr;      // FP32 master parameters
    uint16_t* p16 = nullptr; // BF16 weights for the matrix cores, [in][out]
    uint16_t* p16t = nullptr; // and [out][in]
    float* g = nullptr;      // gradients
    float* m = nullptr;      // Adam moments
    float* v = nullptr;
    float* part = nullptr;   // gradients and loss per workgroup of the training kernel
    float* wout = nullptr;   // output weights of the loss [out]
    float* loss = nullptr;   // [1]
};

static void mlp_release(assist_mlp* n) {
    if (!n) return;
    for (void* q : {(void*)n->p, (void*)n->p16, (void*)n->p16t, (void*)n->g, (void*)n->m, (void*)n->v, (void*)n->part,
                    (void*)n->wout, (void*)n->loss})
        if (q) (void)hipFree(q);
    delete n;
}

// Workgroups of the training kernel for M rows.
static int train_blocks(int M) {
    const int b = (M + kTRows - 1) / kTRows;
    return b < kTMaxBlocks ? b : kTMaxBlocks;
}

extern "C" {

int assist_mlp_num_params(void) { return (int)w_off(kLayers); }

struct assist_mlp* assist_mlp_create(int max_batch, unsigned long long seed) {
    if (max_batch <= 0) return nullptr;
    auto* n = new assist_mlp();
    n->max_batch = max_batch;
    const size_t np = w_off(kLayers);
    const size_t O = ASSIST_MLP_OUT;
    bool good = ok(hipGetDevice(&n->device), "hipGetDevice") && ok(hipMalloc(&n->p, np * 4), "hipMalloc") &&
                ok(hipMalloc(&n->p16, np * 2), "hipMalloc") && ok(hipMalloc(&n->p16t, np * 2), "hipMalloc") &&
                ok(hipMalloc(&n->g, np * 4), "hipMalloc") &&
                ok(hipMalloc(&n->m, np * 4), "hipMalloc") && ok(hipMalloc(&n->v, np * 4), "hipMalloc") &&
                ok(hipMalloc(&n->part, (size_t)train_blocks(max_batch) * kPartStride * 4), "hipMalloc") &&
                ok(hipMalloc(&n->wout, O * 4), "hipMalloc") &&
                ok(hipMalloc(&n->loss, 4), "hipMalloc");
    if (!good) {
        mlp_release(n);
        return nullptr;
    }
    // Glorot-uniform weights from a 64-bit LCG, zero biases.
    std::vector<float> h(np, 0.f);
    unsigned long long st = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    for (int l = 0; l < kLayers; l++) {
        const double lim = sqrt(6.0 / (kDims[l] + kDims[l + 1]));
        for (size_t i = 0; i < (size_t)kDims[l] * kDims[l + 1]; i++) {
            st = st * 6364136223846793005ULL + 1442695040888963407ULL;
            const double u = (double)(st >> 11) * (1.0 / 9007199254740992.0);
            h[w_off(l) + i] = (float)((2.0 * u - 1.0) * lim);
        }
    }
    std::vector<float> ones(O, 1.f);
    if (assist_mlp_set_params(n, h.data()) != 0 || !ok(hipMemcpy(n->wout, ones.data(), O * 4, hipMemcpyHostToDevice), "hipMemcpy")) {
        mlp_release(n);
        return nullptr;
    }
    return n;
}

void assist_mlp_free(struct assist_mlp* n) { mlp_release(n); }

int assist_mlp_max_batch(const struct assist_mlp* n) { return n ? n->max_batch : 0; }

int assist_mlp_set_params(struct assist_mlp* n, const float* host) {
    if (!n || !host) return ASSIST_BATCH_ERROR_ARG;
    const size_t np = w_off(kLayers);
    if (!ok(hipMemcpy(n->p, host, np * 4, hipMemcpyHostToDevice), "hipMemcpy") ||
        !ok(hipMemset(n->m, 0, np * 4), "hipMemset") || !ok(hipMemset(n->v, 0, np * 4), "hipMemset"))
        return ASSIST_BATCH_ERROR_DEVICE;
    hipLaunchKernelGGL(to_bf16_kernel, dim3(grid1(np)), dim3(256), 0, 0, n->p, n->p16, n->p16t, (int)np);
    if (!ok(hipGetLastError(), "to_bf16") || !ok(hipDeviceSynchronize(), "to_bf16")) return ASSIST_BATCH_ERROR_DEVICE;
    return 0;
}

int assist_mlp_get_params(const struct assist_mlp* n, float* host) {
    if (!n || !host) return ASSIST_BATCH_ERROR_ARG;
    return ok(hipMemcpy(host, n->p, w_off(kLayers) * 4, hipMemcpyDeviceToHost), "hipMemcpy") ? 0 : ASSIST_BATCH_ERROR_DEVICE;
}

int assist_mlp_set_output_weights(struct assist_mlp* n, const float* host_w) {
    if (!n || !host_w) return ASSIST_BATCH_ERROR_ARG;
    return ok(hipMemcpy(n->wout, host_w, ASSIST_MLP_OUT * 4, hipMemcpyHostToDevice), "hipMemcpy") ? 0
                                                                                              : ASSIST_BATCH_ERROR_DEVICE;
}

// Forward pass of any number of rows: d_X [M][16] -> d_Y [M][32].
int assist_mlp_predict(struct assist_mlp* n, const float* d_X, int M, float* d_Y, void* stream) {
    if (!n || !d_X || !d_Y || M < 0) return ASSIST_BATCH_ERROR_ARG;
    if (M == 0) return 0;
    if (!ok(hipFuncSetAttribute((const void*)mlp_predict_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)kPLdsBytes),
            "hipFuncSetAttribute(mlp_predict)"))
        return ASSIST_BATCH_ERROR_DEVICE;
    int dev = 0, ncu = 0;
    if (!ok(hipGetDevice(&dev), "hipGetDevice") ||
        !ok(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute"))
        return ASSIST_BATCH_ERROR_DEVICE;
    PredictArgs g;
    g.p16t = n->p16t;
    g.p = n->p;
    g.X = d_X;
    g.Y = d_Y;
    g.M = M;
    // one workgroup per CU (the staged weights and 16 activation tiles fill its LDS), or fewer
    // for small batches
    const int tiles = (M + 15) / 16;
    int blocks = (tiles + kPWaves - 1) / kPWaves;
    if (blocks > ncu) blocks = ncu;
    hipLaunchKernelGGL(mlp_predict_kernel, dim3(blocks), dim3(64 * kPWaves), kPLdsBytes, (hipStream_t)stream, g);
    return ok(hipGetLastError(), "mlp predict") ? 0 : ASSIST_BATCH_ERROR_DEVICE;
}

// Forward pass of at most max_batch rows (the same kernel; nothing to do without an output).
int assist_mlp_forward(struct assist_mlp* n, const float* d_X, int M, float* d_Y, void* stream) {
    if (!n || !d_X || M < 0 || M > n->max_batch) return ASSIST_BATCH_ERROR_ARG;
    return d_Y ? assist_mlp_predict(n, d_X, M, d_Y, stream) : 0;
}

// Forward and backward pass of the weighted squared error against d_T [M][32]; leaves the
// gradients in the network (and copies them to host_grad when given) and returns the loss.
int assist_mlp_loss_grad(struct assist_mlp* n, const float* d_X, const float* d_T, int M, float* loss,
                         float* host_grad, void* stream) {
    if (!n || !d_X || !d_T || M <= 0 || M > n->max_batch) return ASSIST_BATCH_ERROR_ARG;
    hipStream_t s = (hipStream_t)stream;
    TrainArgs g;
    g.p16 = n->p16;
    g.p16t = n->p16t;
    g.p = n->p;
    g.X = d_X;
    g.T = d_T;
    g.w = n->wout;
    g.part = n->part;
    g.M = M;
    const int blocks = train_blocks(M);
    hipLaunchKernelGGL(mlp_train_kernel, dim3(blocks), dim3(64 * kTWaves), 0, s, g);
    if (!ok(hipGetLastError(), "mlp train")) return ASSIST_BATCH_ERROR_DEVICE;
    hipLaunchKernelGGL(reduce_grad_kernel, dim3((kPartStride / 4 + 63) / 64), dim3(256), 0, s, (const float*)n->part,
                       blocks, M, n->g, n->loss);
    if (!ok(hipGetLastError(), "mlp reduce")) return ASSIST_BATCH_ERROR_DEVICE;
    if (loss && !ok(hipMemcpyAsync(loss, n->loss, 4, hipMemcpyDeviceToHost, s), "hipMemcpyAsync")) return ASSIST_BATCH_ERROR_DEVICE;
    if (host_grad && !ok(hipMemcpyAsync(host_grad, n->g, (size_t)kNumParams * 4, hipMemcpyDeviceToHost, s), "hipMemcpyAsync"))
        return ASSIST_BATCH_ERROR_DEVICE;
    if (!ok(hipStreamSynchronize(s), "mlp backward")) return ASSIST_BATCH_ERROR_DEVICE;
    return 0;
}

int assist_mlp_adam_step(struct assist_mlp* n, float lr, float beta1, float beta2, float eps, int step, void* stream) {
    if (!n || step < 1) return ASSIST_BATCH_ERROR_ARG;
    const size_t np = w_off(kLayers);
    const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(grid1(np)), dim3(256), 0, (hipStream_t)stream, n->p, n->p16, n->p16t,
                       (const float*)n->g, n->m, n->v, (int)np, lr, beta1, beta2, eps, c1, c2);
    return ok(hipGetLastError(), "adam") ? 0 : ASSIST_BATCH_ERROR_DEVICE;
}

}  // extern "C"
