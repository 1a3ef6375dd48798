// rp_mlp.hip -- the network of the learned candidate ordering (no counterpart in the reference).
//
// A multilayer perceptron 12 -> 64 -> 64 -> 64 -> 1 with GELU hidden units (the tanh form) and a sigmoid output
// predicts, from the pose of a candidate relative to a trial pose (position in the trial body frame divided by the
// total interaction range, and the relative rotation matrix), the probability that the exact overlap test finds an
// overlap.  The sweep's exact test stays the judge; the scores only order the candidates.
//
//   * training (FP32): one kernel for the hidden layers forward, the output head with the binary cross-entropy, one
//     kernel for the hidden layers backward, the weight gradients as sums over parts of the batch, and Adam;
//   * inference (BF16 MFMA, FP32 accumulation): one wavefront per 16 pairs, v_mfma_f32_16x16x16bf16 tiles for the
//     three hidden layers, the output as a dot product of the last hidden layer with the head weights.
//
// Parameters, FP32, one array (MLP_PARAMS floats): W1 [64][12], b1 [64], W2 [64][64], b2 [64], W3 [64][64], b3 [64],
// w4 [64], b4.
#include "rp_mlp.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

namespace rp {

namespace {

constexpr int WAVE = 64;

__device__ __forceinline__ float gelu(float x) {
    const float c = 0.7978845608028654f;  // sqrt(2 / pi)
    const float t = tanhf(c * (x + 0.044715f * x * x * x));
    return 0.5f * x * (1.f + t);
}

__device__ __forceinline__ float gelu_grad(float x) {
    const float c = 0.7978845608028654f;
    const float t = tanhf(c * (x + 0.044715f * x * x * x));
    return 0.5f * (1.f + t) + 0.5f * x * (1.f - t * t) * c * (1.f + 3.f * 0.044715f * x * x);
}

// The gradient's matrix work in FP32.  A workgroup has ROWS samples and 16 threads per sample, each with four of the 64
// units of a layer; a layer's weights are staged in LDS with the four units adjacent, and every sum runs over the inputs in
// order.  The three hidden layers of a pass run in one launch, their activations between layers in LDS.
constexpr int ROWS = 16;
constexpr int GRAD_THREADS = 16 * ROWS;

// acc[j] += sum_i in[i] w[i][4 q + j], w [n][64] in LDS
__device__ __forceinline__ void grad_layer(const float *w, const float *in, int n, int q, float acc[4]) {
    const float4 *w4 = reinterpret_cast<const float4 *>(w) + q;
#pragma unroll 4
    for (int i = 0; i < n; i++) {
        const float v = in[i];
        const float4 c = w4[16 * i];
        acc[0] = fmaf(c.x, v, acc[0]);
        acc[1] = fmaf(c.y, v, acc[1]);
        acc[2] = fmaf(c.z, v, acc[2]);
        acc[3] = fmaf(c.w, v, acc[3]);
    }
}

// Hidden layers forward: a_l[s][o] = gelu(pre_l[s][o]), pre_l[s][o] = b[o] + sum_i W[o][i] in[s][i] (kept for the
// backward pass).
__global__ __launch_bounds__(GRAD_THREADS) void k_mlp_forward(const float *__restrict__ x,
                                                              const float *__restrict__ theta, int B, MlpWork w) {
    __shared__ __attribute__((aligned(16))) float sW[MLP_H * MLP_H];  // W[o][i] at i * 64 + o
    __shared__ float sIn[ROWS * (MLP_H + 1)];
    const int tid = threadIdx.x, r = tid / 16, q = tid % 16;
    const int s = (int)blockIdx.x * ROWS + r;
    for (int e = tid; e < ROWS * MLP_IN; e += GRAD_THREADS) {
        const int row = e / MLP_IN, i = e - row * MLP_IN, at = (int)blockIdx.x * ROWS + row;
        sIn[row * (MLP_H + 1) + i] = at < B ? x[(size_t)at * MLP_IN + i] : 0.f;
    }
    for (int layer = 0; layer < 3; layer++) {
        const int n = layer == 0 ? MLP_IN : MLP_H;
        const float *W = theta + (layer == 0 ? MLP_OFF_W1 : layer == 1 ? MLP_OFF_W2 : MLP_OFF_W3);
        const float *bias = theta + (layer == 0 ? MLP_OFF_B1 : layer == 1 ? MLP_OFF_B2 : MLP_OFF_B3);
        float *pre = layer == 0 ? w.pre1 : layer == 1 ? w.pre2 : w.pre3;
        float *act = layer == 0 ? w.a1 : layer == 1 ? w.a2 : w.a3;
        for (int e = tid; e < MLP_H * n; e += GRAD_THREADS) {
            const int i = e / MLP_H, o = e - i * MLP_H;
            sW[e] = W[o * n + i];
        }
        __syncthreads();
        float acc[4], a[4];
        for (int j = 0; j < 4; j++) acc[j] = bias[4 * q + j];
        grad_layer(sW, sIn + r * (MLP_H + 1), n, q, acc);
        for (int j = 0; j < 4; j++) a[j] = gelu(acc[j]);
        // (the work arrays are not aligned beyond a float)
        for (int j = 0; j < 4 && s < B; j++) {
            pre[(size_t)s * MLP_H + 4 * q + j] = acc[j];
            act[(size_t)s * MLP_H + 4 * q + j] = a[j];
        }
        __syncthreads();  // every thread has read sIn and sW
        for (int j = 0; j < 4; j++) sIn[r * (MLP_H + 1) + 4 * q + j] = a[j];
    }
}

// Output head: z = b4 + w4 . h, p = sigmoid(z), dz = (p - y) / B; the batch's binary cross-entropy summed per block
// in a fixed order into lossPart[block].
__global__ __launch_bounds__(256) void k_mlp_head(const float *__restrict__ h, const float *__restrict__ theta,
                                                  const float *__restrict__ y, int B, float *dz, float *lossPart) {
    __shared__ float sLoss[256];
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (s < B) {
        float z = theta[MLP_OFF_B4];
        for (int j = 0; j < MLP_H; j++) z += theta[MLP_OFF_W4 + j] * h[s * MLP_H + j];
        const float p = 1.f / (1.f + expf(-z));
        dz[s] = (p - y[s]) / (float)B;
        // log(1 + exp(-|z|)) form: y log p + (1 - y) log(1 - p) without cancellation
        l = fmaxf(z, 0.f) - z * y[s] + log1pf(expf(-fabsf(z)));
    }
    sLoss[threadIdx.x] = l;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sLoss[threadIdx.x] += sLoss[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) lossPart[blockIdx.x] = sLoss[0];
}

// Hidden layers backward: d3[s][i] = dz[s] w4[i] gelu'(pre3[s][i]), then d[s][i] = (sum_o W[o][i] d'[s][o]) gelu'(pre[s][i]).
__global__ __launch_bounds__(GRAD_THREADS) void k_mlp_backward(const float *__restrict__ theta, int B, MlpWork w) {
    __shared__ __attribute__((aligned(16))) float sW[MLP_H * MLP_H];  // W[o][i] at o * 64 + i, as stored
    __shared__ float sIn[ROWS * (MLP_H + 1)];
    const int tid = threadIdx.x, r = tid / 16, q = tid % 16;
    const int s = (int)blockIdx.x * ROWS + r;
    for (int layer = 2; layer >= 0; layer--) {
        const float *pre = layer == 2 ? w.pre3 : layer == 1 ? w.pre2 : w.pre1;
        float *delta = layer == 2 ? w.d3 : layer == 1 ? w.d2 : w.d1;
        float d[4] = {0.f, 0.f, 0.f, 0.f};
        if (layer == 2) {
            const float dz = s < B ? w.dz[s] : 0.f;
            for (int j = 0; j < 4; j++) d[j] = theta[MLP_OFF_W4 + 4 * q + j] * dz;
        } else {
            const float *W = theta + (layer == 1 ? MLP_OFF_W3 : MLP_OFF_W2);
            for (int e = tid; e < MLP_H * MLP_H; e += GRAD_THREADS) sW[e] = W[e];
            __syncthreads();
            grad_layer(sW, sIn + r * (MLP_H + 1), MLP_H, q, d);
            __syncthreads();  // every thread has read sIn and sW
        }
        for (int j = 0; j < 4 && s < B; j++) {
            d[j] *= gelu_grad(pre[(size_t)s * MLP_H + 4 * q + j]);
            delta[(size_t)s * MLP_H + 4 * q + j] = d[j];
        }
        for (int j = 0; j < 4; j++) sIn[r * (MLP_H + 1) + 4 * q + j] = d[j];
    }
}

// Weight gradients gW[o][i] = sum_s delta[s][o] act[s][i] and gb[o] = sum_s delta[s][o] of all four layers (blockIdx.y),
// over the samples of one of `splits` parts (blockIdx.x): a thread has four units o and four inputs i (the biases: their
// first thread per o), the part's samples pass through LDS GRAD_TILE at a time.  part: the parts' sums, MLP_PARAMS floats
// apart in the gradient's own layout (the gradient itself for a single part).  The sums over all samples by one thread
// per weight that this replaces took 1.6 ms per layer at 4096 samples.
constexpr int GRAD_TILE = 32;
__global__ __launch_bounds__(256) void k_mlp_wgrad(const float *__restrict__ x, int B, int splits, MlpWork w, float *part) {
    __shared__ __attribute__((aligned(16))) float sD[GRAD_TILE * MLP_H], sA[GRAD_TILE * MLP_H];
    const int tid = threadIdx.x, layer = blockIdx.y, split = blockIdx.x;
    const int first = (int)((long long)B * split / splits), last = (int)((long long)B * (split + 1) / splits);
    const int nout = layer == 3 ? 1 : MLP_H, nin = layer == 0 ? MLP_IN : MLP_H;
    const float *delta = layer == 0 ? w.d1 : layer == 1 ? w.d2 : layer == 2 ? w.d3 : w.dz;
    const float *act = layer == 0 ? x : layer == 1 ? w.a1 : layer == 2 ? w.a2 : w.a3;
    const int offW = layer == 0 ? MLP_OFF_W1 : layer == 1 ? MLP_OFF_W2 : layer == 2 ? MLP_OFF_W3 : MLP_OFF_W4;
    const int offB = layer == 0 ? MLP_OFF_B1 : layer == 1 ? MLP_OFF_B2 : layer == 2 ? MLP_OFF_B3 : MLP_OFF_B4;
    const int o0 = 4 * (tid / 16), i0 = 4 * (tid % 16);
    float acc[4][4] = {}, bias[4] = {};
    for (int t0 = first; t0 < last; t0 += GRAD_TILE) {
        const int rows = min(GRAD_TILE, last - t0);
        __syncthreads();  // the previous tile has been read
        for (int e = tid; e < GRAD_TILE * MLP_H; e += 256) {
            const int s = e / MLP_H, c = e - s * MLP_H;
            sD[e] = s < rows && c < nout ? delta[(size_t)(t0 + s) * nout + c] : 0.f;
            sA[e] = s < rows && c < nin ? act[(size_t)(t0 + s) * nin + c] : 0.f;
        }
        __syncthreads();
        for (int s = 0; s < rows; s++) {
            const float4 d = *reinterpret_cast<const float4 *>(sD + s * MLP_H + o0);
            const float4 a = *reinterpret_cast<const float4 *>(sA + s * MLP_H + i0);
            const float dv[4] = {d.x, d.y, d.z, d.w}, av[4] = {a.x, a.y, a.z, a.w};
            for (int j = 0; j < 4; j++) {
                for (int i = 0; i < 4; i++) acc[j][i] = fmaf(dv[j], av[i], acc[j][i]);
                bias[j] += dv[j];
            }
        }
    }
    part += (size_t)split * MLP_PARAMS;
    for (int j = 0; j < 4; j++) {
        if (o0 + j >= nout) continue;
        for (int i = 0; i < 4; i++)
            if (i0 + i < nin) part[offW + (o0 + j) * nin + i0 + i] = acc[j][i];
        if (i0 == 0) part[offB + o0 + j] = bias[j];
    }
}

// The parts' sums in their order.
__global__ __launch_bounds__(256) void k_mlp_wgrad_sum(const float *__restrict__ part, int splits, float *grad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MLP_PARAMS) return;
    float acc = part[i];
    for (int k = 1; k < splits; k++) acc += part[(size_t)k * MLP_PARAMS + i];
    grad[i] = acc;
}

// Adam (Kingma & Ba, 2015): m <- b1 m + (1 - b1) g, v <- b2 v + (1 - b2) g^2, theta -= lr m^ / (sqrt(v^) + eps).
__global__ __launch_bounds__(256) void k_adam(float *theta, const float *__restrict__ g, float *m, float *v, int n,
                                              float lr, float bc1, float bc2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    m[i] = b1 * m[i] + (1.f - b1) * g[i];
    v[i] = b2 * v[i] + (1.f - b2) * g[i] * g[i];
    theta[i] -= lr * (m[i] / bc1) / (sqrtf(v[i] / bc2) + eps);
}

// Rows of a dataset in the order of `rows` (a permutation) into a contiguous batch.
__global__ __launch_bounds__(256) void k_mlp_gather(const float *__restrict__ x, const float *__restrict__ y,
                                                    const int *__restrict__ rows, int B, float *bx, float *by) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= B * (MLP_IN + 1)) return;
    const int s = idx / (MLP_IN + 1), f = idx - s * (MLP_IN + 1);
    const int r = rows[s];
    if (f < MLP_IN) bx[s * MLP_IN + f] = x[(size_t)r * MLP_IN + f];
    else by[s] = y[r];
}

// Round to nearest even BF16 (the upper 16 bits of the FP32 pattern); finite inputs.
__device__ __forceinline__ unsigned short bf16_bits(float x) {
    unsigned u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

// One MFMA layer for a 16-row tile: D[16][64] = A[16][K] B[K][64] with A rows in LDS (bf16, row stride lda) and the
// weights in LDS as bf16 W[n][k] (row stride ldw), so B[k][n] = W[n][k].  v_mfma_f32_16x16x16bf16: lane l supplies
// A[l % 16][4 (l / 16) .. + 3] and B[4 (l / 16) .. + 3][l % 16] and receives D[4 (l / 16) + r][l % 16], r = 0..3.
template <int K>
__device__ __forceinline__ void mfma_layer(const unsigned short *A, int lda, const unsigned short *W, int ldw,
                                           float4v acc[4]) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int row = lane & 15, kq = 4 * (lane >> 4);
    for (int t = 0; t < 4; t++) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 16) {
        short4v a;
        for (int q = 0; q < 4; q++) a[q] = (short)A[row * lda + k0 + kq + q];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            short4v bv;
            const int n = 16 * t + row;
            for (int q = 0; q < 4; q++) bv[q] = (short)W[n * ldw + k0 + kq + q];
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bv, acc[t], 0, 0, 0);
        }
    }
}

constexpr int INFER_WAVES = 4;

// BF16 MFMA inference: one wavefront per tile of 16 pairs (features padded from 12 to 16 with zeros), FP32
// accumulation, biases and GELU in FP32, activations rounded to BF16 between layers.
__global__ __launch_bounds__(WAVE *INFER_WAVES) void k_mlp_infer(const float *__restrict__ x, int P,
                                                                 const float *__restrict__ theta, float *score) {
    __shared__ unsigned short sW1[64 * 16], sW2[64 * 64], sW3[64 * 64];
    __shared__ float sB[3 * 64 + 64 + 1];
    __shared__ unsigned short sA[INFER_WAVES][16 * 64];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    for (int e = tid; e < 64 * 16; e += blockDim.x) {
        const int n = e / 16, k = e - n * 16;
        sW1[e] = k < MLP_IN ? bf16_bits(theta[MLP_OFF_W1 + n * MLP_IN + k]) : 0;
    }
    for (int e = tid; e < 64 * 64; e += blockDim.x) {
        sW2[e] = bf16_bits(theta[MLP_OFF_W2 + e]);
        sW3[e] = bf16_bits(theta[MLP_OFF_W3 + e]);
    }
    for (int e = tid; e < 64; e += blockDim.x) {
        sB[e] = theta[MLP_OFF_B1 + e];
        sB[64 + e] = theta[MLP_OFF_B2 + e];
        sB[128 + e] = theta[MLP_OFF_B3 + e];
        sB[192 + e] = theta[MLP_OFF_W4 + e];
    }
    if (tid == 0) sB[256] = theta[MLP_OFF_B4];
    __syncthreads();
    unsigned short *A = sA[wave];
    const int row = lane & 15, r0 = 4 * (lane >> 4);
    const int tiles = (P + 15) / 16;
    for (int tile = blockIdx.x * INFER_WAVES + wave; tile < tiles; tile += gridDim.x * INFER_WAVES) {
        // input tile: 16 rows x 16 features (12 used), bf16
        for (int e = lane; e < 16 * 16; e += WAVE) {
            const int rr = e / 16, k = e - rr * 16;
            const int p = tile * 16 + rr;
            A[rr * 64 + k] = (k < MLP_IN && p < P) ? bf16_bits(x[(size_t)p * MLP_IN + k]) : 0;
        }
        __builtin_amdgcn_wave_barrier();
        float4v acc[4];
        mfma_layer<16>(A, 64, sW1, 16, acc);
        __builtin_amdgcn_wave_barrier();  // every lane has read the inputs before they are overwritten
        for (int layer = 0; layer < 3; layer++) {
            // bias + GELU of the layer just computed, rounded into the A tile (row r0 + r, column 16 t + row)
            float h[4][4];
            for (int t = 0; t < 4; t++)
                for (int r = 0; r < 4; r++) h[t][r] = gelu(acc[t][r] + sB[64 * layer + 16 * t + row]);
            if (layer == 2) {
                // output: z = b4 + sum_j w4[j] h3[j]; each lane sums its 4 columns, then the 16 lanes of a row group
                float z[4];
                for (int r = 0; r < 4; r++) {
                    float s = 0.f;
                    for (int t = 0; t < 4; t++) s += sB[192 + 16 * t + row] * h[t][r];
                    z[r] = s;
                }
                for (int off = 8; off > 0; off >>= 1)
                    for (int r = 0; r < 4; r++) z[r] += __shfl_xor(z[r], off, 16);
                if (row == 0)
                    for (int r = 0; r < 4; r++) {
                        const int p = tile * 16 + r0 + r;
                        if (p < P) score[p] = 1.f / (1.f + expf(-(z[r] + sB[256])));
                    }
                break;
            }
            for (int t = 0; t < 4; t++)
                for (int r = 0; r < 4; r++) A[(r0 + r) * 64 + 16 * t + row] = bf16_bits(h[t][r]);
            __builtin_amdgcn_wave_barrier();
            mfma_layer<64>(A, 64, layer == 0 ? sW2 : sW3, 64, acc);
            __builtin_amdgcn_wave_barrier();
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------------------------------------------

hipError_t mlp_forward_backward(hipStream_t s, const float *theta, int B, const float *x, const float *y,
                                MlpWork &w, float *grad) {
    const dim3 rows((unsigned)((B + ROWS - 1) / ROWS));
    hipLaunchKernelGGL(k_mlp_forward, rows, dim3(GRAD_THREADS), 0, s, x, theta, B, w);
    hipLaunchKernelGGL(k_mlp_head, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, s, w.a3, theta, y, B, w.dz,
                       w.lossPart);
    hipLaunchKernelGGL(k_mlp_backward, rows, dim3(GRAD_THREADS), 0, s, theta, B, w);
    // parts of the samples, as many as fit in pre3 (B x 64 floats), which nothing reads any more
    const int splits = std::max(1, (int)((size_t)B * MLP_H / MLP_PARAMS));
    hipLaunchKernelGGL(k_mlp_wgrad, dim3((unsigned)splits, 4), dim3(256), 0, s, x, B, splits, w,
                       splits > 1 ? w.pre3 : grad);
    if (splits > 1)
        hipLaunchKernelGGL(k_mlp_wgrad_sum, dim3((MLP_PARAMS + 255) / 256), dim3(256), 0, s, w.pre3, splits, grad);
    return hipGetLastError();
}

int mlp_loss_blocks(int B) { return (B + 255) / 256; }

hipError_t mlp_adam(hipStream_t s, float *theta, const float *grad, float *m, float *v, float lr, int step) {
    const float bc1 = 1.f - powf(0.9f, (float)step), bc2 = 1.f - powf(0.999f, (float)step);
    hipLaunchKernelGGL(k_adam, dim3((MLP_PARAMS + 255) / 256), dim3(256), 0, s, theta, grad, m, v, MLP_PARAMS, lr,
                       bc1, bc2);
    return hipGetLastError();
}

hipError_t mlp_gather(hipStream_t s, const float *x, const float *y, const int *rows, int B, float *bx, float *by) {
    hipLaunchKernelGGL(k_mlp_gather, dim3((unsigned)((B * (MLP_IN + 1) + 255) / 256)), dim3(256), 0, s, x, y, rows,
                       B, bx, by);
    return hipGetLastError();
}

hipError_t mlp_infer(hipStream_t s, const float *theta, int P, const float *x, float *score) {
    if (P <= 0) return hipSuccess;
    const int tiles = (P + 15) / 16;
    const unsigned blocks = (unsigned)std::min((tiles + INFER_WAVES - 1) / INFER_WAVES, 4096);
    hipLaunchKernelGGL(k_mlp_infer, dim3(blocks), dim3(WAVE * INFER_WAVES), 0, s, x, P, theta, score);
    return hipGetLastError();
}

}  // namespace rp
