// Small FP32 multilayer perceptron for the learned step-size controller:
// F inputs -> H (ReLU) -> H (ReLU) -> C logits, trained with minibatch Adam
// on the tracker's own step logs.  The controller's own shape runs forward and
// back in one kernel on the FP32 matrix cores; other shapes as tiled FP32
// matrix products staged through LDS plus elementwise kernels.
//
// The reference has no learned component; the step rule it keeps as judge
// and fallback is the pole step of LU_Prediction
// (Deformations/Curves/standard_predictor_convolutions.adb:1142-1185).
//
// Parameter vector layout (floats): W1[F][H], b1[H], W2[H][H], b2[H],
// W3[H][C], b3[C].  Loss: mean over the batch of the binary cross-entropy of
// the logit of the candidate that was tried, sigmoid(o[cand]) vs accepted.
#include <hip/hip_runtime.h>
#include <vector>
#include "common.hpp"
#include "../../include/phcmd.h"

namespace {

constexpr int TILE = 16;

// C[M][N] = op(A)[M][Kd] * op(B)[Kd][N] (+ C when accumulate)
// op(A)[m][k] = ta ? A[k*lda+m] : A[m*lda+k]; op(B)[k][n] = tb ? B[n*ldb+k] : B[k*ldb+n]
__global__ void gemm_kernel(int M, int N, int Kd, const float *__restrict__ A, int lda, int ta,
                            const float *__restrict__ B, int ldb, int tb, float *__restrict__ C,
                            int ldc, int accumulate) {
  __shared__ float As[TILE][TILE + 1], Bs[TILE][TILE + 1];
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int row = blockIdx.y * TILE + ty, col = blockIdx.x * TILE + tx;
  float acc = 0.0f;
  for (int k0 = 0; k0 < Kd; k0 += TILE) {
    const int ka = k0 + tx, kb = k0 + ty;
    float a = 0.0f, b = 0.0f;
    if (row < M && ka < Kd) a = ta ? A[(size_t)ka * lda + row] : A[(size_t)row * lda + ka];
    if (col < N && kb < Kd) b = tb ? B[(size_t)col * ldb + kb] : B[(size_t)kb * ldb + col];
    As[ty][tx] = a;
    Bs[ty][tx] = b;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TILE; ++k) acc += As[ty][k] * Bs[k][tx];
    __syncthreads();
  }
  if (row < M && col < N) {
    float *c = C + (size_t)row * ldc + col;
    *c = accumulate ? *c + acc : acc;
  }
}

// H = relu(Z + b) (relu optional), Z, H [M][N]
__global__ void bias_act_kernel(int M, int N, const float *Z, const float *b, float *H, int relu) {
  const size_t n = (size_t)M * N;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    float v = Z[i] + b[i % N];
    H[i] = (relu && v < 0.0f) ? 0.0f : v;
  }
}

// dO[i][c] = (c == cand_i) ? (sigmoid(O[i][c]) - y_i) * scale : 0; loss += scale * BCE
__global__ void loss_grad_kernel(int B, int C, const float *O, const int *cand, const float *y,
                                 float scale, float *dO, float *loss) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < B; i += gridDim.x * blockDim.x) {
    const int c = cand[i];
    for (int j = 0; j < C; ++j) dO[(size_t)i * C + j] = 0.0f;
    if (c < 0 || c >= C) continue;
    const float o = O[(size_t)i * C + c];
    const float p = 1.0f / (1.0f + expf(-o));
    dO[(size_t)i * C + c] = (p - y[i]) * scale;
    // log(1 + e^o) - y*o, computed stably
    const float l = fmaxf(o, 0.0f) - o * y[i] + log1pf(expf(-fabsf(o)));
    if (loss) atomicAdd(loss, l * scale);
  }
}

// dZ = dH * (H > 0)
__global__ void relu_back_kernel(size_t n, const float *H, const float *dH, float *dZ) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dZ[i] = H[i] > 0.0f ? dH[i] : 0.0f;
}

// db[j] = sum_i dZ[i][j]; one block per column
__global__ void colsum_kernel(int M, int N, const float *dZ, float *db) {
  __shared__ float part[256];
  const int j = blockIdx.x;
  float s = 0.0f;
  for (int i = threadIdx.x; i < M; i += blockDim.x) s += dZ[(size_t)i * N + j];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int m = blockDim.x / 2; m > 0; m >>= 1) {
    if (threadIdx.x < m) part[threadIdx.x] += part[threadIdx.x + m];
    __syncthreads();
  }
  if (threadIdx.x == 0) db[j] = part[0];
}

__global__ void adam_kernel(int n, float *w, const float *g, float *m, float *v, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float gi = g[i];
    m[i] = b1 * m[i] + (1.0f - b1) * gi;
    v[i] = b2 * v[i] + (1.0f - b2) * gi * gi;
    w[i] -= lr * (m[i] / c1) / (sqrtf(v[i] / c2) + eps);
  }
}

struct Dims {
  int F, H, C;
  __host__ __device__ size_t nW1() const { return (size_t)F * H; }
  __host__ __device__ size_t oW1() const { return 0; }
  __host__ __device__ size_t ob1() const { return nW1(); }
  __host__ __device__ size_t oW2() const { return ob1() + H; }
  __host__ __device__ size_t ob2() const { return oW2() + (size_t)H * H; }
  __host__ __device__ size_t oW3() const { return ob2() + H; }
  __host__ __device__ size_t ob3() const { return oW3() + (size_t)H * C; }
  __host__ __device__ size_t total() const { return ob3() + C; }
};

void gemm(hipStream_t st, int M, int N, int Kd, const float *A, int lda, int ta, const float *B,
          int ldb, int tb, float *C, int ldc, int acc) {
  dim3 grid((N + TILE - 1) / TILE, (M + TILE - 1) / TILE), block(TILE, TILE);
  hipLaunchKernelGGL(gemm_kernel, grid, block, 0, st, M, N, Kd, A, lda, ta, B, ldb, tb, C, ldc, acc);
}

// forward on B samples; Z1,H1,Z2,H2 [B][H], O [B][C]
void forward(hipStream_t st, const Dims &d, const float *w, int B, const float *X, float *Z1,
             float *H1, float *Z2, float *H2, float *O) {
  const int g = phc::grid_for((size_t)B * d.H, 256);
  gemm(st, B, d.H, d.F, X, d.F, 0, w + d.oW1(), d.H, 0, Z1, d.H, 0);
  hipLaunchKernelGGL(bias_act_kernel, dim3(g), dim3(256), 0, st, B, d.H, Z1, w + d.ob1(), H1, 1);
  gemm(st, B, d.H, d.H, H1, d.H, 0, w + d.oW2(), d.H, 0, Z2, d.H, 0);
  hipLaunchKernelGGL(bias_act_kernel, dim3(g), dim3(256), 0, st, B, d.H, Z2, w + d.ob2(), H2, 1);
  gemm(st, B, d.C, d.H, H2, d.H, 0, w + d.oW3(), d.C, 0, O, d.C, 0);
  hipLaunchKernelGGL(bias_act_kernel, dim3(phc::grid_for((size_t)B * d.C, 256)), dim3(256), 0, st,
                     B, d.C, O, w + d.ob3(), O, 0);
}

// gradient of the mean loss over B samples into grad (same layout as w)
void backward(hipStream_t st, const Dims &d, const float *w, int B, const float *X, const int *cand,
              const float *y, const float *H1, const float *H2, const float *O, float *dO,
              float *dH, float *dZ, float *grad, float *loss) {
  const size_t nh = (size_t)B * d.H;
  hipLaunchKernelGGL(loss_grad_kernel, dim3(phc::grid_for(B, 256)), dim3(256), 0, st, B, d.C, O,
                     cand, y, 1.0f / (float)B, dO, loss);
  // layer 3: dW3 = H2^T dO, db3 = colsum dO, dH2 = dO W3^T
  gemm(st, d.H, d.C, B, H2, d.H, 1, dO, d.C, 0, grad + d.oW3(), d.C, 0);
  hipLaunchKernelGGL(colsum_kernel, dim3(d.C), dim3(256), 0, st, B, d.C, dO, grad + d.ob3());
  gemm(st, B, d.H, d.C, dO, d.C, 0, w + d.oW3(), d.C, 1, dH, d.H, 0);
  hipLaunchKernelGGL(relu_back_kernel, dim3(phc::grid_for(nh, 256)), dim3(256), 0, st, nh, H2, dH, dZ);
  // layer 2
  gemm(st, d.H, d.H, B, H1, d.H, 1, dZ, d.H, 0, grad + d.oW2(), d.H, 0);
  hipLaunchKernelGGL(colsum_kernel, dim3(d.H), dim3(256), 0, st, B, d.H, dZ, grad + d.ob2());
  gemm(st, B, d.H, d.H, dZ, d.H, 0, w + d.oW2(), d.H, 1, dH, d.H, 0);
  hipLaunchKernelGGL(relu_back_kernel, dim3(phc::grid_for(nh, 256)), dim3(256), 0, st, nh, H1, dH, dZ);
  // layer 1
  gemm(st, d.F, d.H, B, X, d.F, 1, dZ, d.H, 0, grad + d.oW1(), d.H, 0);
  hipLaunchKernelGGL(colsum_kernel, dim3(d.H), dim3(256), 0, st, B, d.H, dZ, grad + d.ob1());
}

struct Scratch {
  float *Z1 = nullptr, *H1, *Z2, *H2, *O, *dO, *dH, *dZ;
  int alloc(int B, const Dims &d) {
    const size_t nh = (size_t)B * d.H, nc = (size_t)B * d.C;
    float *base = nullptr;
    PHC_HIP(hipMalloc(&base, sizeof(float) * (6 * nh + 2 * nc)));
    Z1 = base; H1 = Z1 + nh; Z2 = H1 + nh; H2 = Z2 + nh; dH = H2 + nh; dZ = dH + nh;
    O = dZ + nh; dO = O + nc;
    return 0;
  }
  void release() { if (Z1) (void)hipFree(Z1); Z1 = nullptr; }
};

// ---- the controller's network (at most 16 inputs, 64 hidden units, at most 16
// candidates) in one kernel on the FP32 matrix cores.
//   The layers one by one moved every activation through HBM and left the
// weight gradients, products over all rows, to 16 workgroups: 8.6 ms for the
// gradient over 65536 rows.  Here a wavefront takes 16 rows at a time through
// the network and back (272 v_mfma_f32_16x16x4), the weights and its
// activations in LDS, the weight gradients in 96 accumulators that it keeps
// over all its rows; blocks leave partial sums that reduce_kernel adds in order
// (for training together with the Adam step).
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int FH = 64, FF = 16, FC = 16;      // hidden units; padded inputs and candidates
constexpr int SH = FH + 1, SN = FF + 1;       // LDS row strides
constexpr int FW = 4, FROWS = 16;             // wavefronts per block, rows of a wavefront's tile
constexpr int FBLOCKS = 256;
// LDS in floats: W1, W2, W3, b1, b2, b3, then per wavefront X, H1, H2, dZ2, dO
constexpr int LW1 = 0, LW2 = LW1 + FF * SH, LW3 = LW2 + FH * SH, LB1 = LW3 + FH * SN, LB2 = LB1 + FH,
              LB3 = LB2 + FH, LWAVE = LB3 + FC;
constexpr int WX = 0, WH1 = WX + FROWS * SN, WH2 = WH1 + FROWS * SH, WD2 = WH2 + FROWS * SH,
              WDO = WD2 + FROWS * SH, WTOT = WDO + FROWS * SN;
constexpr size_t FLDS = sizeof(float) * (LWAVE + FW * WTOT);

bool fused(const Dims &d) { return d.F <= FF && d.H == FH && d.C <= FC; }
int fused_blocks(int B) {
  const int b = (B + FW * FROWS - 1) / (FW * FROWS);
  return b < FBLOCKS ? b : FBLOCKS;
}

__device__ __forceinline__ void wave_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// c[t] += sum_k a(k) b(k, t) over 4 S values of k: lane l gives A's row l % 16
// and B's column l % 16 at k = 4 s + l / 16, and holds C's column l % 16 in rows
// 4 (l / 16) + 0..3
template <int S, int T, class A, class B>
__device__ __forceinline__ void tile_mac(v4f *c, const A &a, const B &b) {
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = 4 * s + ((threadIdx.x & 63) >> 4);
    const float av = a(k);
#pragma unroll
    for (int t = 0; t < T; ++t) c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, b(k, t), c[t], 0, 0, 0);
  }
}

// GRAD false: logits [B][C].  GRAD: part[block][total + 1], the block's sums of
// the gradient (times scale) in the layout of w, then of the loss.
template <bool GRAD>
__global__ void __launch_bounds__(64 * FW)
fused_kernel(Dims d, const float *__restrict__ w, int B, const float *__restrict__ X,
             const int *__restrict__ cand, const float *__restrict__ y, float scale,
             float *__restrict__ logits, float *__restrict__ part) {
  extern __shared__ float lds[];
  const int t = threadIdx.x, l = t & 63, wv = t >> 6, n = l & 15, q = l >> 4;
  for (int e = t; e < FF * FH; e += 64 * FW) lds[LW1 + e / FH * SH + e % FH] = e < d.F * FH ? w[d.oW1() + e] : 0.0f;
  for (int e = t; e < FH * FH; e += 64 * FW) lds[LW2 + e / FH * SH + e % FH] = w[d.oW2() + e];
  for (int e = t; e < FH * FC; e += 64 * FW)
    lds[LW3 + e / FC * SN + e % FC] = e % FC < d.C ? w[d.oW3() + e / FC * d.C + e % FC] : 0.0f;
  if (t < FH) {
    lds[LB1 + t] = w[d.ob1() + t];
    lds[LB2 + t] = w[d.ob2() + t];
  }
  if (t < FC) lds[LB3 + t] = t < d.C ? w[d.ob3() + t] : 0.0f;
  __syncthreads();
  const float *W1 = lds + LW1, *W2 = lds + LW2, *W3 = lds + LW3;
  float *mine = lds + LWAVE + wv * WTOT, *Xs = mine + WX, *H1 = mine + WH1, *H2 = mine + WH2,
        *D2 = mine + WD2, *dO = mine + WDO, *D1 = H2;
  v4f g1[4] = {}, g2[4][4] = {}, g3[4] = {};
  float s1[4] = {}, s2[4] = {}, s3 = 0.0f, loss = 0.0f;
  const int tiles = (B + FROWS - 1) / FROWS;
  for (int tile = blockIdx.x * FW + wv; tile < tiles; tile += gridDim.x * FW) {
    const int row0 = tile * FROWS;
    for (int e = l; e < FROWS * FF; e += 64) {
      const int r = e / FF, f = e % FF;
      Xs[r * SN + f] = (row0 + r < B && f < d.F) ? X[(size_t)(row0 + r) * d.F + f] : 0.0f;
    }
    wave_lds();
    // a layer's 64 units: relu of the products plus the bias, to LDS
    auto hidden = [&](v4f *c, const float *bias, float *H) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = c[u][r] + bias[16 * u + n];
          H[(4 * q + r) * SH + 16 * u + n] = v < 0.0f ? 0.0f : v;
        }
      wave_lds();
    };
    {
      v4f c[4] = {};
      tile_mac<4, 4>(c, [&](int k) { return Xs[n * SN + k]; }, [&](int k, int u) { return W1[k * SH + 16 * u + n]; });
      hidden(c, lds + LB1, H1);
    }
    {
      v4f c[4] = {};
      tile_mac<16, 4>(c, [&](int k) { return H1[n * SH + k]; }, [&](int k, int u) { return W2[k * SH + 16 * u + n]; });
      hidden(c, lds + LB2, H2);
    }
    v4f o[1] = {};
    tile_mac<16, 1>(o, [&](int k) { return H2[n * SH + k]; }, [&](int k, int) { return W3[k * SN + n]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 4 * q + r;
      const float z = o[0][r] + lds[LB3 + n];
      if constexpr (!GRAD) {
        if (row < B && n < d.C) logits[(size_t)row * d.C + n] = z;
      } else {
        float g = 0.0f;
        if (row < B && n < d.C && cand[row] == n) {
          const float yy = y[row], p = 1.0f / (1.0f + expf(-z));
          g = (p - yy) * scale;
          // log(1 + e^z) - y z, computed stably
          loss += (fmaxf(z, 0.0f) - z * yy + log1pf(expf(-fabsf(z)))) * scale;
        }
        dO[(4 * q + r) * SN + n] = g;
        s3 += g;
      }
    }
    wave_lds();
    if constexpr (GRAD) {
      {
        // dZ2 = (dO W3^T) where H2 > 0
        v4f c[4] = {};
        tile_mac<4, 4>(c, [&](int k) { return dO[n * SN + k]; }, [&](int k, int u) { return W3[(16 * u + n) * SN + k]; });
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int e = (4 * q + r) * SH + 16 * u + n;
            const float v = H2[e] > 0.0f ? c[u][r] : 0.0f;
            D2[e] = v;
            s2[u] += v;
          }
      }
      // dW3 += H2^T dO
#pragma unroll
      for (int u = 0; u < 4; ++u)
        tile_mac<4, 1>(g3 + u, [&](int k) { return H2[k * SH + 16 * u + n]; }, [&](int k, int) { return dO[k * SN + n]; });
      wave_lds();
      {
        // dZ1 = (dZ2 W2^T) where H1 > 0, in H2's place
        v4f c[4] = {};
        tile_mac<16, 4>(c, [&](int k) { return D2[n * SH + k]; }, [&](int k, int u) { return W2[(16 * u + n) * SH + k]; });
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int e = (4 * q + r) * SH + 16 * u + n;
            const float v = H1[e] > 0.0f ? c[u][r] : 0.0f;
            D1[e] = v;
            s1[u] += v;
          }
      }
      // dW2 += H1^T dZ2
#pragma unroll
      for (int u = 0; u < 4; ++u)
        tile_mac<4, 4>(g2[u], [&](int k) { return H1[k * SH + 16 * u + n]; }, [&](int k, int v) { return D2[k * SH + 16 * v + n]; });
      wave_lds();
      // dW1 += X^T dZ1
      tile_mac<4, 4>(g1, [&](int k) { return Xs[k * SN + n]; }, [&](int k, int u) { return D1[k * SH + 16 * u + n]; });
      wave_lds();
    }
  }
  if constexpr (GRAD) {
    // the block's sums: the wavefronts add theirs one after another in LDS
    const int np = (int)d.total();
    float *sum = lds + LWAVE;  // np + 1 floats
    auto column = [&](float v) {
      v += __shfl_xor(v, 16, 64);
      return v + __shfl_xor(v, 32, 64);
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) { s1[u] = column(s1[u]); s2[u] = column(s2[u]); }
    s3 = column(s3);
    for (int m = 1; m < 64; m <<= 1) loss += __shfl_xor(loss, m, 64);
    for (int k = 0; k < FW; ++k) {
      __syncthreads();
      if (wv != k) continue;
      auto put = [&](size_t e, float v) { sum[e] = k ? sum[e] + v : v; };
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (4 * q + r < d.F) put(d.oW1() + (4 * q + r) * FH + 16 * u + n, g1[u][r]);
          if (n < d.C) put(d.oW3() + (16 * u + 4 * q + r) * d.C + n, g3[u][r]);
#pragma unroll
          for (int v = 0; v < 4; ++v) put(d.oW2() + (16 * u + 4 * q + r) * FH + 16 * v + n, g2[u][v][r]);
        }
      if (q == 0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          put(d.ob1() + 16 * u + n, s1[u]);
          put(d.ob2() + 16 * u + n, s2[u]);
        }
        if (n < d.C) put(d.ob3() + n, s3);
      }
      if (l == 0) put(np, loss);
    }
    __syncthreads();
    for (int e = t; e <= np; e += 64 * FW) part[(size_t)blockIdx.x * (np + 1) + e] = sum[e];
  }
}

// sums of the blocks' partial sums (four quarters of the blocks, then those):
// the gradient to g, or (ADAM) an Adam step on w; the loss added to *loss
// (or stored when set)
template <bool ADAM>
__global__ void __launch_bounds__(256)
reduce_kernel(int np, int blocks, const float *__restrict__ part, float *g, float *loss, int set, float *w,
              float *m, float *v, float lr, float b1, float b2, float eps, float c1, float c2) {
  __shared__ float quarter[4][64];
  const int i = blockIdx.x * 64 + (threadIdx.x & 63), s = threadIdx.x >> 6;
  float x = 0.0f;
  if (i <= np)
    for (int b = s; b < blocks; b += 4) x += part[(size_t)b * (np + 1) + i];
  quarter[s][threadIdx.x & 63] = x;
  __syncthreads();
  if (s || i > np) return;
  x = (quarter[0][threadIdx.x] + quarter[1][threadIdx.x]) + (quarter[2][threadIdx.x] + quarter[3][threadIdx.x]);
  if (i == np) {
    if (loss) *loss = set ? x : *loss + x;
  } else if constexpr (ADAM) {
    m[i] = b1 * m[i] + (1.0f - b1) * x;
    v[i] = b2 * v[i] + (1.0f - b2) * x * x;
    w[i] -= lr * (m[i] / c1) / (sqrtf(v[i] / c2) + eps);
  } else {
    g[i] = x;
  }
}

template <bool GRAD>
int launch_fused(hipStream_t st, const Dims &d, const float *w, int B, const float *X, const int *cand,
                 const float *y, float *logits, float *part) {
  PHC_HIP(hipFuncSetAttribute((const void *)fused_kernel<GRAD>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)FLDS));
  hipLaunchKernelGGL(fused_kernel<GRAD>, dim3(fused_blocks(B)), dim3(64 * FW), FLDS, st, d, w, B, X, cand, y,
                     1.0f / (float)B, logits, part);
  PHC_HIP(hipGetLastError());
  return 0;
}

}  // namespace

extern "C" {

int phc_mlp_size(int F, int H, int C, int *nparams) {
  PHC_REQUIRE(nparams && F >= 1 && H >= 1 && C >= 1, "phc_mlp_size: bad sizes");
  *nparams = (int)Dims{F, H, C}.total();
  return 0;
}

int phc_mlp_forward(int F, int H, int C, const float *w, int B, const float *X, float *logits,
                    void *stream) {
  PHC_REQUIRE(F >= 1 && H >= 1 && C >= 1 && B >= 0, "phc_mlp_forward: bad sizes");
  if (B == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  Dims d{F, H, C};
  if (fused(d)) {
    if (launch_fused<false>(st, d, w, B, X, nullptr, nullptr, logits, nullptr) != 0) return -1;
    PHC_HIP(hipStreamSynchronize(st));
    return 0;
  }
  Scratch s;
  if (s.alloc(B, d) != 0) return -1;
  forward(st, d, w, B, X, s.Z1, s.H1, s.Z2, s.H2, s.O);
  PHC_HIP(hipMemcpyAsync(logits, s.O, sizeof(float) * B * C, hipMemcpyDeviceToDevice, st));
  PHC_HIP(hipStreamSynchronize(st));
  s.release();
  PHC_HIP(hipGetLastError());
  return 0;
}

int phc_mlp_grad(int F, int H, int C, const float *w, int B, const float *X, const int *cand,
                 const float *y, float *grad, float *loss, void *stream) {
  PHC_REQUIRE(F >= 1 && H >= 1 && C >= 1 && B >= 1, "phc_mlp_grad: bad sizes");
  hipStream_t st = (hipStream_t)stream;
  Dims d{F, H, C};
  if (fused(d)) {
    const int np = (int)d.total(), blocks = fused_blocks(B);
    float *part = nullptr;
    PHC_HIP(hipMalloc(&part, sizeof(float) * (np + 1) * blocks));
    int rc = launch_fused<true>(st, d, w, B, X, cand, y, nullptr, part);
    if (rc == 0)
      hipLaunchKernelGGL(reduce_kernel<false>, dim3(np / 64 + 1), dim3(256), 0, st, np, blocks, part, grad,
                         loss, 1, nullptr, nullptr, nullptr, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f);
    const hipError_t e = hipStreamSynchronize(st);
    (void)hipFree(part);
    if (rc) return rc;
    PHC_HIP(e);
    PHC_HIP(hipGetLastError());
    return 0;
  }
  Scratch s;
  if (s.alloc(B, d) != 0) return -1;
  if (loss) PHC_HIP(hipMemsetAsync(loss, 0, sizeof(float), st));
  forward(st, d, w, B, X, s.Z1, s.H1, s.Z2, s.H2, s.O);
  backward(st, d, w, B, X, cand, y, s.H1, s.H2, s.O, s.dO, s.dH, s.dZ, grad, loss);
  PHC_HIP(hipStreamSynchronize(st));
  s.release();
  PHC_HIP(hipGetLastError());
  return 0;
}

int phc_mlp_train(int F, int H, int C, float *w, int N, const float *X, const int *cand,
                  const float *y, int epochs, int batch, float lr, unsigned seed, float *losses,
                  void *stream) {
  PHC_REQUIRE(F >= 1 && H >= 1 && C >= 1 && N >= 1 && epochs >= 0 && batch >= 1,
              "phc_mlp_train: bad sizes");
  hipStream_t st = (hipStream_t)stream;
  Dims d{F, H, C};
  const int B = batch < N ? batch : N;
  const size_t np = d.total();
  Scratch s;
  const bool one = fused(d);
  const int blocks = fused_blocks(B);
  float *part = nullptr;
  if (one)
    PHC_HIP(hipMalloc(&part, sizeof(float) * (np + 1) * blocks));
  else if (s.alloc(B, d) != 0)
    return -1;
  float *opt = nullptr, *loss = nullptr;
  PHC_HIP(hipMalloc(&opt, sizeof(float) * (3 * np + 1)));
  float *grad = opt, *m = opt + np, *v = m + np;
  loss = v + np;
  PHC_HIP(hipMemsetAsync(opt, 0, sizeof(float) * (3 * np + 1), st));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  float c1 = 1.0f, c2 = 1.0f;
  // minibatches are consecutive slices of an epoch-dependent rotation of the
  // data (deterministic given the seed; the caller shuffles rows once)
  const int nb = N / B > 0 ? N / B : 1;
  for (int e = 0; e < epochs; ++e) {
    PHC_HIP(hipMemsetAsync(loss, 0, sizeof(float), st));
    const int rot = (int)((seed + 7919u * (unsigned)e) % (unsigned)nb);
    for (int q = 0; q < nb; ++q) {
      const size_t off = (size_t)((q + rot) % nb) * B;
      if (one) {
        if (launch_fused<true>(st, d, w, B, X + off * F, cand + off, y + off, nullptr, part) != 0) {
          (void)hipFree(opt);
          (void)hipFree(part);
          return -1;
        }
        c1 *= b1;
        c2 *= b2;
        hipLaunchKernelGGL(reduce_kernel<true>, dim3(np / 64 + 1), dim3(256), 0, st, (int)np, blocks, part,
                           nullptr, loss, 0, w, m, v, lr, b1, b2, eps, 1.0f - c1, 1.0f - c2);
        continue;
      }
      forward(st, d, w, B, X + off * F, s.Z1, s.H1, s.Z2, s.H2, s.O);
      backward(st, d, w, B, X + off * F, cand + off, y + off, s.H1, s.H2, s.O, s.dO, s.dH, s.dZ,
               grad, loss);
      c1 *= b1;
      c2 *= b2;
      hipLaunchKernelGGL(adam_kernel, dim3(phc::grid_for(np, 256)), dim3(256), 0, st, (int)np, w,
                         grad, m, v, lr, b1, b2, eps, 1.0f - c1, 1.0f - c2);
    }
    if (losses) {
      float l = 0.0f;
      PHC_HIP(hipMemcpyAsync(&l, loss, sizeof(float), hipMemcpyDeviceToHost, st));
      PHC_HIP(hipStreamSynchronize(st));
      losses[e] = l / (float)nb;
    }
  }
  PHC_HIP(hipStreamSynchronize(st));
  (void)hipFree(opt);
  (void)hipFree(part);
  s.release();
  PHC_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
