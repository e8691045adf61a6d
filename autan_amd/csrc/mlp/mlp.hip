// The warm-start network on gfx950: a multilayer perceptron with SiLU activations, BF16 weights and
// activations on the matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation), FP32 master
// weights with Adam. No counterpart in the reference: the learned initial state of the bump sweep.
//
// Layout: samples are rows. Layer l maps K_l inputs to N_l outputs with weights W_l stored N_l x K_l
// (row n holds the weights into output n), so every operand of the forward product is read along
// K; beside the FP32 masters the BF16 weights are packed as the matrix cores read them (1 KB per 16
// outputs x 32 inputs) for the fused kernels. The input width is padded to 32 and the output width to 16 with zero weights.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <random>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

#include "../../../include/mxmlp.h"

namespace mxm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
using bf16 = __bf16;

constexpr int kThreads = 256;
constexpr int kTileM = 64, kTileN = 64, kTileK = 32;
constexpr int kPad = 8;  // LDS row padding (bf16) against bank conflicts

inline void check(hipError_t e, const char* what) {
  if (e == hipSuccess) return;
  (void)hipGetLastError();  // reported here: the next launch's check must not find it
  throw std::runtime_error(std::string("E1101: ") + what + ": " + hipGetErrorString(e));
}

// SiLU and its derivative through the logistic s(z) = 1 / (1 + e^-z), with the hardware exponential
// and reciprocal (about 1 ulp each; the activations are rounded to BF16 right after).
__device__ __forceinline__ float logistic(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) { return z * logistic(z); }
__device__ __forceinline__ float silu_grad(float z) {
  const float s = logistic(z);
  return s * (1.0f + z * (1.0f - s));
}

// Epilogues of the product C = op(A) op(B).
enum Epi : int {
  kStoreF32 = 0,     // Cf = C
  kAtomicF32 = 1,    // Cf += C (split over K)
  kBiasSiLU = 2,     // Zf = C + bias, Hb = silu(Z)
  kBias = 3,         // Cf = C + bias
  kSiLUGrad = 4,     // Hb = C * silu'(Z[m, n])  (Z read from Cf)
};

// C[M x N] = op(A) op(B), op(A)[m][k] = TA ? A[k lda + m] : A[m lda + k], op(B)[k][n] = TB ? B[n ldb + k]
// : B[k ldb + n]. One 64 x 64 tile per workgroup of four waves (32 x 32 each, 2 x 2 matrix-core
// tiles of 16 x 16 x 32), K in steps of 32 staged through LDS with K contiguous; blockIdx.z splits
// K into chunks of kchunk. Elements outside M, N, K read as zero.
template <bool TA, bool TB, int EPI>
__global__ __launch_bounds__(kThreads) void k_gemm(const bf16* __restrict__ A, const bf16* __restrict__ B, int M, int N,
                                                   int K, int lda, int ldb, int kchunk, float* __restrict__ Cf,
                                                   bf16* __restrict__ Hb, const float* __restrict__ bias, int ldc) {
  __shared__ __align__(16) bf16 As[kTileM][kTileK + kPad];
  __shared__ __align__(16) bf16 Bs[kTileN][kTileK + kPad];
  const int m0 = blockIdx.y * kTileM, n0 = blockIdx.x * kTileN;
  const int kb = blockIdx.z * kchunk, ke = min(K, kb + kchunk);
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int wm = (wave / 2) * 32, wn = (wave % 2) * 32;
  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i) {
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bf16 zero = static_cast<bf16>(0.0f);
  for (int k0 = kb; k0 < ke; k0 += kTileK) {
    // Stage A: 64 rows x 32 k, 8 elements per thread.
    if constexpr (!TA) {
      const int r = t / 4, kk = (t % 4) * 8;
      const int m = m0 + r, k = k0 + kk;
      bf16x8 v;
      if (m < M && k + 8 <= ke) {
        v = *reinterpret_cast<const bf16x8*>(A + static_cast<long long>(m) * lda + k);
      } else {
        for (int q = 0; q < 8; ++q) v[q] = (m < M && k + q < ke) ? A[static_cast<long long>(m) * lda + k + q] : zero;
      }
      *reinterpret_cast<bf16x8*>(&As[r][kk]) = v;
    } else {
      const int kk = t / 8, r = (t % 8) * 8;
      const int k = k0 + kk, m = m0 + r;
      bf16x8 v;
      if (k < ke && m + 8 <= M) {
        v = *reinterpret_cast<const bf16x8*>(A + static_cast<long long>(k) * lda + m);
      } else {
        for (int q = 0; q < 8; ++q) v[q] = (k < ke && m + q < M) ? A[static_cast<long long>(k) * lda + m + q] : zero;
      }
      for (int q = 0; q < 8; ++q) As[r + q][kk] = v[q];
    }
    // Stage B as Bs[n][k].
    if constexpr (TB) {
      const int r = t / 4, kk = (t % 4) * 8;
      const int n = n0 + r, k = k0 + kk;
      bf16x8 v;
      if (n < N && k + 8 <= ke) {
        v = *reinterpret_cast<const bf16x8*>(B + static_cast<long long>(n) * ldb + k);
      } else {
        for (int q = 0; q < 8; ++q) v[q] = (n < N && k + q < ke) ? B[static_cast<long long>(n) * ldb + k + q] : zero;
      }
      *reinterpret_cast<bf16x8*>(&Bs[r][kk]) = v;
    } else {
      const int kk = t / 8, r = (t % 8) * 8;
      const int k = k0 + kk, n = n0 + r;
      bf16x8 v;
      if (k < ke && n + 8 <= N) {
        v = *reinterpret_cast<const bf16x8*>(B + static_cast<long long>(k) * ldb + n);
      } else {
        for (int q = 0; q < 8; ++q) v[q] = (k < ke && n + q < N) ? B[static_cast<long long>(k) * ldb + n + q] : zero;
      }
      for (int q = 0; q < 8; ++q) Bs[r + q][kk] = v[q];
    }
    __syncthreads();
    // Lane l holds row (l mod 16) of A and column (l mod 16) of B at k = 8 (l / 16) .. + 7.
    const int row = lane % 16, kq = 8 * (lane / 16);
    bf16x8 a[2], b[2];
    for (int i = 0; i < 2; ++i) a[i] = *reinterpret_cast<const bf16x8*>(&As[wm + 16 * i + row][kq]);
    for (int j = 0; j < 2; ++j) b[j] = *reinterpret_cast<const bf16x8*>(&Bs[wn + 16 * j + row][kq]);
    for (int i = 0; i < 2; ++i) {
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // Lane l holds rows 4 (l / 16) .. + 3 of column (l mod 16) of each 16 x 16 tile.
  for (int i = 0; i < 2; ++i) {
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn + 16 * j + lane % 16;
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * (lane / 16) + r;
        if (m >= M || n >= N) continue;
        const float c = acc[i][j][r];
        const long long at = static_cast<long long>(m) * ldc + n;
        if constexpr (EPI == kStoreF32) {
          Cf[at] = c;
        } else if constexpr (EPI == kAtomicF32) {
          atomicAdd(Cf + at, c);
        } else if constexpr (EPI == kBiasSiLU) {
          const float z = c + bias[n];
          Cf[at] = z;
          Hb[at] = static_cast<bf16>(silu(z));
        } else if constexpr (EPI == kBias) {
          Cf[at] = c + bias[n];
        } else {
          Hb[at] = static_cast<bf16>(c * silu_grad(Cf[at]));
        }
      }
    }
  }
}

// Inputs normalised and rounded to BF16, padded to `width` columns with zeros.
__global__ void k_inputs(const float* __restrict__ x, int n, int d, const float* __restrict__ mean,
                         const float* __restrict__ scale, bf16* __restrict__ X, int width) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<long long>(n) * width) return;
  const long long r = i / width;
  const int c = static_cast<int>(i % width);
  X[i] = static_cast<bf16>(c < d ? (x[r * d + c] - mean[c]) / scale[c] : 0.0f);
}

// Mean squared error of the first d of `width` outputs against normalised targets, and its
// gradient 2 (y - t) / (n d) in BF16 (zero in the padding columns); the squared errors summed into
// *sum (each block's partial added once).
__global__ void k_loss(const float* __restrict__ y, const float* __restrict__ t, int n, int d, int width,
                       const float* __restrict__ mean, const float* __restrict__ scale, bf16* __restrict__ dy,
                       double* __restrict__ sum) {
  __shared__ float red[256];
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  float e2 = 0.0f;
  if (i < static_cast<long long>(n) * width) {
    const long long r = i / width;
    const int c = static_cast<int>(i % width);
    float g = 0.0f;
    if (c < d) {
      const float e = y[i] - (t[r * d + c] - mean[c]) / scale[c];
      e2 = e * e;
      g = 2.0f * e / (static_cast<float>(n) * d);
    }
    dy[i] = static_cast<bf16>(g);
  }
  red[threadIdx.x] = e2;
  __syncthreads();
  for (int s = 128; s > 0; s /= 2) {
    if (static_cast<int>(threadIdx.x) < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(sum, static_cast<double>(red[0]));
}

// Column sums of a BF16 n x width matrix (the bias gradients) added into g: thread (x, y) sums
// column x over the rows y, y + gridDim.y blockDim.y, ...
__global__ void k_colsum(const bf16* __restrict__ dz, int n, int width, float* __restrict__ g) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= width) return;
  float s = 0.0f;
  for (int r = blockIdx.y; r < n; r += gridDim.y) s += static_cast<float>(dz[static_cast<long long>(r) * width + c]);
  atomicAdd(g + c, s);
}

// A training step's counters, kept on the device so that a recorded step replays unchanged: the
// batch of the epoch, Adam's step and its bias corrections 1 - b^step.
struct StepState {
  long long batch;
  long long step;
  float c1, c2;
};

// Adam's next step (one thread): the step count and its bias corrections; the next batch.
__global__ void k_next_step(StepState* st, float b1, float b2) {
  st->batch += 1;
  st->step += 1;
  const float t = static_cast<float>(st->step);
  st->c1 = 1.0f - powf(b1, t);
  st->c2 = 1.0f - powf(b2, t);
}

__global__ void k_set_batch(StepState* st, long long b) { st->batch = b; }

// Batch `st->batch` of the shuffled order (n samples from idx[batch n]) into bx, bt.
__global__ void k_gather(const long long* __restrict__ idx, const StepState* __restrict__ st, int n,
                         const float* __restrict__ x, int dx, const float* __restrict__ t, int dt, float* __restrict__ bx,
                         float* __restrict__ bt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long long r = idx[st->batch * n + i];
  for (int c = 0; c < dx; ++c) bx[static_cast<long long>(i) * dx + c] = x[r * dx + c];
  for (int c = 0; c < dt; ++c) bt[static_cast<long long>(i) * dt + c] = t[r * dt + c];
}

__global__ void k_fill(float* __restrict__ p, long long n, float v) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// The splits' partial gradients added in split order.
__device__ __forceinline__ float sum_parts(const float* __restrict__ part, long long np, int splits, long long i) {
  float v = 0.0f;
#pragma unroll 8
  for (int q = 0; q < splits; ++q) v += part[q * np + i];
  return v;
}

// The BF16 weights: row-major for the layer-by-layer products, and, where the network is as narrow as the
// fused kernels, as their operands, packed (pack_place) as they are and transposed, at the places `at`
// gives each parameter (x the packed copy's, y the transposed one's, -1: none; null: no such copies).
struct WeightCopies {
  bf16* row;
  bf16* packed;
  bf16* turned;
  const int2* at;
};

__device__ __forceinline__ void store_copies(const WeightCopies& c, long long i, float w) {
  const bf16 v = static_cast<bf16>(w);
  c.row[i] = v;
  if (c.at == nullptr) return;
  const int2 p = c.at[i];
  if (p.x >= 0) c.packed[p.x] = v;
  if (p.y >= 0) c.turned[p.y] = v;
}

// Adam (Kingma and Ba 2015) on the FP32 master weights, then their BF16 copies. `mask` marks the entries that exist (padding stays zero); the
// bias corrections are the step state's. The gradient is the sum of `splits` partial ones, in the order
// `order` gives (place j is parameter order[j]; null: the parameters').
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ part, int splits,
                       const int* __restrict__ order, float* __restrict__ m1,
                       float* __restrict__ m2, const unsigned char* __restrict__ mask, long long n, float lr, float b1,
                       float b2, float eps, const StepState* __restrict__ st, WeightCopies copies) {
  const long long j = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const long long i = order != nullptr ? order[j] : j;
  const float c1 = st->c1, c2 = st->c2;
  if (mask[i]) {
    const float gi = sum_parts(part, n, splits, j);
    const float a = b1 * m1[i] + (1.0f - b1) * gi;
    const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    w[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
  }
  store_copies(copies, i, w[i]);
}

__global__ void k_to_bf16(const float* __restrict__ w, long long n, WeightCopies copies) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) store_copies(copies, i, w[i]);
}

// Network outputs back in physical units: y * scale + mean for the first d columns.
__global__ void k_out(const float* __restrict__ y, int n, int d, int width, const float* __restrict__ mean,
                      const float* __restrict__ scale, float* __restrict__ out) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<long long>(n) * d) return;
  const long long r = i / d;
  const int c = static_cast<int>(i % d);
  out[i] = y[r * width + c] * scale[c] + mean[c];
}

// The fused kernels' weights: for each 16 outputs and each 32 inputs (of `steps` such) the 1 KB that a
// wave reads as one matrix-core operand, lane l the eight inputs 8 (l / 16) .. of output l mod 16. A
// load is then eight consecutive cache lines, in eight of the L2's channels; read from rows of 512
// bytes, sixteen half lines in four channels, every CU's loads of a layer queued on those.
__host__ __device__ constexpr long long pack_place(int out, int in, int steps) {
  return ((static_cast<long long>(out / 16) * steps + in / 32) * 64 + in % 32 / 8 * 16 + out % 16) * 8 + in % 8;
}
// The operand of outputs 16 tile .. and inputs 32 step .. for this lane.
__device__ __forceinline__ bf16x8 packed_operand(const bf16* W, int tile, int step, int steps) {
  return *reinterpret_cast<const bf16x8*>(W + ((static_cast<long long>(tile) * steps + step) * 64 + threadIdx.x % 64) * 8);
}

// The layers of a network as k_infer reads them: weight and bias offsets into the parameter arrays.
constexpr int kMaxLayers = 18;
struct LayerTable {
  long long w[kMaxLayers], b[kMaxLayers];
  int nl;
};

// The whole forward of 16 RT samples per workgroup (inference): the normalised inputs, then every
// layer's activations, stay in one 16 RT x (hidden + 8) BF16 LDS tile (dynamic shared memory); the
// weights stream from L2, each weight column read once per workgroup and used for all 16 RT rows,
// so the L2 bytes per product fall as RT grows. Each of the WAVES waves computes 16 CT output
// columns of the tile's rows as RT x CT matrix-core tiles, K in steps of 32 in the order of
// k_gemm, and the epilogues are k_gemm's (bias + SiLU, then bias and the output scaling of
// k_out): the outputs are the layer-by-layer path's bits whatever RT, without its HBM round trip
// of every layer's activations. The hidden layers' tiles are computed transposed (W H^T), so that
// a lane's four results are four consecutive outputs of one sample: one 8-byte LDS store of two
// packed BF16 conversions each, instead of four 2-byte stores.
template <int CT, int RT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_infer(const float* __restrict__ x, int n, int d_in, int d_out,
                                                      const float* __restrict__ norm, const bf16* __restrict__ wb,
                                                      const float* __restrict__ params, LayerTable L,
                                                      float* __restrict__ y) {
  constexpr int kThreads = 64 * WAVES;
  constexpr int H = 16 * CT * WAVES, ld = H + kPad, kIn = 32, M = 16 * RT;
  extern __shared__ __align__(16) unsigned char infer_smem[];
  bf16* act = reinterpret_cast<bf16*>(infer_smem);
  const long long m0 = static_cast<long long>(blockIdx.x) * M;
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int row = lane % 16, kq = 8 * (lane / 16);
  for (int i = t; i < M * kIn; i += kThreads) {
    const int r = i / kIn, c = i % kIn;
    const long long m = m0 + r;
    act[r * ld + c] = static_cast<bf16>(m < n && c < d_in ? (x[m * d_in + c] - norm[c]) / norm[32 + c] : 0.0f);
  }
  for (int l = 0; l < L.nl; ++l) {
    const int K = l == 0 ? kIn : H;
    const bf16* W = wb + L.w[l];
    const float* bias = params + L.b[l];
    __syncthreads();  // the layer's input is complete
    if (l < L.nl - 1) {
      f32x4 acc[RT][CT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      const int nb = wave * 16 * CT, steps = K / kTileK;
      // The next K step's weights are in flight while this step's products run.
      bf16x8 b_next[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) b_next[j] = packed_operand(W, wave * CT + j, 0, steps);
      for (int k0 = 0; k0 < K; k0 += kTileK) {
        bf16x8 b[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) b[j] = b_next[j];
        if (k0 + kTileK < K) {
#pragma unroll
          for (int j = 0; j < CT; ++j) b_next[j] = packed_operand(W, wave * CT + j, k0 / kTileK + 1, steps);
        }
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(&act[(16 * i + row) * ld + k0 + kq]);
          // The weights as the first operand: the tile is W H^T, so each lane ends with four
          // consecutive outputs of one sample. Every output is the same sum of the same exact
          // BF16 products as in k_gemm's H W^T.
#pragma unroll
          for (int j = 0; j < CT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a, acc[i][j], 0, 0, 0);
        }
      }
      __syncthreads();  // every wave has read the layer's input: the tile takes its output
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        // Lane l holds outputs f .. f + 3 of sample 16 i + l mod 16 of each row tile i.
        const int f = nb + 16 * j + 4 * (lane / 16);
        float bn[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) bn[r] = bias[f + r];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          f32x4 h;
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = silu(acc[i][j][r] + bn[r]);
          *reinterpret_cast<bf16x4*>(&act[(16 * i + lane % 16) * ld + f]) = __builtin_convertvector(h, bf16x4);
        }
      }
    } else {
      // The padded output layer (16 columns): wave w takes the row tiles w, w + 4, ...
      for (int i = wave; i < RT; i += kThreads / 64) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < K; k0 += kTileK) {
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(&act[(16 * i + row) * ld + k0 + kq]);
          const bf16x8 b = packed_operand(W, 0, k0 / kTileK, K / kTileK);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        }
        const int nn = lane % 16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const long long m = m0 + 16 * i + 4 * (lane / 16) + r;
          if (m < n && nn < d_out) {
            const float z = acc[r] + bias[nn];
            y[m * d_out + nn] = z * norm[96 + nn] + norm[64 + nn];
          }
        }
      }
    }
  }
}

// LDS bytes of the tile of 16 rt samples of width h.
constexpr std::size_t infer_lds(int h, int rt) { return std::size_t(16 * rt) * std::size_t(h + kPad) * 2; }

// Launches k_infer<CT, RT, WAVES> for n samples, raising its dynamic LDS limit once per process.
template <int CT, int RT, int WAVES>
void launch_infer(const float* x, int n, int d_in, int d_out, const float* norm, const bf16* wb, const float* params,
                  const LayerTable& L, float* y, hipStream_t s) {
  constexpr int h = 16 * CT * WAVES;
  static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_infer<CT, RT, WAVES>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       static_cast<int>(infer_lds(h, RT)));
  check(raised, "hipFuncSetAttribute(k_infer)");
  const int g = static_cast<int>((static_cast<long long>(n) + 16 * RT - 1) / (16 * RT));
  k_infer<CT, RT, WAVES><<<g, 64 * WAVES, infer_lds(h, RT), s>>>(x, n, d_in, d_out, norm, wb, params, L, y);
}

// The fused forward for hidden width 64 q (q = 1 .. 4) and a tile of `rows` samples: four waves of
// 16 q columns each (64, 96 or 128 samples), or, for 128 samples and an even q, eight waves of 8 q
// columns each (half the accumulators per wave, so twice the waves per SIMD).
template <int Q>
void launch_infer_rows(int rows, const float* x, int n, int d_in, int d_out, const float* norm, const bf16* wb,
                       const float* params, const LayerTable& L, float* y, hipStream_t s) {
  switch (rows) {
    case 64: launch_infer<Q, 4, 4>(x, n, d_in, d_out, norm, wb, params, L, y, s); break;
    case 96: launch_infer<Q, 6, 4>(x, n, d_in, d_out, norm, wb, params, L, y, s); break;
    case 128:
      if constexpr (Q % 2 == 0) {
        launch_infer<Q / 2, 8, 8>(x, n, d_in, d_out, norm, wb, params, L, y, s);
      } else {
        launch_infer<Q, 8, 4>(x, n, d_in, d_out, norm, wb, params, L, y, s);
      }
      break;
    default: throw std::invalid_argument("inference tile: 64, 96 or 128 samples per workgroup");
  }
}

// ------------------------------------------------------------------------ the fused training step
//
// One batch is three kernels (hidden widths up to 256): k_train, the forward, the loss and the
// backward's dZ chain of 32 samples per workgroup, the samples' activations and gradients in LDS; k_dw,
// every layer's weight and bias gradients; k_adam, which adds k_dw's partial sums and takes Adam's
// step. What k_dw contracts over the samples, the activations H and the gradients dZ, is stored by
// k_train as k_dw's matrix-core operands read it: for each tile of 32 samples and each feature four
// packs of eight samples, pack g the samples 4 g .. + 3 and 16 + 4 g .. + 3 (what one lane of a 16 x 16
// product over two row tiles holds of a feature), so that k_dw needs no transposition and no LDS.
constexpr int kPackTile = 32;

// The training step's places: `hidden` layers of width H after 32 inputs, 16 outputs (padded widths),
// `rows` samples (whole tiles). Worked out rather than read from a table in the kernel's arguments,
// whose first reads a workgroup waits on one after the other.
struct TrainPlan {
  int hidden, width;
  long long rows;
  // Layer l's weights in the parameters (its biases follow them), l = 0 .. hidden.
  __host__ __device__ long long w(int l) const {
    const long long H = width;
    return l == 0 ? 0 : 33 * H + (l - 1) * (H * H + H);
  }
  __host__ __device__ long long b(int l) const {
    return w(l) + static_cast<long long>(l == 0 ? 32 : width) * (l == hidden ? 16 : width);
  }
  // The transposed weights of layer l = 1 .. hidden (outputs and inputs exchanged; the output layer's
  // 16 outputs filled up to 32 with zeros).
  __host__ __device__ long long wt(int l) const { return static_cast<long long>(l - 1) * width * width; }
  // Where the partial gradients hold the weight of layer l from input k into output n: 16 x 16 products,
  // lane 16 (n mod 16 / 4) + k mod 16 of each four consecutive outputs. Biases stand at b(l) + n.
  __host__ __device__ long long part_place(int l, int n, int k) const {
    const int kf = (l == 0 ? 32 : width) / 16;
    return w(l) + ((static_cast<long long>(n / 16) * kf + k / 16) * 64 + n % 16 / 4 * 16 + k % 16) * 4 + n % 4;
  }
  // The packs of H_l and dZ_l.
  __host__ __device__ long long h(int l) const { return rows * (l == 0 ? 0 : 32 + width + (l - 1) * 2LL * width); }
  __host__ __device__ long long dz(int l) const { return h(l) + rows * (l == 0 ? 32 : width); }
};

// Every parameter's places: in the packed copies (WeightCopies::at), every layer's weights and the
// transposes of the layers after the first, the backward's operands; and in the partial gradients,
// `order`'s entry there. (A kernel: built by the host and copied, the two tables made a
// 256-wide network of four layers take 2.0 ms to make instead of 1.5.)
__global__ void k_places(TrainPlan P, long long np, int2* __restrict__ at, int* __restrict__ order) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  int l = 0;
  while (l < P.hidden && i >= P.w(l + 1)) ++l;
  const int K = l == 0 ? 32 : P.width, N = l == P.hidden ? 16 : P.width;
  int2 place = make_int2(-1, -1);
  long long part = i;  // a bias
  if (i < P.b(l)) {
    const int n = static_cast<int>((i - P.w(l)) / K), k = static_cast<int>((i - P.w(l)) % K);
    place.x = static_cast<int>(P.w(l) + pack_place(n, k, K / 32));
    if (l > 0) place.y = static_cast<int>(P.wt(l) + pack_place(k, n, (N < 32 ? 32 : N) / 32));
    part = P.part_place(l, n, k);
  }
  at[i] = place;
  order[part] = static_cast<int>(i);
}

// Where a traced batch's tensors go, row-major by layer (for tests): inputs, pre-activations, dZ.
struct TraceTable {
  bf16* h[kMaxLayers];
  float* z[kMaxLayers];
  bf16* dz[kMaxLayers];
};

// A workgroup barrier that orders LDS alone: loads and stores of global memory stay in flight across
// it (__syncthreads waits for them all).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The forward and the dZ chain of RT row tiles of 16 samples, Q = width / 64, 2 Q waves of 32 columns.
// A layer costs its weights' way from L2 to the CU (131 KB at 256 wide, about 1 us) and its
// epilogue's arithmetic: the weights are loaded once per workgroup straight to the lanes that use
// them, all of a layer in flight together while the layer before ends, and one row tile per workgroup
// spreads the epilogues over all CUs up to 8192 samples (512 workgroups, two per CU; 4096 samples 25 us,
// 28 with two row tiles), past which two halve the weights' traffic.
// The pre-activations wait for the backward in `zs`, each lane its own (read by the lane that wrote
// them, from L2). Each product
// accumulates over K in steps of 32 from zero and its epilogue is k_gemm's, so Z, H and dZ are the
// layer-by-layer path's bits. At 4096 samples of 4 x 256 this takes 25 us (38 with
// the weights read by rows), k_dw 11 and k_adam 6, where the 24 launches of the layer-by-layer step
// took 260.
// GATHER: sample i of the batch is idx[batch n + i] of x and t; else sample i.
template <int Q, int RT, bool GATHER, bool TRACE>
__global__ __launch_bounds__(128 * Q) void k_train(const float* __restrict__ x, const float* __restrict__ t, int n,
                                                   int d_in, int d_out, const long long* __restrict__ idx,
                                                   const StepState* __restrict__ st, const float* __restrict__ norm,
                                                   const bf16* __restrict__ wb, const bf16* __restrict__ wbt,
                                                   const float* __restrict__ params, TrainPlan P,
                                                   bf16* __restrict__ packs, f32x4* __restrict__ zs,
                                                   double* __restrict__ sum, TraceTable tr) {
  constexpr int H = 64 * Q, kThreads = 128 * Q, ld = H + kPad, KS = H / kTileK, kIn = 32, ldz = kTileK + kPad, M = 16 * RT;
  __shared__ __align__(16) bf16 act[M * ld];
  __shared__ __align__(16) bf16 dzl[M * ldz];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int row = lane % 16, g = lane / 16, kq = 8 * g, nb = 32 * wave;
  const int m0 = static_cast<int>(blockIdx.x) * M;
  // The tile of 32 samples, and with one row tile which half of its packs.
  const long long tile = m0 / kPackTile;
  const int half = RT == 1 ? m0 / 16 % 2 : 0;
  const long long from = GATHER ? st->batch * n : 0;
  bf16x8 w[KS][2];
  f32x4 acc[RT][2];
  auto load_w = [&](const bf16* W, int steps) {
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (k >= steps) break;
#pragma unroll
      for (int j = 0; j < 2; ++j) w[k][j] = packed_operand(W, 2 * wave + j, k, steps);
    }
  };
  auto product = [&](const bf16* a0, int lda, int steps) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (k >= steps) break;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(a0 + (16 * i + row) * lda + kTileK * k + kq);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[k][j], acc[i][j], 0, 0, 0);
      }
    }
  };
  // Column f of this lane's row tiles (acc's values after an epilogue): the tile's LDS rows for the
  // next product, the pack (or the half of it that this row tile is), the traced tensor.
  auto keep = [&](int f, const f32x4 (&v)[RT], long long at, bf16* traced) {
    bf16x4 c[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      c[i] = __builtin_convertvector(v[i], bf16x4);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        act[(16 * i + 4 * g + r) * ld + f] = c[i][r];
        if constexpr (TRACE) {
          const int m = m0 + 16 * i + 4 * g + r;
          if (m < n) traced[static_cast<long long>(m) * H + f] = c[i][r];
        }
      }
    }
    bf16* p = packs + at + ((tile * H + f) * 4 + g) * 8;
    if constexpr (RT == 2) {
      *reinterpret_cast<bf16x8*>(p) = __builtin_shufflevector(c[0], c[RT - 1], 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      *reinterpret_cast<bf16x4*>(p + 4 * half) = c[0];
    }
  };
  load_w(wb + P.w(0), 1);
  for (int i = tid; i < M * kIn; i += kThreads) {
    const int r = i / kIn, c = i % kIn;
    float v = 0.0f;
    if (m0 + r < n && c < d_in) {
      const long long s = GATHER ? idx[from + m0 + r] : m0 + r;
      v = (x[s * d_in + c] - norm[c]) / norm[32 + c];
    }
    const bf16 b = static_cast<bf16>(v);
    act[r * ld + c] = b;
    if constexpr (TRACE) {
      if (m0 + r < n) tr.h[0][static_cast<long long>(m0 + r) * kIn + c] = b;
    }
  }
  for (int i = tid; i < M * ldz; i += kThreads) dzl[i] = static_cast<bf16>(0.0f);
  lds_barrier();
  // The packs of the first f_count features of an LDS tile of leading dimension lda.
  auto pack_tile = [&](const bf16* a0, int lda, int f_count, long long at) {
    for (int i = tid; i < 4 * RT * f_count; i += kThreads) {
      const int f = i / (4 * RT), p = i / RT % 4, h = i % RT;
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = a0[(16 * h + 4 * p + r) * lda + f];
      *reinterpret_cast<bf16x4*>(packs + at + ((tile * f_count + f) * 4 + p) * 8 + 4 * (half + h)) = v;
    }
  };
  pack_tile(act, ld, kIn, P.h(0));
  const int hidden = P.hidden;
  f32x4* zl = zs + static_cast<long long>(blockIdx.x) * hidden * 2 * RT * kThreads + tid;
  for (int l = 0; l < hidden; ++l) {
    product(act, ld, l == 0 ? 1 : KS);
    // The next product's weights, in flight over this layer's end: the next hidden layer's, or the
    // transposed output weights the backward starts with.
    if (l + 1 < hidden) {
      load_w(wb + P.w(l + 1), KS);
    } else {
      load_w(wbt + P.wt(hidden), 1);
    }
    lds_barrier();  // every wave has read the layer's input: the tile takes its output
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int f = nb + 16 * j + row;
      const float bf = params[P.b(l) + f];
      f32x4 h[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        f32x4 z;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          z[r] = acc[i][j][r] + bf;
          h[i][r] = silu(z[r]);
          if constexpr (TRACE) {
            const int m = m0 + 16 * i + 4 * g + r;
            if (m < n) tr.z[l][static_cast<long long>(m) * H + f] = z[r];
          }
        }
        zl[((2 * l + j) * RT + i) * kThreads] = z;
      }
      keep(f, h, P.h(l + 1), TRACE ? tr.h[l + 1] : nullptr);
    }
    lds_barrier();
  }
  // The output layer (16 columns): wave i the row tile i; then the loss and its gradient.
  if (wave < RT) {
    const bf16* W = wb + P.w(hidden);
    f32x4 o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(&act[(16 * wave + row) * ld + kTileK * k + kq]);
      const bf16x8 b = packed_operand(W, 0, k, KS);
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, o, 0, 0, 0);
    }
    const float bo = params[P.b(hidden) + row];
    float e2 = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ml = 16 * wave + 4 * g + r, m = m0 + ml;
      const float z = o[r] + bo;
      float dv = 0.0f;
      if (m < n && row < d_out) {
        const long long s = GATHER ? idx[from + m] : m;
        const float e = z - (t[s * d_out + row] - norm[64 + row]) / norm[96 + row];
        e2 += e * e;
        dv = 2.0f * e / (static_cast<float>(n) * d_out);
      }
      dzl[ml * ldz + row] = static_cast<bf16>(dv);
      if constexpr (TRACE) {
        if (m < n) {
          tr.z[hidden][static_cast<long long>(m) * 16 + row] = z;
          tr.dz[hidden][static_cast<long long>(m) * 16 + row] = static_cast<bf16>(dv);
        }
      }
    }
#pragma unroll
    for (int o2 = 32; o2 > 0; o2 /= 2) e2 += __shfl_xor(e2, o2);
    if (lane == 0) atomicAdd(sum, static_cast<double>(e2));
  }
  lds_barrier();
  pack_tile(dzl, ldz, 16, P.dz(hidden));
  // dZ_{l-1} = (dZ_l W_l) * silu'(Z_{l-1}).
  for (int l = hidden; l > 0; --l) {
    if (l == hidden) {
      product(dzl, ldz, 1);
    } else {
      product(act, ld, KS);
    }
    if (l > 1) load_w(wbt + P.wt(l - 1), KS);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int f = nb + 16 * j + row;
      f32x4 dv[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const f32x4 z = zl[((2 * (l - 1) + j) * RT + i) * kThreads];
#pragma unroll
        for (int r = 0; r < 4; ++r) dv[i][r] = acc[i][j][r] * silu_grad(z[r]);
      }
      keep(f, dv, P.dz(l - 1), TRACE ? tr.dz[l - 1] : nullptr);
    }
    lds_barrier();
  }
}

// dW_l = dZ_l^T H_l (N_l x K_l) and db_l = the column sums of dZ_l for every layer, over the samples'
// tiles of split blockIdx.x, into partial sums of their own (no atomics; summed in split
// order by k_adam or k_sum_parts, so a step's gradients do not depend on the launch). A workgroup
// has a 64 x 64 tile of one layer, each wave 32 x 32 of it, its operands read as the packs hold them,
// one KB per 16 features and 32 samples, and stores its 16 x 16 products as it holds them, one KB each
// (part_place): rows of a 64 x 64 tile are 1 KB apart, two of the L2's sixteen channels, and those
// stores alone took 13 us.
// With four tiles' packs in flight the loads' latency is hidden by few waves. Block 0 also counts the
// step (the batch, Adam's step and bias corrections), after k_train has read it and before k_adam.
__global__ __launch_bounds__(kThreads) void k_dw(const bf16* __restrict__ packs, TrainPlan P, int tiles, int per_split,
                                                 float* __restrict__ part, long long np, StepState* st, float b1,
                                                 float b2) {
  if (st != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    st->batch += 1;
    st->step += 1;
    const float s = static_cast<float>(st->step);
    st->c1 = 1.0f - powf(b1, s);
    st->c2 = 1.0f - powf(b2, s);
  }
  // The layer and its 64 x 64 tile: q tiles of the first layer, q q of each hidden one, q of the last.
  const int q = P.width / 64;
  int l = 0, at = static_cast<int>(blockIdx.y);
  if (at >= q) {
    l = 1 + (at - q) / (q * q);
    at = (at - q) % (q * q);
  }
  const int nf = l == P.hidden ? 1 : 4 * q, kf = l == 0 ? 2 : 4 * q;  // 16-feature fragments of N_l, K_l
  const int kt = l == 0 ? 1 : q;
  const long long ow = P.w(l), ob = P.b(l);
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int row = lane % 16, g = lane / 16;
  const int n0 = 4 * (at / kt) + 2 * (wave / 2), k0 = 4 * (at % kt) + 2 * (wave % 2);  // fragments
  if (n0 >= nf || k0 >= kf) return;
  const bool n1 = n0 + 1 < nf, k1 = k0 + 1 < kf;
  const bool bias = k0 == 0;
  const bf16* A = packs + P.dz(l) + (16LL * n0 * 4 + 4 * row + g) * 8;
  const bf16* B = packs + P.h(l) + (16LL * k0 * 4 + 4 * row + g) * 8;
  const long long as = 16LL * nf * 32, bs = 16LL * kf * 32;  // values per sample tile
  constexpr int kFrag = 16 * 32;
  f32x4 acc[2][2];
  float db[2] = {0.0f, 0.0f};
  for (int i = 0; i < 2; ++i) {
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // A fragment past the layer's is read as the one before it, and its product not kept.
  const long long a1 = n1 ? kFrag : 0, b1f = k1 ? kFrag : 0;
  auto tiles_of = [&](int t, auto count) {
    constexpr int kCount = decltype(count)::value;
    bf16x8 a[kCount][2], b[kCount][2];
#pragma unroll
    for (int u = 0; u < kCount; ++u) {
      const bf16* pa = A + (t + u) * as;
      const bf16* pb = B + (t + u) * bs;
      a[u][0] = *reinterpret_cast<const bf16x8*>(pa);
      a[u][1] = *reinterpret_cast<const bf16x8*>(pa + a1);
      b[u][0] = *reinterpret_cast<const bf16x8*>(pb);
      b[u][1] = *reinterpret_cast<const bf16x8*>(pb + b1f);
    }
#pragma unroll
    for (int u = 0; u < kCount; ++u) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i], b[u][j], acc[i][j], 0, 0, 0);
      }
    }
    if (bias) {
#pragma unroll
      for (int u = 0; u < kCount; ++u) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
          for (int q8 = 0; q8 < 8; ++q8) db[i] += static_cast<float>(a[u][i][q8]);
        }
      }
    }
  };
  int t = static_cast<int>(blockIdx.x) * per_split;
  const int t1 = min(tiles, t + per_split);
  constexpr int kAhead = 4;
  for (; t + kAhead <= t1; t += kAhead) tiles_of(t, std::integral_constant<int, kAhead>{});
  for (; t < t1; ++t) tiles_of(t, std::integral_constant<int, 1>{});
  float* out = part + static_cast<long long>(blockIdx.x) * np;
  for (int i = 0; i < 2; ++i) {
    if (i == 1 && !n1) break;
    for (int j = 0; j < 2; ++j) {
      if (j == 1 && !k1) break;
      reinterpret_cast<f32x4*>(out + ow)[((n0 + i) * kf + k0 + j) * 64 + lane] = acc[i][j];
    }
    if (bias) {
      float v = db[i];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (g == 0) out[ob + 16 * (n0 + i) + row] = v;
    }
  }
}

__global__ void k_sum_parts(const float* __restrict__ part, long long np, int splits, const int* __restrict__ order,
                            float* __restrict__ g) {
  const long long j = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (j < np) g[order[j]] = sum_parts(part, np, splits, j);
}

template <class T>
class Buf {
 public:
  Buf() = default;
  explicit Buf(std::size_t n) : n_(n) {
    if (n) check(hipMalloc(reinterpret_cast<void**>(&p_), n * sizeof(T)), "hipMalloc");
  }
  Buf(const Buf&) = delete;
  Buf& operator=(const Buf&) = delete;
  Buf(Buf&& o) noexcept : p_(o.p_), n_(o.n_) {
    o.p_ = nullptr;
    o.n_ = 0;
  }
  Buf& operator=(Buf&& o) noexcept {
    std::swap(p_, o.p_);
    std::swap(n_, o.n_);
    return *this;
  }
  ~Buf() {
    if (p_) (void)hipFree(p_);
  }
  T* get() const { return p_; }
  std::size_t size() const { return n_; }

 private:
  T* p_ = nullptr;
  std::size_t n_ = 0;
};

inline int cdiv(long long a, long long b) { return static_cast<int>((a + b - 1) / b); }

class Net {
 public:
  Net(int inputs, int hidden, int layers, int outputs, uint64_t seed) : d_in_(inputs), d_out_(outputs) {
    if (inputs < 1 || inputs > 32 || outputs < 1 || outputs > 16 || hidden < 16 || hidden % 64 != 0 || layers < 1 ||
        layers > 16) {
      throw std::invalid_argument("mlp: 1-32 inputs, 1-16 outputs, hidden a multiple of 64, 1-16 hidden layers");
    }
    check(hipStreamCreateWithFlags(&s_, hipStreamNonBlocking), "hipStreamCreate");
    // Widths: 32 (padded inputs), hidden x layers, 16 (padded outputs).
    w_.push_back(kInPad);
    for (int l = 0; l < layers; ++l) w_.push_back(hidden);
    w_.push_back(kOutPad);
    const int nl = static_cast<int>(w_.size()) - 1;
    std::mt19937_64 rng(seed);
    std::size_t count = 0;
    for (int l = 0; l < nl; ++l) count += (std::size_t(w_[l]) + 1) * std::size_t(w_[l + 1]);
    std::vector<float> host;
    std::vector<unsigned char> mask;
    host.reserve(count);
    mask.reserve(count);
    for (int l = 0; l < nl; ++l) {
      const int K = w_[l], N = w_[l + 1];
      const int k_real = l == 0 ? inputs : K, n_real = l == nl - 1 ? outputs : N;
      woff_.push_back(static_cast<long long>(host.size()));
      // He-style uniform initialisation over the real fan-in; biases zero.
      const float bound = std::sqrt(6.0f / static_cast<float>(k_real));
      std::uniform_real_distribution<float> u(-bound, bound);
      for (int n = 0; n < N; ++n) {
        for (int k = 0; k < K; ++k) {
          const bool real = n < n_real && k < k_real;
          host.push_back(real ? u(rng) : 0.0f);
          mask.push_back(real ? 1 : 0);
        }
      }
      boff_.push_back(static_cast<long long>(host.size()));
      for (int n = 0; n < N; ++n) {
        host.push_back(0.0f);
        mask.push_back(n < n_real ? 1 : 0);
      }
    }
    np_ = static_cast<long long>(host.size());
    params_ = Buf<float>(std::size_t(np_));
    grads_ = Buf<float>(std::size_t(np_));
    m1_ = Buf<float>(std::size_t(np_));
    m2_ = Buf<float>(std::size_t(np_));
    wb_ = Buf<bf16>(std::size_t(np_));
    mask_ = Buf<unsigned char>(std::size_t(np_));
    if (fused_width()) {
      const TrainPlan plan{layers, hidden, 0};
      const std::size_t nt = std::size_t(plan.wt(layers)) + std::size_t(hidden) * 32;
      place_ = Buf<int2>(std::size_t(np_));
      order_ = Buf<int>(std::size_t(np_));
      wp_ = Buf<bf16>(std::size_t(np_));
      wt_ = Buf<bf16>(nt);
      check(hipMemsetAsync(wt_.get(), 0, nt * sizeof(bf16), s_), "hipMemsetAsync");
      k_places<<<cdiv(np_, 256), 256, 0, s_>>>(plan, np_, place_.get(), order_.get());
      check(hipGetLastError(), "k_places");
    }
    check(hipMemcpy(params_.get(), host.data(), np_ * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
    check(hipMemcpy(mask_.get(), mask.data(), np_, hipMemcpyHostToDevice), "hipMemcpy");
    check(hipMemset(m1_.get(), 0, np_ * sizeof(float)), "hipMemset");
    check(hipMemset(m2_.get(), 0, np_ * sizeof(float)), "hipMemset");
    state_ = Buf<StepState>(1);
    check(hipMemset(state_.get(), 0, sizeof(StepState)), "hipMemset");
    refresh_bf16();
    std::vector<float> ones(32, 1.0f), zeros(32, 0.0f);
    norm_ = Buf<float>(4 * 32);
    set_normalization(zeros.data(), ones.data(), zeros.data(), ones.data());
  }
  ~Net() {
    (void)hipStreamSynchronize(s_);
    (void)hipStreamDestroy(s_);
  }

  long long param_count() const { return np_; }
  int layers() const { return static_cast<int>(w_.size()) - 1; }

  void set_normalization(const float* in_mean, const float* in_scale, const float* out_mean, const float* out_scale) {
    std::vector<float> h(4 * 32, 0.0f);
    for (int i = 0; i < 32; ++i) h[32 + i] = h[96 + i] = 1.0f;
    for (int i = 0; i < d_in_; ++i) {
      h[i] = in_mean[i];
      h[32 + i] = in_scale[i];
      if (!(in_scale[i] > 0.0f)) throw std::invalid_argument("mlp: input scales must be positive");
    }
    for (int i = 0; i < d_out_; ++i) {
      h[64 + i] = out_mean[i];
      h[96 + i] = out_scale[i];
      if (!(out_scale[i] > 0.0f)) throw std::invalid_argument("mlp: output scales must be positive");
    }
    check(hipMemcpy(norm_.get(), h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
  }

  void get_params(float* out) {
    check(hipMemcpy(out, params_.get(), np_ * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
  }
  void set_params(const float* in) {
    check(hipMemcpy(params_.get(), in, np_ * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
    refresh_bf16();
  }

  // Forward of n samples (host arrays, n x inputs -> n x outputs, physical units).
  void predict(const float* x, long long n, float* y) {
    const long long chunk = std::min(n, fused_inference() ? kChunk : kLayeredChunk);
    Staging staging(*this, chunk);
    const Buf<float>&xd = staging.x(), &yd = staging.t();
    for (long long at = 0; at < n; at += chunk) {
      const int m = static_cast<int>(std::min(chunk, n - at));
      check(hipMemcpyAsync(xd.get(), x + at * d_in_, std::size_t(m) * d_in_ * sizeof(float), hipMemcpyHostToDevice, s_),
            "hipMemcpyAsync");
      infer(xd.get(), m, yd.get());
      check(hipMemcpyAsync(y + at * d_out_, yd.get(), std::size_t(m) * d_out_ * sizeof(float), hipMemcpyDeviceToHost, s_),
            "hipMemcpyAsync");
      check(hipStreamSynchronize(s_), "predict");
    }
    staging.keep();
  }

  // Loss and gradients (FP32, in parameter order) of one batch; grads may be null.
  float gradients(const float* x, const float* t, int n, float* grads) {
    Staging staging(*this, n);
    const Buf<float>&xd = staging.x(), &td = staging.t();
    check(hipMemcpyAsync(xd.get(), x, std::size_t(n) * d_in_ * sizeof(float), hipMemcpyHostToDevice, s_), "hipMemcpy");
    check(hipMemcpyAsync(td.get(), t, std::size_t(n) * d_out_ * sizeof(float), hipMemcpyHostToDevice, s_), "hipMemcpy");
    ensure_loss();
    check(hipMemsetAsync(loss_sum_.get(), 0, sizeof(double), s_), "hipMemsetAsync");
    if (fused_width()) {
      train_batch<false>(xd.get(), td.get(), n, nullptr);
      k_sum_parts<<<cdiv(np_, 256), 256, 0, s_>>>(part_.get(), np_, splits_of(n), order_.get(), grads_.get());
      check(hipGetLastError(), "k_sum_parts");
    } else {
      backward(xd.get(), td.get(), n);
    }
    double sum = 0.0;
    check(hipMemcpyAsync(&sum, loss_sum_.get(), sizeof(double), hipMemcpyDeviceToHost, s_), "hipMemcpyAsync");
    check(hipStreamSynchronize(s_), "gradients");
    staging.keep();
    const float loss = static_cast<float>(sum / (static_cast<double>(n) * d_out_));
    if (grads != nullptr) check(hipMemcpy(grads, grads_.get(), np_ * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
    return loss;
  }

  // One batch's forward and backward, then one of its tensors to the host as FP32, row-major
  // n x width: what 0 the input activations of layer `layer` (BF16: the normalised inputs for
  // layer 0), 1 its pre-activations Z (FP32), 2 the gradient dZ of its pre-activations (BF16).
  void trace(const float* x, const float* t, int n, int what, int layer, float* out) {
    const int nl = layers();
    if (layer < 0 || layer >= nl || what < 0 || what > 2) throw std::invalid_argument("trace: no such tensor");
    Buf<float> xd(std::size_t(n) * d_in_), td(std::size_t(n) * d_out_);
    check(hipMemcpyAsync(xd.get(), x, std::size_t(n) * d_in_ * sizeof(float), hipMemcpyHostToDevice, s_), "hipMemcpy");
    check(hipMemcpyAsync(td.get(), t, std::size_t(n) * d_out_ * sizeof(float), hipMemcpyHostToDevice, s_), "hipMemcpy");
    ensure(n);
    ensure_loss();
    check(hipMemsetAsync(loss_sum_.get(), 0, sizeof(double), s_), "hipMemsetAsync");
    if (fused_width()) {
      TraceTable tr{};
      for (std::size_t q = 0; q < std::size_t(nl); ++q) {
        tr.h[q] = acts_[q].get();
        tr.z[q] = z_[q].get();
        tr.dz[q] = dz_[q].get();
      }
      train_batch<false>(xd.get(), td.get(), n, &tr);
    } else {
      backward(xd.get(), td.get(), n);
    }
    const std::size_t l = static_cast<std::size_t>(layer);
    const std::size_t count = std::size_t(n) * std::size_t(what == 0 ? w_[l] : w_[l + 1]);
    if (what == 1) {
      check(hipMemcpyAsync(out, z_[l].get(), count * sizeof(float), hipMemcpyDeviceToHost, s_), "hipMemcpy");
      check(hipStreamSynchronize(s_), "trace");
      return;
    }
    std::vector<bf16> h(count);
    const bf16* src = what == 0 ? acts_[l].get() : dz_[l].get();
    check(hipMemcpyAsync(h.data(), src, count * sizeof(bf16), hipMemcpyDeviceToHost, s_), "hipMemcpy");
    check(hipStreamSynchronize(s_), "trace");
    for (std::size_t i = 0; i < count; ++i) out[i] = static_cast<float>(h[i]);
  }

  // Training data resident on the device; epochs of shuffled batches with Adam.
  void set_data(const float* x, const float* t, long long n) {
    // Without data until all of it is there: after a failed allocation train() refuses, and the next
    // call makes every buffer again.
    const bool as_many = n == n_data_;
    n_data_ = 0;
    if (!as_many) {
      data_x_ = Buf<float>(std::size_t(n) * d_in_);
      data_t_ = Buf<float>(std::size_t(n) * d_out_);
      idx_ = Buf<long long>(std::size_t(n));
    }
    check(hipMemcpy(data_x_.get(), x, std::size_t(n) * d_in_ * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
    check(hipMemcpy(data_t_.get(), t, std::size_t(n) * d_out_ * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
    n_data_ = n;
  }

  // `epochs` passes over the data in batches of `batch` (the order shuffled per epoch with
  // `seed`), one Adam step each. Returns the last epoch's mean batch loss.
  float train(int epochs, int batch, float lr, uint64_t seed, double* seconds) {
    if (n_data_ < batch || batch < 64) throw std::invalid_argument("mlp: batch >= 64 and <= the data");
    const long long nb = n_data_ / batch;
    const bool fused = fused_width();
    Buf<float> bx(fused ? 0 : std::size_t(batch) * d_in_), bt(fused ? 0 : std::size_t(batch) * d_out_);
    const Buf<long long>& idx = idx_;
    std::vector<long long> order(static_cast<std::size_t>(n_data_));
    std::mt19937_64 rng(seed);
    float last = 0.0f;
    hipGraphExec_t step_graph = nullptr;
    struct GraphGuard {
      hipGraphExec_t* g;
      ~GraphGuard() {
        if (*g != nullptr) (void)hipGraphExecDestroy(*g);
      }
    } guard{&step_graph};
    hipEvent_t e0, e1;
    check(hipEventCreate(&e0), "hipEventCreate");
    check(hipEventCreate(&e1), "hipEventCreate");
    check(hipEventRecord(e0, s_), "hipEventRecord");
    for (int ep = 0; ep < epochs; ++ep) {
      for (long long i = 0; i < n_data_; ++i) order[std::size_t(i)] = i;
      std::shuffle(order.begin(), order.end(), rng);
      check(hipMemcpyAsync(idx.get(), order.data(), order.size() * sizeof(long long), hipMemcpyHostToDevice, s_),
            "hipMemcpyAsync");
      if (fused) {
        ensure_packs(batch);
      } else {
        ensure(batch);
      }
      ensure_loss();
      check(hipMemsetAsync(loss_sum_.get(), 0, sizeof(double), s_), "hipMemsetAsync");
      k_set_batch<<<1, 1, 0, s_>>>(state_.get(), 0);
      check(hipGetLastError(), "k_set_batch");
      if (fused) {
        // Three launches a step: plain ones keep ahead of the GPU (a graph of one step leaves 8 us
        // between replays).
        for (long long b = 0; b < nb; ++b) {
          train_batch<true>(data_x_.get(), data_t_.get(), batch, nullptr, idx.get());
          adam(lr, part_.get(), splits_of(batch), order_.get());
        }
      } else if (step_graph == nullptr) {
        // One step (gather of the state's batch, forward, loss, backward, Adam, next batch)
        // recorded once and replayed for every batch: its launches cost one graph launch.
        check(hipStreamBeginCapture(s_, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        hipGraph_t g = nullptr;
        try {
          k_gather<<<cdiv(batch, 256), 256, 0, s_>>>(idx.get(), state_.get(), batch, data_x_.get(), d_in_,
                                                     data_t_.get(), d_out_, bx.get(), bt.get());
          check(hipGetLastError(), "k_gather");
          backward(bx.get(), bt.get(), batch);
          next_step();
          adam(lr, grads_.get(), 1, nullptr);
        } catch (...) {
          (void)hipStreamEndCapture(s_, &g);
          if (g != nullptr) (void)hipGraphDestroy(g);
          throw;
        }
        check(hipStreamEndCapture(s_, &g), "hipStreamEndCapture");
        const hipError_t e = hipGraphInstantiate(&step_graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        check(e, "hipGraphInstantiate");
      }
      for (long long b = 0; b < nb && !fused; ++b) check(hipGraphLaunch(step_graph, s_), "hipGraphLaunch");
      double sum = 0.0;
      check(hipMemcpyAsync(&sum, loss_sum_.get(), sizeof(double), hipMemcpyDeviceToHost, s_), "hipMemcpyAsync");
      check(hipStreamSynchronize(s_), "train");
      last = static_cast<float>(sum / (static_cast<double>(nb) * batch * d_out_));
    }
    check(hipEventRecord(e1, s_), "hipEventRecord");
    check(hipEventSynchronize(e1), "hipEventSynchronize");
    float ms = 0.0f;
    check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
    if (seconds) *seconds = ms * 1e-3;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return last;
  }

  void adam_step(float lr) {
    next_step();
    adam(lr, grads_.get(), 1, nullptr);
    check(hipStreamSynchronize(s_), "adam");
  }

  // Inference: n device-resident samples to n x outputs in physical units, by the fused forward
  // (hidden widths up to 256) or, with fused_ off or wider layers, the training path's
  // layer-by-layer products; the same bits either way.
  void infer(const float* x, int n, float* y) {
    const int h = w_[1];
    if (fused_inference()) {
      LayerTable L{};
      L.nl = layers();
      for (int l = 0; l < L.nl; ++l) {
        L.w[l] = woff_[std::size_t(l)];
        L.b[l] = boff_[std::size_t(l)];
      }
      const float* nm = norm_.get();
      const float* pr = params_.get();
      switch (h / 64) {
        case 1: launch_infer_rows<1>(infer_rows_, x, n, d_in_, d_out_, nm, wp_.get(), pr, L, y, s_); break;
        case 2: launch_infer_rows<2>(infer_rows_, x, n, d_in_, d_out_, nm, wp_.get(), pr, L, y, s_); break;
        case 3: launch_infer_rows<3>(infer_rows_, x, n, d_in_, d_out_, nm, wp_.get(), pr, L, y, s_); break;
        default: launch_infer_rows<4>(infer_rows_, x, n, d_in_, d_out_, nm, wp_.get(), pr, L, y, s_); break;
      }
      check(hipGetLastError(), "k_infer");
      return;
    }
    forward(x, n);
    k_out<<<cdiv(static_cast<long long>(n) * d_out_, 256), 256, 0, s_>>>(z_.back().get(), n, d_out_, kOutPad,
                                                                         norm_.get() + 64, norm_.get() + 96, y);
    check(hipGetLastError(), "k_out");
  }

  void set_fused(bool on) { fused_ = on; }
  void set_infer_rows(int rows) {
    if (rows != 64 && rows != 96 && rows != 128)
      throw std::invalid_argument("inference tile: 64, 96 or 128 samples per workgroup");
    infer_rows_ = rows;
  }

  // Milliseconds of one inference of n samples (device-resident inputs and outputs, HIP events).
  double time_forward(int n, int repeats) {
    Buf<float> xd(std::size_t(n) * d_in_), yd(std::size_t(n) * d_out_);
    check(hipMemsetAsync(xd.get(), 0, std::size_t(n) * d_in_ * sizeof(float), s_), "hipMemset");
    infer(xd.get(), n, yd.get());
    hipEvent_t e0, e1;
    check(hipEventCreate(&e0), "hipEventCreate");
    check(hipEventCreate(&e1), "hipEventCreate");
    check(hipEventRecord(e0, s_), "hipEventRecord");
    for (int r = 0; r < repeats; ++r) infer(xd.get(), n, yd.get());
    check(hipEventRecord(e1, s_), "hipEventRecord");
    check(hipEventSynchronize(e1), "hipEventSynchronize");
    float ms = 0.0f;
    check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return ms / repeats;
  }

 private:
  static constexpr int kInPad = 32, kOutPad = 16;

  // Samples predict takes to the device at a time: with the fused forward, which needs no memory beside
  // the samples, and layer by layer, which holds every layer's activations, pre-activations and room
  // for their gradients (8 bytes of each width per sample, kept: 8.6 GB for 16 layers of 1024).
  static constexpr long long kChunk = 1 << 18, kLayeredChunk = 1 << 16;

  // A call's device copies of n host samples: their inputs, and their targets or outputs. The call
  // has them to itself: another one at the same time (mxmlp_predict may be called from several host
  // threads) finds none kept and allocates its own, as every call would. One pair of at most kChunk
  // samples (48 MB with every input and output in use) is kept between calls, for its two
  // allocations and frees (83,300 predictions: 293 us with them, 250 without).
  class Staging {
   public:
    Staging(Net& net, long long n) : net_(net) {
      {
        const std::lock_guard<std::mutex> lock(net_.staging_mutex_);
        std::swap(x_, net_.staging_x_);
        std::swap(t_, net_.staging_t_);
      }
      if (x_.size() < std::size_t(n) * net_.d_in_) x_ = Buf<float>(std::size_t(n) * net_.d_in_);
      if (t_.size() < std::size_t(n) * net_.d_out_) t_ = Buf<float>(std::size_t(n) * net_.d_out_);
    }
    Buf<float>& x() { return x_; }
    Buf<float>& t() { return t_; }
    // Given back for a later call, the call's work on the stream being done (a call that throws frees them).
    void keep() {
      if (x_.size() > std::size_t(kChunk) * net_.d_in_ || t_.size() > std::size_t(kChunk) * net_.d_out_) return;
      const std::lock_guard<std::mutex> lock(net_.staging_mutex_);
      if (net_.staging_x_.size() >= x_.size()) return;  // another call's, as large
      std::swap(x_, net_.staging_x_);
      std::swap(t_, net_.staging_t_);
    }

   private:
    Net& net_;
    Buf<float> x_, t_;
  };

  // The fused kernels, of inference and of training, are built for these widths; wider networks run and
  // train layer by layer.
  bool fused_width() const { return w_[1] <= 256 && layers() <= kMaxLayers; }
  bool fused_inference() const { return fused_ && fused_width(); }

  void refresh_bf16() {
    k_to_bf16<<<cdiv(np_, 256), 256, 0, s_>>>(params_.get(), np_, copies());
    check(hipGetLastError(), "k_to_bf16");
    check(hipStreamSynchronize(s_), "refresh");
  }

  void ensure(int n) {
    if (n <= cap_) return;
    cap_ = n;
    acts_.clear();
    z_.clear();
    dz_.clear();
    acts_.emplace_back(std::size_t(n) * kInPad);
    for (std::size_t l = 1; l < w_.size(); ++l) {
      acts_.emplace_back(std::size_t(n) * w_[l]);
      z_.emplace_back(std::size_t(n) * w_[l]);
      dz_.emplace_back(std::size_t(n) * w_[l]);
    }
  }

  void ensure_loss() {
    if (loss_sum_.size() == 0) loss_sum_ = Buf<double>(1);
  }

  // Up to this many samples a workgroup takes one row tile.
  static constexpr int kOneRowTile = 8192;
  static int tiles_of(int n) { return cdiv(n, kPackTile); }
  // Partial gradients of a batch: eight sample tiles each where that gives at most 8, one per XCD (at 56
  // tiles of weights for four hidden layers of 256, 4096 samples then make 448 workgroups; 16 take the
  // same 11 us and cost k_adam 1 more). From 4608 samples on, one per 512 samples up to 32, so that no
  // FP32 chain gets longer than the layer-by-layer step's: with 8 a weight gradient's error against 64
  // bits was 2.4e-7 of it at 131072 samples and 6e-7 at 524288, now 1.1e-7 and 1.5e-7, as there; and a
  // narrow network, of few tiles of weights, has more workgroups (128-wide, three layers: 347 us a batch
  // of 65536 with 8, 289 now; four layers of 256 at 8192: 86 and 87 us).
  static int splits_of(int n) {
    const int tiles = tiles_of(n), want = std::max(std::min(8, cdiv(tiles, 8)), std::min(32, tiles / 16));
    return cdiv(tiles, cdiv(tiles, want));
  }

  // The packs, pre-activations and partial gradients of batches of up to n samples.
  void ensure_packs(int n) {
    const int splits = splits_of(n);
    if (splits > part_splits_) {
      part_ = Buf<float>(std::size_t(splits) * std::size_t(np_));
      part_splits_ = splits;
    }
    if (n <= pack_cap_) return;
    const std::size_t rows = std::size_t(tiles_of(n)) * kPackTile;
    const std::size_t hidden = w_.size() - 2;
    packs_ = Buf<bf16>(rows * (kInPad + kOutPad + 2 * hidden * std::size_t(w_[1])));
    zs_ = Buf<f32x4>(rows * hidden * std::size_t(w_[1]) / 4);
    pack_cap_ = n;
  }

  // The forward, loss and gradients of one batch of device-resident samples (of `idx`'s batch of the
  // state, with GATHER): the partial gradients into part_, the squared errors added to loss_sum_. With
  // GATHER it also counts the step. No host synchronisation.
  template <bool GATHER>
  void train_batch(const float* x, const float* t, int n, const TraceTable* tr, const long long* idx = nullptr) {
    ensure_packs(n);
    const int tiles = tiles_of(n), width = w_[1], q = width / 64;
    const TrainPlan plan{layers() - 1, width, static_cast<long long>(tiles) * kPackTile};
    auto run = [&](auto quarter, auto row_tiles, auto traced) {
      constexpr int Q = decltype(quarter)::value, RT = decltype(row_tiles)::value;
      k_train<Q, RT, GATHER, decltype(traced)::value><<<tiles * (2 / RT), 128 * Q, 0, s_>>>(
          x, t, n, d_in_, d_out_, idx, state_.get(), norm_.get(), wp_.get(), wt_.get(), params_.get(), plan,
          packs_.get(), zs_.get(), loss_sum_.get(), tr != nullptr ? *tr : TraceTable{});
    };
    auto sized = [&](auto quarter, auto traced) {
      if (n <= kOneRowTile) {
        run(quarter, std::integral_constant<int, 1>{}, traced);
      } else {
        run(quarter, std::integral_constant<int, 2>{}, traced);
      }
    };
    auto pick = [&](auto traced) {
      switch (q) {
        case 1: sized(std::integral_constant<int, 1>{}, traced); break;
        case 2: sized(std::integral_constant<int, 2>{}, traced); break;
        case 3: sized(std::integral_constant<int, 3>{}, traced); break;
        default: sized(std::integral_constant<int, 4>{}, traced); break;
      }
    };
    if constexpr (!GATHER) {
      if (tr != nullptr) {
        pick(std::true_type{});
      } else {
        pick(std::false_type{});
      }
    } else {
      pick(std::false_type{});
    }
    check(hipGetLastError(), "k_train");
    const int splits = splits_of(n);
    const int weight_tiles = 2 * q + (plan.hidden - 1) * q * q;
    k_dw<<<dim3(splits, weight_tiles), kThreads, 0, s_>>>(packs_.get(), plan, tiles, cdiv(tiles, splits), part_.get(), np_,
                                                  GATHER ? state_.get() : nullptr, kBeta1, kBeta2);
    check(hipGetLastError(), "k_dw");
  }

  template <bool TA, bool TB, int EPI>
  void gemm(const bf16* A, const bf16* B, int M, int N, int K, int lda, int ldb, float* Cf, bf16* Hb, const float* bias,
            int ldc, int splits = 1) {
    const int kchunk = ((cdiv(K, splits) + kTileK - 1) / kTileK) * kTileK;
    dim3 grid(cdiv(N, kTileN), cdiv(M, kTileM), cdiv(K, kchunk));
    k_gemm<TA, TB, EPI><<<grid, kThreads, 0, s_>>>(A, B, M, N, K, lda, ldb, kchunk, Cf, Hb, bias, ldc);
    check(hipGetLastError(), "k_gemm");
  }

  const bf16* W(int l) const { return wb_.get() + woff_[std::size_t(l)]; }
  const float* bias(int l) const { return params_.get() + boff_[std::size_t(l)]; }

  void forward(const float* x, int n) {
    ensure(n);
    k_inputs<<<cdiv(static_cast<long long>(n) * kInPad, 256), 256, 0, s_>>>(x, n, d_in_, norm_.get(), norm_.get() + 32,
                                                                             acts_[0].get(), kInPad);
    check(hipGetLastError(), "k_inputs");
    const int nl = layers();
    for (int l = 0; l < nl; ++l) {
      const int K = w_[std::size_t(l)], N = w_[std::size_t(l) + 1];
      if (l < nl - 1) {
        gemm<false, true, kBiasSiLU>(acts_[std::size_t(l)].get(), W(l), n, N, K, K, K, z_[std::size_t(l)].get(),
                                      acts_[std::size_t(l) + 1].get(), bias(l), N);
      } else {
        gemm<false, true, kBias>(acts_[std::size_t(l)].get(), W(l), n, N, K, K, K, z_[std::size_t(l)].get(), nullptr,
                                 bias(l), N);
      }
    }
  }


  // Forward and backward of one batch: gradients into grads_, the squared errors added to
  // loss_sum_ (cleared by the caller). No host synchronisation.
  void backward(const float* x, const float* t, int n) {
    forward(x, n);
    const int nl = layers();
    const int blocks = cdiv(static_cast<long long>(n) * kOutPad, 256);
    k_loss<<<blocks, 256, 0, s_>>>(z_.back().get(), t, n, d_out_, kOutPad, norm_.get() + 64, norm_.get() + 96,
                                  dz_.back().get(), loss_sum_.get());
    check(hipGetLastError(), "k_loss");
    k_fill<<<cdiv(np_, 256), 256, 0, s_>>>(grads_.get(), np_, 0.0f);  // a kernel: the step may be recorded
    check(hipGetLastError(), "k_fill");
    const int splits = std::max(1, std::min(32, n / 512));
    for (int l = nl - 1; l >= 0; --l) {
      const int K = w_[std::size_t(l)], N = w_[std::size_t(l) + 1];
      // dW_l = dZ_l^T H_{l-1} (N x K, over the samples), db_l = column sums of dZ_l.
      gemm<true, false, kAtomicF32>(dz_[std::size_t(l)].get(), acts_[std::size_t(l)].get(), N, K, n, N, K,
                                    grads_.get() + woff_[std::size_t(l)], nullptr, nullptr, K, splits);
      k_colsum<<<dim3(cdiv(N, 64), std::min(n, 256)), 64, 0, s_>>>(dz_[std::size_t(l)].get(), n, N,
                                                                    grads_.get() + boff_[std::size_t(l)]);
      check(hipGetLastError(), "k_colsum");
      if (l > 0) {
        // dZ_{l-1} = (dZ_l W_l) * silu'(Z_{l-1}).
        gemm<false, false, kSiLUGrad>(dz_[std::size_t(l)].get(), W(l), n, K, N, N, K, z_[std::size_t(l) - 1].get(),
                                      dz_[std::size_t(l) - 1].get(), nullptr, K);
      }
    }
  }

  WeightCopies copies() const { return {wb_.get(), wp_.get(), wt_.get(), place_.get()}; }

  void next_step() {
    k_next_step<<<1, 1, 0, s_>>>(state_.get(), kBeta1, kBeta2);
    check(hipGetLastError(), "k_next_step");
  }

  // Adam's update of the counted step, by the sum of `splits` partial gradients.
  void adam(float lr, const float* part, int splits, const int* order) {
    k_adam<<<cdiv(np_, 256), 256, 0, s_>>>(params_.get(), part, splits, order, m1_.get(), m2_.get(), mask_.get(), np_, lr,
                                           kBeta1, kBeta2, 1e-8f, state_.get(), copies());
    check(hipGetLastError(), "k_adam");
  }

  static constexpr float kBeta1 = 0.9f, kBeta2 = 0.999f;
  int d_in_, d_out_;
  hipStream_t s_ = nullptr;
  std::vector<int> w_;
  std::vector<long long> woff_, boff_;
  long long np_ = 0;
  Buf<float> params_, grads_, m1_, m2_, norm_;
  Buf<StepState> state_;
  Buf<double> loss_sum_;
  Buf<bf16> wb_;  // the BF16 weights by row
  // For the fused kernels, at their widths alone: the weights packed and packed transposed, each
  // parameter's places there, and the parameter at each place of the partial gradients.
  Buf<bf16> wp_, wt_;
  Buf<int2> place_;
  Buf<int> order_;
  Buf<bf16> packs_;
  Buf<f32x4> zs_;
  Buf<float> part_;
  int pack_cap_ = 0, part_splits_ = 0;
  Buf<unsigned char> mask_;
  std::vector<Buf<bf16>> acts_, dz_;
  std::vector<Buf<float>> z_;
  int cap_ = 0;
  bool fused_ = true;
  int infer_rows_ = 128;  // the fastest tile on an MI355X (eight waves, 4 waves per SIMD)
  Buf<float> data_x_, data_t_;
  Buf<long long> idx_;             // the epoch's order
  std::mutex staging_mutex_;
  Buf<float> staging_x_, staging_t_;  // the pair kept between calls (Staging)
  long long n_data_ = 0;
};

int fail(const std::exception& e, char* err, size_t len) {
  if (err != nullptr && len > 0) {
    std::strncpy(err, e.what(), len - 1);
    err[len - 1] = '\0';
  }
  return 1;
}

template <class F>
int guarded(char* err, size_t len, F&& f) {
  try {
    f();
    return 0;
  } catch (const std::exception& e) {
    return fail(e, err, len);
  }
}

}  // namespace mxm

struct mxmlp {
  std::unique_ptr<mxm::Net> net;
};

extern "C" {

int mxmlp_create(int32_t inputs, int32_t hidden, int32_t layers, int32_t outputs, uint64_t seed, mxmlp** out, char* err,
                 size_t err_len) {
  return mxm::guarded(err, err_len, [&] {
    if (!out) throw std::invalid_argument("null argument");
    auto h = std::make_unique<mxmlp>();
    h->net = std::make_unique<mxm::Net>(inputs, hidden, layers, outputs, seed);
    *out = h.release();
  });
}

void mxmlp_destroy(mxmlp* h) { delete h; }

int64_t mxmlp_param_count(const mxmlp* h) { return h ? h->net->param_count() : 0; }

int mxmlp_set_normalization(mxmlp* h, const float* in_mean, const float* in_scale, const float* out_mean,
                            const float* out_scale, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->set_normalization(in_mean, in_scale, out_mean, out_scale); });
}

int mxmlp_get_params(mxmlp* h, float* params, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->get_params(params); });
}

int mxmlp_set_params(mxmlp* h, const float* params, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->set_params(params); });
}

int mxmlp_predict(mxmlp* h, const float* x, int64_t n, float* y, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] {
    if (n < 0) throw std::invalid_argument("n < 0");
    h->net->predict(x, n, y);
  });
}

int mxmlp_gradients(mxmlp* h, const float* x, const float* t, int32_t n, float* grads, float* loss, char* err,
                    size_t err_len) {
  return mxm::guarded(err, err_len, [&] {
    if (n < 1) throw std::invalid_argument("n >= 1");
    *loss = h->net->gradients(x, t, n, grads);
  });
}

int mxmlp_trace(mxmlp* h, const float* x, const float* t, int32_t n, int32_t what, int32_t layer, float* out,
                char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] {
    if (n < 1 || !x || !t || !out) throw std::invalid_argument("trace: n >= 1 and arrays");
    h->net->trace(x, t, n, what, layer, out);
  });
}

int mxmlp_adam_step(mxmlp* h, float lr, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->adam_step(lr); });
}

int mxmlp_set_data(mxmlp* h, const float* x, const float* t, int64_t n, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->set_data(x, t, n); });
}

int mxmlp_train(mxmlp* h, int32_t epochs, int32_t batch, float lr, uint64_t seed, float* loss, double* seconds,
                char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { *loss = h->net->train(epochs, batch, lr, seed, seconds); });
}

int mxmlp_time_forward(mxmlp* h, int32_t n, int32_t repeats, double* ms, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] {
    if (n < 1 || repeats < 1) throw std::invalid_argument("n >= 1 and repeats >= 1");
    *ms = h->net->time_forward(n, repeats);
  });
}

int mxmlp_set_fused(mxmlp* h, int32_t on, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->set_fused(on != 0); });
}

int mxmlp_set_infer_rows(mxmlp* h, int32_t rows, char* err, size_t err_len) {
  return mxm::guarded(err, err_len, [&] { h->net->set_infer_rows(rows); });
}

}  // extern "C"
