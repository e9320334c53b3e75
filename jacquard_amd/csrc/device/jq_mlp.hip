// FP32 MLP (in -> h1 -> h2 -> 1, ReLU) for the learned partition cost model:
// forward, mean-squared-error backward and SGD, hand-written for gfx950.
//
// Parameters are packed W1[h1][in], b1[h1], W2[h2][h1], b2[h2], W3[h2], b3.
// Training is deterministic: each workgroup writes the gradient of its 64
// samples to its own workspace row, a second kernel sums the rows in a
// fixed order and applies the update.
//
// Every matrix product runs on the matrix cores in FP32
// (v_mfma_f32_16x16x4_f32: FP32 inputs, FP32 accumulation).  A pair of waves
// owns 16 samples from their inputs to their pre-activation gradients, each
// wave half of a layer's units; then the pair owns 16 rows of each weight
// gradient.  Dimensions are padded with zeros to multiples of 16 in LDS.
// What bounds it is the chain load - layer - layer - ... of one workgroup
// per 64 samples, whose products are a dependent chain per tile.  A thread
// per sample (its activations in scratch, weights read one by one) kept one
// wave of a workgroup busy: a step of 4096 samples took 340 us and takes
// 20.4 (gradients 16, update 5), a forward of 5013 samples 140 and 6.8, with
// the same result bit for bit.  One wave to 16 samples: 23.3 and 6.9.
#include <hip/hip_runtime.h>

#include <mutex>

#include "jq_common.hpp"

namespace jqd {
namespace {

constexpr int kMaxIn = 32, kMaxH = 64, kSamples = 64;

// Workspace of jq_mlp_train_step_noalloc: the per-workgroup gradient rows
// and losses of a batch of at most kNoAllocMaxSamples samples at the largest
// dimensions (64 rows of 6337 parameters + 64 losses, 1.6 MB).  Every GPU
// the library runs on holds its own copy until the process ends.
constexpr int kNoAllocMaxSamples = 4096;
constexpr size_t kNoAllocFloats =
    (size_t)(kNoAllocMaxSamples / kSamples) *
        (kMaxH * kMaxIn + kMaxH + kMaxH * kMaxH + kMaxH + kMaxH + 1) +
    kNoAllocMaxSamples / kSamples;
__device__ __align__(256) float scratch[kNoAllocFloats];

struct Dims {
  int in, h1, h2, np;
  __host__ __device__ int oW1() const { return 0; }
  __host__ __device__ int ob1() const { return h1 * in; }
  __host__ __device__ int oW2() const { return ob1() + h1; }
  __host__ __device__ int ob2() const { return oW2() + h2 * h1; }
  __host__ __device__ int oW3() const { return ob2() + h2; }
  __host__ __device__ int ob3() const { return oW3() + h2; }
};

inline Dims dims(int in, int h1, int h2) {
  Dims d{in, h1, h2, 0};
  d.np = d.ob3() + 1;
  return d;
}

using f4 = __attribute__((ext_vector_type(4))) float;

// LDS rows are padded by 4 floats so that 16-byte reads of 16 consecutive
// rows spread over the banks.
constexpr int kLdIn = kMaxIn + 4, kLdH = kMaxH + 4;

// acc[t] += A[16 rows][16 * KT] * B[16 t .. 16 t + 15][16 * KT]^T for NT
// column tiles: both operands have the summed index contiguous, at slot(k).
// Lane l holds row l % 16 of A and of each B tile; its group g = l / 16 reads
// slots 16 s + 4 g .. + 3 with one 16-byte read, and the j-th matrix
// instruction of a step sums the j-th of them over the four groups: k = 16 s
// + 4 j + g.  The matrix instruction adds its four products one after the
// other, each with one rounding, so every sum is the fmaf chain over
// k = 0, 1, .. that starts from acc, bit for bit: which units a ReLU cuts
// off, and every gradient, are what a loop over k gives.  The result has rows
// 4 g .. 4 g + 3 of column l % 16 in lane l.  The tile counts are those of
// the largest dimensions: with loops over the batch's own counts every step
// waited for its reads (a step of 4096 samples took 12 us more).
__host__ __device__ constexpr int slot(int k) {
  return (k & ~15) | ((k & 3) << 2) | ((k >> 2) & 3);
}
template <int NT, int KT>
__device__ __forceinline__ void mul_tiles(f4 (&acc)[NT], const float *a, int lda, const float *b,
                                          int ldb) {
  const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
#pragma unroll
  for (int s = 0; s < KT; ++s) {
    const f4 av = *reinterpret_cast<const f4 *>(a + r * lda + 16 * s + 4 * g);
    f4 bv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
      bv[t] = *reinterpret_cast<const f4 *>(b + (16 * t + r) * ldb + 16 * s + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv[t][j], acc[t], 0, 0, 0);
  }
}

// The same for one tile of B whose rows past the first `rows` are zero and
// not stored (a vector, or a few of them).
template <int KT>
__device__ __forceinline__ void mul_rows(f4 &acc, const float *a, int lda, const float *b, int ldb,
                                         int rows) {
  const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
#pragma unroll
  for (int s = 0; s < KT; ++s) {
    const f4 av = *reinterpret_cast<const f4 *>(a + r * lda + 16 * s + 4 * g);
    f4 bv = {};
    if (r < rows) bv = *reinterpret_cast<const f4 *>(b + r * ldb + 16 * s + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv[j], acc, 0, 0, 0);
  }
}

__device__ __forceinline__ float relu(float a) { return a > 0.f ? a : 0.f; }

// A workgroup has 8 waves, two to 16 samples: half 0 of a pair computes units
// 0 .. 31 of a layer, half 1 the others.
constexpr int kMlpT = 512;

// The weights and the workgroup's 64 samples into LDS, rows of
// kLdIn and kLdH floats, zeros around them.  A wave reads a row of weights,
// its lanes the columns; every load is issued before the first store.
// TRANSPOSED: W2 and the samples transposed as well.
template <bool TRANSPOSED>
__device__ __forceinline__ void load_tiles(float *W1, float *W2, float *X, const Dims &d,
                                           const float *p, const float *x, int s0, int n,
                                           float *W3, float *W2T, float *XT) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, c = l & 31;
  float a[8], b[8], v[4];
  const float w3 = l < d.h2 ? p[d.oW3() + l] : 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r = 8 * k + w;
    a[k] = (r < d.h1 && l < d.in) ? p[d.oW1() + r * d.in + l] : 0.f;
    b[k] = (r < d.h2 && l < d.h1) ? p[d.oW2() + r * d.h1 + l] : 0.f;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = 8 * w + 2 * k + (l >> 5);
    v[k] = (s0 + r < n && c < d.in) ? x[(size_t)(s0 + r) * d.in + c] : 0.f;
  }
  if (w == 0) W3[slot(l)] = w3;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r = 8 * k + w;
    if (l < kMaxIn) W1[r * kLdIn + slot(l)] = a[k];
    W2[r * kLdH + slot(l)] = b[k];
    if (TRANSPOSED) W2T[l * kLdH + slot(r)] = b[k];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = 8 * w + 2 * k + (l >> 5);
    X[r * kLdIn + slot(c)] = v[k];
    if (TRANSPOSED) XT[c * kLdH + slot(r)] = v[k];
  }
}

// Place of a wave: its 16 samples, its 32 units; of a lane: column c of its
// tiles, group g.
struct Place {
  int w, u, c, g;
};
__device__ __forceinline__ Place place() {
  const int l = threadIdx.x & 63;
  return Place{(int)(threadIdx.x >> 6) & 3, 32 * (int)(threadIdx.x >> 8), l & 15, l >> 4};
}

// The wave's tiles into rows of samples, and into columns of units: 4
// consecutive samples of a unit are strided by 4 slots.
__device__ __forceinline__ void store_rows(float *rows, const Place &q, const f4 (&v)[2]) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      rows[(16 * q.w + 4 * q.g + r) * kLdH + q.u + 16 * t + slot(q.c)] = v[t][r];
}
__device__ __forceinline__ void store_columns(float *cols, const Place &q, const f4 (&v)[2]) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      cols[(q.u + 16 * t + q.c) * kLdH + 16 * q.w + slot(4 * q.g + r)] = v[t][r];
}

// Activations of a hidden layer for the wave's 16 samples and 32 units from
// the samples' inputs a: a lane holds samples 4 g .. 4 g + 3 of units u + c
// and u + 16 + c.
template <int KT>
__device__ __forceinline__ void layer(f4 (&acc)[2], const Place &q, const float *bias, int units,
                                      const float *a, int lda, const float *W, int ldw) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int u = q.u + 16 * t + q.c;
    const float b = u < units ? bias[u] : 0.f;
    acc[t] = f4{b, b, b, b};
  }
  mul_tiles<2, KT>(acc, a + 16 * q.w * lda, lda, W + q.u * ldw, ldw);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[t][r] = relu(acc[t][r]);
}

__global__ __launch_bounds__(kMlpT) void mlp_forward_kernel(Dims d, const float *p,
                                                            const float *x, int n,
                                                            float *y) {
  __shared__ __align__(16) float W1[kMaxH * kLdIn], W2[kMaxH * kLdH], W3[kMaxH],
      X[kSamples * kLdIn], H1[kSamples * kLdH], H2[kSamples * kLdH];
  const int s0 = blockIdx.x * kSamples;
  load_tiles<false>(W1, W2, X, d, p, x, s0, n, W3, nullptr, nullptr);
  __syncthreads();
  const Place q = place();
  f4 h[2];
  layer<kMaxIn / 16>(h, q, p + d.ob1(), d.h1, X, kLdIn, W1, kLdIn);
  store_rows(H1, q, h);
  __syncthreads();
  layer<kMaxH / 16>(h, q, p + d.ob2(), d.h2, H1, kLdH, W2, kLdH);
  store_rows(H2, q, h);
  __syncthreads();
  if (q.u) return;
  const float b3 = p[d.ob3()];
  f4 out = {b3, b3, b3, b3};
  mul_rows<kMaxH / 16>(out, H2 + 16 * q.w * kLdH, kLdH, W3, 0, 1);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = s0 + 16 * q.w + 4 * q.g + r;
    if (q.c == 0 && s < n) y[s] = out[r];
  }
}

// LDS of the gradient kernel, in floats
constexpr int kW1 = 0, kW2 = kW1 + kMaxH * kLdIn, kW2T = kW2 + kMaxH * kLdH;
constexpr int kX = kW2T + kMaxH * kLdH, kXT = kX + kSamples * kLdIn;
constexpr int kRows = kXT + kMaxIn * kLdH;  // H1, H2, dL/d(pre-activation 2) in turn
constexpr int kH1T = kRows + kSamples * kLdH, kH2T = kH1T + kMaxH * kLdH;
constexpr int kD2T = kH2T + kMaxH * kLdH, kD1T = kD2T + kMaxH * kLdH;
constexpr int kW3 = kD1T + kMaxH * kLdH;
// ones, dL/dy and squared error of every sample
constexpr int kVec = kW3 + kMaxH, kGradLds = kVec + 3 * kLdH;
static_assert(kGradLds * 4 <= 160 * 1024, "LDS of a CU");

// one workgroup = kSamples samples: forward/backward of every sample, then
// the workgroup's gradient sums into ws[blockIdx.x][param]
__global__ __launch_bounds__(kMlpT) void mlp_grad_kernel(Dims d, const float *p,
                                                         const float *x,
                                                         const float *target, int n,
                                                         float *ws, float *wloss) {
  extern __shared__ __align__(16) float lds[];
  float *rows = lds + kRows, *vec = lds + kVec;
  const Place q = place();
  const int l = threadIdx.x & 63;
  const int s0 = blockIdx.x * kSamples;
  load_tiles<true>(lds + kW1, lds + kW2, lds + kX, d, p, x, s0, n, lds + kW3, lds + kW2T,
                   lds + kXT);
  f4 tg;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = s0 + 16 * q.w + 4 * q.g + r;
    tg[r] = s < n ? target[s] : 0.f;
  }
  float w3[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int u = q.u + 16 * t + q.c;
    w3[t] = u < d.h2 ? p[d.oW3() + u] : 0.f;
  }
  const float b3 = p[d.ob3()];
  __syncthreads();
  f4 h1[2], h2[2];
  layer<kMaxIn / 16>(h1, q, p + d.ob1(), d.h1, lds + kX, kLdIn, lds + kW1, kLdIn);
  store_rows(rows, q, h1);
  store_columns(lds + kH1T, q, h1);
  __syncthreads();
  layer<kMaxH / 16>(h2, q, p + d.ob2(), d.h2, rows, kLdH, lds + kW2, kLdH);
  store_columns(lds + kH2T, q, h2);
  __syncthreads();
  store_rows(rows, q, h2);
  __syncthreads();
  f4 y = {b3, b3, b3, b3}, dy;
  mul_rows<kMaxH / 16>(y, rows + 16 * q.w * kLdH, kLdH, lds + kW3, 0, 1);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = 16 * q.w + slot(4 * q.g + r);
    const bool in = s0 + 16 * q.w + 4 * q.g + r < n;
    const float e = __shfl(y[r], l & 48) - tg[r];
    dy[r] = in ? 2.f * e / (float)n : 0.f;
    if (q.c == 0 && q.u == 0) {
      vec[k] = 1.f;
      vec[kLdH + k] = dy[r];
      vec[2 * kLdH + k] = in ? e * e : 0.f;
    }
  }
  f4 d2[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) d2[t][r] = h2[t][r] > 0.f ? dy[r] * w3[t] : 0.f;
  store_columns(lds + kD2T, q, d2);
  __syncthreads();
  store_rows(rows, q, d2);
  __syncthreads();
  f4 d1[2] = {};
  mul_tiles<2, kMaxH / 16>(d1, rows + 16 * q.w * kLdH, kLdH, lds + kW2T + q.u * kLdH, kLdH);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) d1[t][r] = h1[t][r] > 0.f ? d1[t][r] : 0.f;
  store_columns(lds + kD1T, q, d1);
  __syncthreads();
  // a pair of waves sums units 16 w .. 16 w + 15 of every weight gradient over
  // the samples: half 0 columns 0 .. 31 of W2's and the bias gradients, which
  // are sums against ones (column 0), half 1 the rest of W2's, W1's and W3's,
  // against dL/dy (column 1).  Every product is under way before the first
  // store
  float *row = ws + (size_t)blockIdx.x * d.np;
  const float *D1 = lds + kD1T + 16 * q.w * kLdH, *D2 = lds + kD2T + 16 * q.w * kLdH;
  const int u0 = 16 * q.w + 4 * q.g;
  f4 gw2[2] = {};
  mul_tiles<2, kSamples / 16>(gw2, D2, kLdH, lds + kH1T + q.u * kLdH, kLdH);
  if (q.u == 0) {
    f4 b1 = {}, b2 = {}, v = {};
    mul_rows<kSamples / 16>(b1, D1, kLdH, vec, kLdH, 1);
    mul_rows<kSamples / 16>(b2, D2, kLdH, vec, kLdH, 1);
    // b3's gradient and the loss: the sums of vec's own rows 1 and 2 (rows 3
    // .. 15 of the left operand are not used: row 2 again)
    if (q.w == 0)
      mul_rows<kSamples / 16>(v, vec + (q.c < 3 ? 0 : 2 - q.c) * kLdH, kLdH, vec, kLdH, 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (q.c == 0 && u0 + r < d.h1) row[d.ob1() + u0 + r] = b1[r];
      if (q.c == 0 && u0 + r < d.h2) row[d.ob2() + u0 + r] = b2[r];
    }
    if (threadIdx.x == 0) {
      row[d.ob3()] = v[1];
      wloss[blockIdx.x] = v[2];
    }
  } else {
    f4 gw1[kMaxIn / 16] = {}, g3 = {};
    mul_tiles<kMaxIn / 16, kSamples / 16>(gw1, D1, kLdH, lds + kXT, kLdH);
    mul_rows<kSamples / 16>(g3, lds + kH2T + 16 * q.w * kLdH, kLdH, vec, kLdH, 2);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int u = u0 + r;
#pragma unroll
      for (int t = 0; t < kMaxIn / 16; ++t)
        if (u < d.h1 && 16 * t + q.c < d.in) row[d.oW1() + u * d.in + 16 * t + q.c] = gw1[t][r];
      if (q.c == 1 && u < d.h2) row[d.oW3() + u] = g3[r];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int u = u0 + r, k = q.u + 16 * t + q.c;
      if (u < d.h2 && k < d.h1) row[d.oW2() + u * d.h1 + k] = gw2[t][r];
    }
}

// Sums the workspace rows in order, a thread a parameter with 32 rows'
// loads in flight, and applies the SGD update; the last workgroup sums the
// losses.
__global__ __launch_bounds__(64) void mlp_update_kernel(Dims d, float *p, float *grads,
                                                        const float *ws,
                                                        const float *wloss, int nblk,
                                                        int n, float lr,
                                                        float *loss_out) {
  constexpr int kFlight = 32;
  const int q = blockIdx.x * 64 + threadIdx.x;
  if (q < d.np) {
    const float old = p[q];
    float g = 0.f;
    for (int b0 = 0; b0 < nblk; b0 += kFlight) {
      float v[kFlight];
#pragma unroll
      for (int k = 0; k < kFlight; ++k)
        v[k] = b0 + k < nblk ? ws[(size_t)(b0 + k) * d.np + q] : 0.f;
#pragma unroll
      for (int k = 0; k < kFlight; ++k)
        if (b0 + k < nblk) g += v[k];
    }
    grads[q] = g;
    p[q] = fmaf(-lr, g, old);
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0 && loss_out) {
    float s = 0.f;
    for (int b = 0; b < nblk; ++b) s += wloss[b];
    *loss_out = s / (float)n;
  }
}

int check_dims(int in, int h1, int h2) {
  if (in < 1 || in > kMaxIn || h1 < 1 || h1 > kMaxH || h2 < 1 || h2 > kMaxH)
    return set_error("MLP dimensions out of range (in<=32, hidden<=64)");
  return 0;
}

}  // namespace
}  // namespace jqd

using namespace jqd;

extern "C" size_t jq_mlp_num_params(int in, int h1, int h2) { return (size_t)dims(in, h1, h2).np; }

extern "C" size_t jq_mlp_workspace_floats(int in, int h1, int h2, int n) {
  Dims d = dims(in, h1, h2);
  size_t nblk = ((size_t)n + kSamples - 1) / kSamples;
  return nblk * (size_t)d.np + nblk;
}

extern "C" int jq_mlp_forward(const float *params, int in, int h1, int h2,
                              const float *x, int n, float *y, void *stream) {
  if (check_dims(in, h1, h2)) return -1;
  set_error("");
  if (n <= 0) return 0;
  Dims d = dims(in, h1, h2);
  hipLaunchKernelGGL(mlp_forward_kernel, dim3((n - 1) / kSamples + 1), dim3(kMlpT), 0,
                     (hipStream_t)stream, d, params, x, n, y);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_error(hipGetErrorString(e));
}

extern "C" int jq_mlp_train_step(float *params, float *grads, float *workspace,
                                 int in, int h1, int h2, const float *x,
                                 const float *target, int n, float lr,
                                 float *loss_out, void *stream) {
  if (check_dims(in, h1, h2)) return -1;
  set_error("");
  if (n <= 0) return 0;
  if (!workspace) return set_error("MLP train step: workspace missing");
  Dims d = dims(in, h1, h2);
  int nblk = (n - 1) / kSamples + 1;
  const size_t lds = sizeof(float) * kGradLds;
  static bool attr = false;
  if (!attr) {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(&mlp_grad_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
      return set_error("MLP LDS attribute failed");
    attr = true;
  }
  float *ws = workspace, *wloss = workspace + (size_t)nblk * d.np;
  hipLaunchKernelGGL(mlp_grad_kernel, dim3(nblk), dim3(kMlpT), lds, (hipStream_t)stream,
                     d, params, x, target, n, ws, wloss);
  hipLaunchKernelGGL(mlp_update_kernel, dim3((d.np + 63) / 64 + 1), dim3(64), 0,
                     (hipStream_t)stream, d, params, grads, ws, wloss, nblk, n, lr,
                     loss_out);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_error(hipGetErrorString(e));
}

namespace jqd {
namespace {

// Device address of `scratch` on each device, looked up once per device
// with that device current (the array's host-side name is not a device
// address).
constexpr int kMaxDevices = 64;
float *g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mu;

int scratch_for_current_device(float **out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_error("MLP train step (no-alloc): no usable current device");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error("MLP train step (no-alloc): hipGetSymbolAddress(scratch) failed");
    g_scratch_ptr[dev] = static_cast<float *>(p);
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

}  // namespace
}  // namespace jqd

extern "C" size_t jq_mlp_noalloc_max_samples(void) { return (size_t)kNoAllocMaxSamples; }

extern "C" int jq_mlp_train_step_noalloc(float *params, float *grads, int in, int h1,
                                         int h2, const float *x, const float *target,
                                         int n, float lr, float *loss_out,
                                         void *stream) {
  if (check_dims(in, h1, h2)) return -1;
  if (n > kNoAllocMaxSamples)
    return set_error("MLP train step (no-alloc): batch larger than 4096 samples");
  set_error("");
  if (n <= 0) return 0;
  float *ws = nullptr;
  if (scratch_for_current_device(&ws)) return -1;
  if (jq_mlp_workspace_floats(in, h1, h2, n) > kNoAllocFloats)
    return set_error("MLP train step (no-alloc): workspace exceeds the static buffer");
  return jq_mlp_train_step(params, grads, ws, in, h1, h2, x, target, n, lr, loss_out,
                           stream);
}
