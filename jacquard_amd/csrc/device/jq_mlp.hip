// FP32 MLP (in -> h1 -> h2 -> 1, ReLU) for the learned partition cost model:
// forward, mean-squared-error backward and SGD, hand-written for gfx950.
//
// Parameters are packed W1[h1][in], b1[h1], W2[h2][h1], b2[h2], W3[h2], b3.
// Training is deterministic: each workgroup writes the gradient of its 64
// samples to its own workspace row, a second kernel sums the rows in a
// fixed order and applies the update.
//
// Every matrix product runs on the matrix cores in FP32
// (v_mfma_f32_16x16x4_f32: FP32 inputs, FP32 accumulation).  A wave owns 16
// samples from their inputs to their pre-activation gradients, so the forward
// and backward chain needs no workgroup barrier; then a wave owns 16 rows of
// each weight gradient.  Dimensions are padded with zeros to multiples of 16
// in LDS.  A thread per sample (its activations in scratch, weights read one
// by one) kept one wave of a workgroup busy: a step of 4096 samples took
// 340 us and takes 27, a forward of 5013 samples 140 and 11.  Error against
// 64 bits over the step's gradients: 1.3e-7 before, 4.5e-8 now.
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

__host__ __device__ inline int tiles(int n) { return (n + 15) / 16; }

// acc[t] += A[16 rows][16 * kt] * B[16 t .. 16 t + 15][16 * kt]^T for the
// first nt column tiles: both operands have the summed index contiguous.
// Lane l holds row l % 16 of A and of each B tile; its group g = l / 16 reads
// elements 16 s + 4 g .. + 3 with one 16-byte read, and the j-th matrix
// instruction of a step sums the j-th elements of the four groups.  The
// result has rows 4 g .. 4 g + 3 of column l % 16 in lane l.
__device__ __forceinline__ void mul_tiles(f4 (&acc)[4], const float *a, int lda, const float *b,
                                          int ldb, int nt, int kt) {
  const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
  for (int s = 0; s < kt; ++s) {
    const f4 av = *reinterpret_cast<const f4 *>(a + r * lda + 16 * s + 4 * g);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (t < nt) {
        const f4 bv = *reinterpret_cast<const f4 *>(b + (16 * t + r) * ldb + 16 * s + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], bv[j], acc[t], 0, 0, 0);
      }
    }
  }
}

__device__ __forceinline__ float relu(float a) { return a > 0.f ? a : 0.f; }

// Sum over the 16 lanes of a row of the wave, on every one of them; over
// the wave's four rows, lane by lane.
__device__ __forceinline__ float sum16(float v) {
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) v += __shfl_xor(v, m);
  return v;
}
__device__ __forceinline__ float sum_groups(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// Rows 0 .. rows - 1 of the packed matrix m[rows][cols] into dst[64][ld],
// zeros around it up to 64 x width; a wave reads a row, its lanes the columns.
template <int WIDTH>
__device__ __forceinline__ void load_matrix(float *dst, int ld, const float *m, int rows,
                                            int cols) {
  const int w = threadIdx.x >> 6, c = threadIdx.x & 63;
#pragma unroll 8
  for (int k = 0; k < 16; ++k) {
    const int r = 4 * k + w;
    if (c < WIDTH) dst[r * ld + c] = (r < rows && c < cols) ? m[r * cols + c] : 0.f;
  }
}

// The workgroup's 64 samples into X[64][kLdIn], zeros around them; every
// wave loads its own 16.
__device__ __forceinline__ void load_samples(float *X, const float *x, int s0, int n, int in) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, c = l & 31;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r = 16 * w + 2 * k + (l >> 5);
    X[r * kLdIn + c] = (s0 + r < n && c < in) ? x[(size_t)(s0 + r) * in + c] : 0.f;
  }
}

// First layer of the wave's 16 samples: activations in acc (lane l: samples
// 4 g .. 4 g + 3 of unit 16 t + l % 16) and in H1[64][kLdH].
__device__ __forceinline__ void layer1(f4 (&acc)[4], const Dims &d, const float *p,
                                       const float *X, const float *W1, float *H1) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, c = l & 15, g = l >> 4;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int k = 16 * t + c;
    const float b = k < d.h1 ? p[d.ob1() + k] : 0.f;
    acc[t] = f4{b, b, b, b};
  }
  mul_tiles(acc, X + 16 * w * kLdIn, kLdIn, W1, kLdIn, tiles(d.h1), tiles(d.in));
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      acc[t][r] = relu(acc[t][r]);
      H1[(16 * w + 4 * g + r) * kLdH + 16 * t + c] = acc[t][r];
    }
  __builtin_amdgcn_wave_barrier();  // the wave reads only its own rows
}

// Second layer of the wave's 16 samples, laid out as layer1's.
__device__ __forceinline__ void layer2(f4 (&acc)[4], const Dims &d, const float *p,
                                       const float *H1, const float *W2) {
  const int w = threadIdx.x >> 6, c = threadIdx.x & 15;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int j = 16 * t + c;
    const float b = j < d.h2 ? p[d.ob2() + j] : 0.f;
    acc[t] = f4{b, b, b, b};
  }
  mul_tiles(acc, H1 + 16 * w * kLdH, kLdH, W2, kLdH, tiles(d.h2), tiles(d.h1));
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[t][r] = relu(acc[t][r]);
}

// Output of samples 4 g .. 4 g + 3, on every lane of group g.
__device__ __forceinline__ f4 layer3(const Dims &d, const float *p, const f4 (&h2)[4],
                                     const float (&w3)[4]) {
  const float b3 = p[d.ob3()];
  f4 y;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float a = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) a = fmaf(w3[t], h2[t][r], a);
    y[r] = b3 + sum16(a);
  }
  return y;
}

__device__ __forceinline__ void load_w3(float (&w3)[4], const Dims &d, const float *p) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int j = 16 * t + (threadIdx.x & 15);
    w3[t] = j < d.h2 ? p[d.oW3() + j] : 0.f;
  }
}

__global__ __launch_bounds__(256) void mlp_forward_kernel(Dims d, const float *p,
                                                          const float *x, int n,
                                                          float *y) {
  __shared__ __align__(16) float W1[kMaxH * kLdIn], W2[kMaxH * kLdH], X[kSamples * kLdIn],
      H1[kSamples * kLdH];
  const int s0 = blockIdx.x * kSamples;
  load_samples(X, x, s0, n, d.in);
  load_matrix<kMaxIn>(W1, kLdIn, p + d.oW1(), d.h1, d.in);
  load_matrix<kMaxH>(W2, kLdH, p + d.oW2(), d.h2, d.h1);
  float w3[4];
  load_w3(w3, d, p);
  __syncthreads();
  f4 h[4];
  layer1(h, d, p, X, W1, H1);
  layer2(h, d, p, H1, W2);
  const f4 out = layer3(d, p, h, w3);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = s0 + 16 * w + 4 * g + r;
    if ((l & 15) == r && s < n) y[s] = out[r];
  }
}

// LDS of the gradient kernel, in floats
constexpr int kW1 = 0, kW2 = kW1 + kMaxH * kLdIn, kW2T = kW2 + kMaxH * kLdH;
constexpr int kX = kW2T + kMaxH * kLdH, kXT = kX + kSamples * kLdIn;
constexpr int kHD = kXT + kMaxIn * kLdH;    // H1, then dL/d(pre-activation 2)
constexpr int kH1T = kHD + kSamples * kLdH, kD2T = kH1T + kMaxH * kLdH;
constexpr int kD1T = kD2T + kMaxH * kLdH;
constexpr int kSums = kD1T + kMaxH * kLdH;  // per wave: b1, b2, W3 (64 each), b3, loss
constexpr int kSumW = 3 * kMaxH + 2;
constexpr int kGradLds = kSums + 4 * kSumW;

// one workgroup = kSamples samples: forward/backward of every sample, then
// the workgroup's gradient sums into ws[blockIdx.x][param]
__global__ __launch_bounds__(256) void mlp_grad_kernel(Dims d, const float *p,
                                                       const float *x,
                                                       const float *target, int n,
                                                       float *ws, float *wloss) {
  extern __shared__ __align__(16) float lds[];
  float *X = lds + kX, *XT = lds + kXT, *HD = lds + kHD, *H1T = lds + kH1T;
  float *D1T = lds + kD1T, *D2T = lds + kD2T;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const int s0 = blockIdx.x * kSamples;
  load_samples(X, x, s0, n, d.in);
  load_matrix<kMaxIn>(lds + kW1, kLdIn, p + d.oW1(), d.h1, d.in);
  load_matrix<kMaxH>(lds + kW2, kLdH, p + d.oW2(), d.h2, d.h1);
  float w3[4];
  load_w3(w3, d, p);
  f4 tg;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int s = s0 + 16 * w + 4 * g + r;
    tg[r] = s < n ? target[s] : 0.f;
  }
  __syncthreads();
  // transposes for the products that sum over units or samples
  {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int r = 16 * w + k;
      lds[kW2T + l * kLdH + r] = lds[kW2 + r * kLdH + l];
      if (l < kMaxIn) XT[l * kLdH + r] = X[r * kLdIn + l];
    }
  }
  f4 h1[4], h2[4];
  layer1(h1, d, p, X, lds + kW1, HD);
#pragma unroll
  for (int t = 0; t < 4; ++t)
    *reinterpret_cast<f4 *>(H1T + (16 * t + c) * kLdH + 16 * w + 4 * g) = h1[t];
  layer2(h2, d, p, HD, lds + kW2);
  const f4 y = layer3(d, p, h2, w3);
  f4 dy;
  float e2 = 0.f, gb3 = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bool in = s0 + 16 * w + 4 * g + r < n;
    const float e = y[r] - tg[r];
    dy[r] = in ? 2.f * e / (float)n : 0.f;
    e2 += in ? e * e : 0.f;
    gb3 += dy[r];
  }
  float *sums = lds + kSums + w * kSumW;
  // dL/d(pre-activation 2), and the sums over samples that it gives
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f4 d2;
    float gw3 = 0.f, gb2 = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      d2[r] = h2[t][r] > 0.f ? dy[r] * w3[t] : 0.f;
      gw3 = fmaf(dy[r], h2[t][r], gw3);
      gb2 += d2[r];
      HD[(16 * w + 4 * g + r) * kLdH + 16 * t + c] = d2[r];
    }
    *reinterpret_cast<f4 *>(D2T + (16 * t + c) * kLdH + 16 * w + 4 * g) = d2;
    gw3 = sum_groups(gw3);
    gb2 = sum_groups(gb2);
    if (g == 0) {
      sums[kMaxH + 16 * t + c] = gb2;
      sums[2 * kMaxH + 16 * t + c] = gw3;
    }
  }
  e2 = sum_groups(e2);
  gb3 = sum_groups(gb3);
  if (l == 0) {
    sums[3 * kMaxH] = gb3;
    sums[3 * kMaxH + 1] = e2;
  }
  __syncthreads();  // W2T; the wave's own rows of HD need none
  {
    f4 d1[4] = {};
    mul_tiles(d1, HD + 16 * w * kLdH, kLdH, lds + kW2T, kLdH, tiles(d.h1), tiles(d.h2));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float gb1 = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d1[t][r] = h1[t][r] > 0.f ? d1[t][r] : 0.f;
        gb1 += d1[t][r];
      }
      *reinterpret_cast<f4 *>(D1T + (16 * t + c) * kLdH + 16 * w + 4 * g) = d1[t];
      gb1 = sum_groups(gb1);
      if (g == 0) sums[16 * t + c] = gb1;
    }
  }
  __syncthreads();
  float *row = ws + (size_t)blockIdx.x * d.np;
  // rows 16 w .. 16 w + 15 of both weight gradients, summed over the samples
  {
    f4 a[4] = {};
    mul_tiles(a, D2T + 16 * w * kLdH, kLdH, H1T, kLdH, tiles(d.h1), kSamples / 16);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 16 * w + 4 * g + r, k = 16 * t + c;
        if (j < d.h2 && k < d.h1) row[d.oW2() + j * d.h1 + k] = a[t][r];
      }
  }
  {
    f4 a[4] = {};
    mul_tiles(a, D1T + 16 * w * kLdH, kLdH, XT, kLdH, tiles(d.in), kSamples / 16);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * w + 4 * g + r, i = 16 * t + c;
        if (k < d.h1 && i < d.in) row[d.oW1() + k * d.in + i] = a[t][r];
      }
  }
  const int t = threadIdx.x;
  if (t < kSumW) {
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) v += lds[kSums + q * kSumW + t];
    const int u = t & (kMaxH - 1);
    if (t == kSumW - 1)
      wloss[blockIdx.x] = v;
    else if (t == kSumW - 2)
      row[d.ob3()] = v;
    else if (t < kMaxH && u < d.h1)
      row[d.ob1() + u] = v;
    else if (t >= 2 * kMaxH && u < d.h2)
      row[d.oW3() + u] = v;
    else if (t >= kMaxH && t < 2 * kMaxH && u < d.h2)
      row[d.ob2() + u] = v;
  }
}

// Sums the workspace rows, 64 parameters a workgroup: wave q takes rows q,
// q + 4, .. and the four sums are added in order; then the SGD update.
// Workgroup 0's wave 0 sums the losses.  One thread a parameter walked the
// 64 rows of a 4096-sample step one load after another.
__global__ __launch_bounds__(256) void mlp_update_kernel(Dims d, float *p, float *grads,
                                                         const float *ws,
                                                         const float *wloss, int nblk,
                                                         int n, float lr,
                                                         float *loss_out) {
  __shared__ float part[4][64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int q = blockIdx.x * 64 + l;
  float g = 0.f;
  if (q < d.np) {
#pragma unroll 8
    for (int b = w; b < nblk; b += 4) g += ws[(size_t)b * d.np + q];
  }
  part[w][l] = g;
  __syncthreads();
  if (w == 0 && q < d.np) {
    g = ((part[0][l] + part[1][l]) + part[2][l]) + part[3][l];
    grads[q] = g;
    p[q] -= lr * g;
  }
  if (blockIdx.x == 0 && w == 0 && loss_out) {
    float s = 0.f;
    for (int b = l; b < nblk; b += 64) s += wloss[b];
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m);
    if (l == 0) *loss_out = s / (float)n;
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
  hipLaunchKernelGGL(mlp_forward_kernel, dim3((n - 1) / kSamples + 1), dim3(256), 0,
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
  hipLaunchKernelGGL(mlp_grad_kernel, dim3(nblk), dim3(256), lds, (hipStream_t)stream,
                     d, params, x, target, n, ws, wloss);
  hipLaunchKernelGGL(mlp_update_kernel, dim3((d.np + 63) / 64), dim3(256), 0,
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
