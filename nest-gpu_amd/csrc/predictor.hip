// Training and test kernels of the learned step-size predictor (predictor.h).
//
// Training minimises the mean censored squared error of log2(h/dt) over
// (state, accepted h) records logged by the plain RK5 kernel.  The forward
// pass evaluates what inference computes (bfloat16 inputs, W1, W2 and
// layer-1 activations, FP32 accumulation); gradients pass straight through
// the rounding to the FP32 master weights, which Adam updates.  Gradient
// sums are deterministic: every block stages the per-sample vectors of 64
// samples in LDS and thread L accumulates parameters L, L+512, ... over the
// samples in a fixed order, blocks write rows of partial sums, and the
// update kernel adds the rows in block order.
#include <hip/hip_runtime.h>

#include <mutex>
#include <stdexcept>
#include <string>

#include "philox.h"
#include "predictor_device.h"
#include "predictor_kernels.h"

namespace ngpu {

// ---- normalisation: per-block sums of x and x^2 of the 8 raw inputs --------
__global__ void __launch_bounds__(256) pred_stats_kernel(const float* log, long long n,
                                                         double* part) {
  __shared__ double red[256];
  double s[kPI], q[kPI];
#pragma unroll
  for (int k = 0; k < kPI; ++k) s[k] = q[k] = 0.0;
  for (long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x; r < n;
       r += (long long)gridDim.x * blockDim.x) {
#pragma unroll
    for (int k = 0; k < kPI; ++k) {
      const double v = log[r * kLogCols + k];
      s[k] += v;
      q[k] += v * v;
    }
  }
  for (int k = 0; k < 2 * kPI; ++k) {
    red[threadIdx.x] = k < kPI ? s[k] : q[k - kPI];
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)blockIdx.x * 2 * kPI + k] = red[0];
    __syncthreads();
  }
}

void launch_pred_stats(const float* log, long long n, double* part, int grid, hipStream_t s) {
  hipLaunchKernelGGL(pred_stats_kernel, dim3(grid), dim3(256), 0, s, log, n, part);
}

// ---- forward + backward: 64 samples per block and round ----------------------
// Eight waves share a round's samples (lane = sample): wave w computes hidden
// units 4w .. 4w+3 of both layers and of the backward pass, the activations
// going through LDS as rows [unit][sample] (written without bank conflicts,
// read back in 16-byte pieces of 4 samples), then every thread accumulates
// up to kOwn parameters.  Every sum keeps one fixed order (units, then
// samples, then rounds), whatever the number of waves.
// Bound: the dependent LDS reads and additions of a round, not the matrix
// work (0.06 GFLOP a batch): on matrix cores the sums would change.  Batch
// 8192 (128 blocks): 85 us with one wave per block, whose row-major LDS
// writes hit one bank with all 64 lanes and which summed 22 parameters per
// lane; 14 us this way.
constexpr int kGradWaves = 8, kGradThreads = 64 * kGradWaves;
constexpr int kGradUnits = kPH / kGradWaves;   // units per wave
constexpr int kRow = 68;   // floats per [unit][sample] row: 16-byte pieces of consecutive rows in other banks

struct GradLDS {
  float w1q[kPH * kPI], w2q[kPH * kPH], b1[kPH], b2[kPH], w3[kPH], mu[kPI], is[kPI];
  float b3;
  alignas(16) float xq[kPI][kRow];
  alignas(16) float h1q[kPH][kRow], dz1[kPH][kRow], dz2[kPH][kRow], h2[kPH][kRow];
  alignas(16) float dout[kRow], one[kRow];
};

__global__ void __launch_bounds__(kGradThreads) pred_grad_kernel(PredGradArgs a) {
  __shared__ GradLDS L;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
  const int u0 = wv * kGradUnits;
  const float* P = a.params;
  for (int k = tid; k < kPH * kPH; k += kGradThreads) {
    L.w2q[k] = bf16_round(P[kPOffW2 + k]);
    if (k < kPH * kPI) L.w1q[k] = bf16_round(P[kPOffW1 + k]);
    if (k < kPH) {
      L.b1[k] = P[kPOffB1 + k];
      L.b2[k] = P[kPOffB2 + k];
      L.w3[k] = P[kPOffW3 + k];
    }
    if (k < kPI) {
      L.mu[k] = P[kPOffMu + k];
      L.is[k] = P[kPOffIs + k];
    }
    if (k < 64) L.one[k] = 1.0f;
  }
  if (tid == 0) L.b3 = P[kPOffB3];
  __syncthreads();

  // parameter p of the thread: gradient sum over samples of rowA[s] * rowB[s]
  // (times one for the biases, exact)
  constexpr int kOwn = (kPNTrain + kGradThreads - 1) / kGradThreads;
  const float *ra[kOwn], *rb[kOwn];
  float acc[kOwn];
#pragma unroll
  for (int k = 0; k < kOwn; ++k) {
    const int p = tid + kGradThreads * k;
    acc[k] = 0.0f;
    ra[k] = L.dout;
    rb[k] = L.one;   // b3, and threads past the last parameter
    if (p < kPH * kPI) {
      ra[k] = L.dz1[p / kPI];
      rb[k] = L.xq[p % kPI];
    } else if (p < kPH * kPI + kPH) {
      ra[k] = L.dz1[p - kPH * kPI];
    } else if (p < kPH * kPI + kPH + kPH * kPH) {
      const int q = p - kPH * kPI - kPH;
      ra[k] = L.dz2[q / kPH];
      rb[k] = L.h1q[q % kPH];
    } else if (p < kPH * kPI + 2 * kPH + kPH * kPH) {
      ra[k] = L.dz2[p - kPH * kPI - kPH - kPH * kPH];
    } else if (p < kPNTrain - 1) {
      rb[k] = L.h2[p - (kPH * kPI + 2 * kPH + kPH * kPH)];
    }
  }
  float loss = 0.0f;
  const float inv_b = 1.0f / (float)a.batch;

  for (int rd = 0; rd < a.rounds; ++rd) {
    const long long slot = ((long long)blockIdx.x * a.rounds + rd) * 64 + lane;
    long long src = -1;
    if (a.raw) {
      src = slot < a.n_log ? slot : -1;
    } else if (a.idx) {
      src = slot < a.n_idx ? a.idx[slot] : -1;
    } else {
      const U32x4 ctr = {(uint32_t)slot, (uint32_t)(slot >> 32), (uint32_t)a.step,
                         (uint32_t)(a.step >> 32)};
      const U32x4 o = philox4x32_10(ctr, (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
      const unsigned long long r64 = ((unsigned long long)o.x << 32) | o.y;
      src = (long long)(r64 % (unsigned long long)a.n_log);
    }
    // (every wave reads the samples: the same lines, without a barrier more)
    float x[kPI], z1[kGradUnits], z2[kGradUnits], dout = 0.0f;
    float t = 0.0f;
    bool cens = false;
    if (src >= 0 && a.raw) {
      const float* rec = a.raw + src * kPI;
#pragma unroll
      for (int i = 0; i < kPI; ++i) x[i] = bf16_round((rec[i] - L.mu[i]) * L.is[i]);
      t = a.target[src];
      cens = a.cens[src] != 0;
    } else if (src >= 0) {
      const float* rec = a.log + src * kLogCols;
#pragma unroll
      for (int i = 0; i < kPI; ++i) x[i] = bf16_round((rec[i] - L.mu[i]) * L.is[i]);
      t = rec[kPI];
      cens = rec[kPI + 1] != 0.0f;
    } else {
#pragma unroll
      for (int i = 0; i < kPI; ++i) x[i] = 0.0f;
    }
    if (wv == 0) {
#pragma unroll
      for (int i = 0; i < kPI; ++i) L.xq[i][lane] = x[i];
    }
#pragma unroll
    for (int u = 0; u < kGradUnits; ++u) {
      const int o = u0 + u;
      float s = L.b1[o];
#pragma unroll
      for (int i = 0; i < kPI; ++i) s += L.w1q[o * kPI + i] * x[i];
      z1[u] = s;
      L.h1q[o][lane] = bf16_round(s > 0.0f ? s : 0.0f);
    }
    __syncthreads();
    {
#pragma unroll
      for (int u = 0; u < kGradUnits; ++u) z2[u] = L.b2[u0 + u];
#pragma unroll 8
      for (int i = 0; i < kPH; ++i) {
        const float h = L.h1q[i][lane];
#pragma unroll
        for (int u = 0; u < kGradUnits; ++u) z2[u] += L.w2q[(u0 + u) * kPH + i] * h;
      }
#pragma unroll
      for (int u = 0; u < kGradUnits; ++u) L.h2[u0 + u][lane] = z2[u] > 0.0f ? z2[u] : 0.0f;
    }
    __syncthreads();
    float out = L.b3;
#pragma unroll 8
    for (int o = 0; o < kPH; ++o) out += L.w3[o] * L.h2[o][lane];
    if (src >= 0) {
      const float e = out - t;
      if (!(cens && e > 0.0f)) {
        loss += e * e;
        dout = 2.0f * e * inv_b;
      }
    }
#pragma unroll
    for (int u = 0; u < kGradUnits; ++u)
      L.dz2[u0 + u][lane] = z2[u] > 0.0f ? dout * L.w3[u0 + u] : 0.0f;
    if (wv == 0) L.dout[lane] = dout;
    __syncthreads();
    {
      float s[kGradUnits];
#pragma unroll
      for (int u = 0; u < kGradUnits; ++u) s[u] = 0.0f;
#pragma unroll 8
      for (int o = 0; o < kPH; ++o) {
        const float g = L.dz2[o][lane];
#pragma unroll
        for (int u = 0; u < kGradUnits; ++u) s[u] += g * L.w2q[o * kPH + u0 + u];
      }
#pragma unroll
      for (int u = 0; u < kGradUnits; ++u) L.dz1[u0 + u][lane] = z1[u] > 0.0f ? s[u] : 0.0f;
    }
    __syncthreads();
    float sum[kOwn];
#pragma unroll
    for (int k = 0; k < kOwn; ++k) sum[k] = 0.0f;
#pragma unroll 4
    for (int s = 0; s < 64; s += 4) {
#pragma unroll
      for (int k = 0; k < kOwn; ++k) {
        const float4 p = *reinterpret_cast<const float4*>(ra[k] + s);
        const float4 q = *reinterpret_cast<const float4*>(rb[k] + s);
        sum[k] += p.x * q.x;
        sum[k] += p.y * q.y;
        sum[k] += p.z * q.z;
        sum[k] += p.w * q.w;
      }
    }
#pragma unroll
    for (int k = 0; k < kOwn; ++k) acc[k] += sum[k];
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kOwn; ++k) {
    const int p = tid + kGradThreads * k;
    if (p < kPNTrain) a.gpart[(size_t)blockIdx.x * kPNTrain + p] = acc[k];
  }
  if (wv == 0) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) a.lpart[blockIdx.x] = loss;
  }
}

void launch_pred_grad(const PredGradArgs& a, int blocks, hipStream_t s) {
  hipLaunchKernelGGL(pred_grad_kernel, dim3(blocks), dim3(kGradThreads), 0, s, a);
}

// ---- sum of the block rows, then Adam (or only the sum) ---------------------
// A block takes 32 parameters: its threads read kUpdRows rows of them into
// LDS at once, then one thread per parameter adds them in row order (the
// loss sums as a further column of the last block).  Bound: the latency of
// the row reads; one thread per parameter reading 128 rows one after the
// other took 37 us, this 5 us.
constexpr int kUpdCols = 32, kUpdRows = 128, kUpdThreads = 512;

__global__ void __launch_bounds__(kUpdThreads) pred_update_kernel(PredUpdateArgs a) {
  __shared__ float tile[kUpdRows][kUpdCols + 1];
  const int col = threadIdx.x % kUpdCols, row0 = threadIdx.x / kUpdCols;
  const int p = blockIdx.x * kUpdCols + col;   // p == kPNTrain: the loss
  float g = 0.0f;
  for (int b0 = 0; b0 < a.blocks; b0 += kUpdRows) {
    const int nb = a.blocks - b0 < kUpdRows ? a.blocks - b0 : kUpdRows;
    if (p <= kPNTrain) {
#pragma unroll
      for (int r = row0; r < kUpdRows; r += kUpdThreads / kUpdCols)
        if (r < nb)
          tile[r][col] = p < kPNTrain ? a.gpart[(size_t)(b0 + r) * kPNTrain + p] : a.lpart[b0 + r];
    }
    __syncthreads();
    if (row0 == 0 && p <= kPNTrain) {
#pragma unroll 16
      for (int r = 0; r < nb; ++r) g += tile[r][col];
    }
    __syncthreads();
  }
  if (row0 != 0) return;
  if (p < kPNTrain) {
    if (a.grad_out) a.grad_out[p] = g;
    if (a.lr > 0.0f) {
      const float m = a.beta1 * a.m[p] + (1.0f - a.beta1) * g;
      const float v = a.beta2 * a.v[p] + (1.0f - a.beta2) * g * g;
      a.m[p] = m;
      a.v[p] = v;
      const float mh = m / a.bc1, vh = v / a.bc2;
      a.params[kPOffW1 + p] -= a.lr * mh / (sqrtf(vh) + a.eps);
    }
  } else if (p == kPNTrain) {
    a.loss_out[0] = g / (float)a.batch;
  }
}

void launch_pred_update(const PredUpdateArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(pred_update_kernel, dim3((kPNTrain + 1 + kUpdCols - 1) / kUpdCols),
                     dim3(kUpdThreads), 0, s, a);
}

// ---- inference through the matrix-core path (the one the RK5 kernel uses) ---
__global__ void __launch_bounds__(256) pred_infer_kernel(const float* P, const float* raw,
                                                         long long n, float* out) {
  __shared__ PredLDS s;
  pred_stage(s, P);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const long long wave = (long long)blockIdx.x * (blockDim.x / 64) + (threadIdx.x / 64);
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long base = wave * 64; base < n; base += stride) {   // uniform per wave
    const long long r = base + lane;
    float in[kPI];
#pragma unroll
    for (int k = 0; k < kPI; ++k) in[k] = r < n ? raw[r * kPI + k] : 0.0f;
    const float o = pred_infer_wave(s, in);
    if (r < n) out[r] = o;
  }
}

void launch_pred_infer(const float* P, const float* raw, long long n, float* out, hipStream_t s) {
  long long waves = (n + 63) / 64;
  int grid = (int)((waves + 3) / 4);
  if (grid > 1024) grid = 1024;
  if (grid < 1) grid = 1;
  hipLaunchKernelGGL(pred_infer_kernel, dim3(grid), dim3(256), 0, s, P, raw, n, out);
}

// ---- loss and gradient without allocation ------------------------------------
// The partial gradient rows and loss sums of pred_grad_kernel live in this
// fixed array (1.4 MB per GPU, held until the process ends): rows
// [kPredScratchMaxBlocks][kPNTrain], then kPredScratchMaxBlocks loss sums.
// Every block writes its whole row and loss sum and the update kernel reads
// only the rows of the current call, so nothing needs clearing between calls.
constexpr size_t kPredScratchFloats =
    (size_t)kPredScratchMaxBlocks * kPNTrain + kPredScratchMaxBlocks;
static __device__ __align__(256) float scratch[kPredScratchFloats];

// Device address of `scratch` on the current device, looked up once per
// device (each GPU holds its own copy of the array at its own address; the
// symbol's name in host code is not that address).
static float* scratch_ptr() {
  constexpr int kMaxDev = 64;
  static float* ptr[kMaxDev] = {};
  static std::mutex mu;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) throw std::runtime_error(std::string("hipGetDevice: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDev) throw std::runtime_error("device index out of range for the predictor scratch");
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      throw std::runtime_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    ptr[dev] = static_cast<float*>(p);
  }
  return ptr[dev];
}

void pred_loss_grad_noalloc(const float* params, const float* raw, const float* target,
                            const unsigned char* cens, int n, float* loss, float* grad,
                            hipStream_t s) {
  if (n < 1 || n > kPredScratchMaxN)
    throw std::runtime_error("predictor loss/gradient without allocation: batch of " +
                             std::to_string(n) + " records outside [1, " +
                             std::to_string(kPredScratchMaxN) + "]");
  float* base = scratch_ptr();
  const int blocks = (n + 63) / 64;
  PredGradArgs ga{};
  ga.params = params;
  ga.n_log = n;
  ga.raw = raw;
  ga.target = target;
  ga.cens = cens;
  ga.rounds = 1;
  ga.batch = n;
  ga.gpart = base;
  ga.lpart = base + (size_t)kPredScratchMaxBlocks * kPNTrain;
  launch_pred_grad(ga, blocks, s);
  PredUpdateArgs ua{};
  ua.params = const_cast<float*>(params);   // lr = 0: read only
  ua.gpart = ga.gpart;
  ua.lpart = ga.lpart;
  ua.blocks = blocks;
  ua.batch = n;
  ua.lr = 0.0f;
  ua.grad_out = grad;
  ua.loss_out = loss;
  launch_pred_update(ua, s);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    throw std::runtime_error(std::string("predictor loss/gradient launch: ") + hipGetErrorString(e));
}

}  // namespace ngpu
