// Device check of the RK5 kernels' fast arithmetic against the forms it
// stands for, over every float of its range: number of differing results.
#include <hip/hip_runtime.h>

#include "../../nest-gpu_amd/csrc/rk5_device.h"

namespace {

using namespace ngpu;

enum { kPowFast, kPowChain, kDivRecip, kDivEps, kExpNearCheck, kDivPairs };

__device__ bool same(float a, float b) {
  return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
}

__device__ bool subnormal(float q) {
  const unsigned int m = __float_as_uint(q) & 0x7fffffffu;
  return m != 0 && m < 0x800000u;
}

__device__ unsigned int mix(unsigned int h) {
  h = (h ^ (h >> 16)) * 0x7feb352du;
  h = (h ^ (h >> 15)) * 0x846ca68bu;
  return h ^ (h >> 16);
}

__device__ bool div_differs(float x, float d) {
  unsigned int tiny = ~0u;
  const float q = div_recip(x, recip_double(d), tiny);
  // a quotient that is noted is divided again
  return !tiny_noted(tiny) && !same(q, x / d);
}

__device__ bool differs(int what, unsigned int u, float d) {
  const float x = __uint_as_float(u);
  switch (what) {
    case kPowFast:
      return x >= kPowLo && x <= kPowHi &&
             !(same(pow_step_fast(x, true), pow_m02(x)) && same(pow_step_fast(x, false), pow_m025(x)));
    case kPowChain: {
      const float r = div_eps(x);
      return r >= kPowLo && r <= kPowHi &&
             !(same(pow_step_chain(x, r, true), pow_m02(r)) &&
               same(pow_step_chain(x, r, false), pow_m025(r)));
    }
    case kDivRecip:
      return div_differs(x, d);
    case kDivEps: {
      const float q = x / ck::eps;
      return x >= 0.0f && !subnormal(q) && !same(div_eps(x), q);
    }
    case kExpNearCheck:
      return fabsf(x) <= kExpNear && !same(exp_fma_near(x), exp_fma(x));
    case kDivPairs: {
      const float y = __uint_as_float(mix(u)), e = __uint_as_float(mix(u ^ 0x9e3779b9u));
      return __builtin_isnormal(e) && div_differs(y, e);
    }
    default:
      return true;
  }
}

__global__ void __launch_bounds__(256)
check_kernel(int what, float d, unsigned long long lo, unsigned long long hi, unsigned long long* bad) {
  unsigned long long n = 0;
  const unsigned long long step = (unsigned long long)gridDim.x * blockDim.x;
  for (unsigned long long u = lo + (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; u < hi;
       u += step)
    n += differs(what, (unsigned int)u, d);
  if (n) atomicAdd(bad, n);
}

}  // namespace

// differing results for the float patterns [lo, hi), hi at most 2^32; -1 on
// a HIP error
extern "C" long long arith_check(int what, float d, unsigned long long lo, unsigned long long hi) {
  if (hi > (1ull << 32) || lo > hi) return -1;
  unsigned long long *bad = nullptr, n = 0;
  if (hipMalloc((void**)&bad, sizeof(n)) != hipSuccess) return -1;
  bool ok = hipMemcpy(bad, &n, sizeof(n), hipMemcpyHostToDevice) == hipSuccess;
  if (ok) {
    hipLaunchKernelGGL(check_kernel, dim3(4096), dim3(256), 0, nullptr, what, d, lo, hi, bad);
    ok = hipGetLastError() == hipSuccess &&
         hipMemcpy(&n, bad, sizeof(n), hipMemcpyDeviceToHost) == hipSuccess;
  }
  return hipFree(bad) == hipSuccess && ok ? (long long)n : -1;
}
