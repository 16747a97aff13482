// The adaptive RK5 update of src/rk5.h:69-207 as HIP kernel templates over
// a neuron model (rk5_models.h): the Cash-Karp attempt, the lane-per-neuron
// kernel, the persistent lane-refill kernel with hot-first scheduling and
// split steps, and the launch helpers.  Each model family instantiates them
// in a file of its own (rk5_*.hip), so the families compile in parallel.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "common.h"
#include "device_common.h"
#include "kernels.h"
#include "predictor_device.h"
#include "rk5_chain.h"
#include "rk5_models.h"
#include "stepfactor.h"

namespace ngpu {

// ---------------------------------------------------------------------------
// Cash-Karp RK5(4) coefficients (published tableau, same float rounding as
// the reference's __constant__ float table, src/rk5.cu:35-72).
namespace ck {
constexpr float a21 = (float)0.2;
constexpr float a31 = (float)(3.0 / 40.0), a32 = (float)(9.0 / 40.0);
constexpr float a41 = (float)0.3, a42 = (float)-0.9, a43 = (float)1.2;
constexpr float a51 = (float)(-11.0 / 54.0), a52 = (float)2.5,
                a53 = (float)(-70.0 / 27.0), a54 = (float)(35.0 / 27.0);
constexpr float a61 = (float)(1631.0 / 55296.0), a62 = (float)(175.0 / 512.0),
                a63 = (float)(575.0 / 13824.0), a64 = (float)(44275.0 / 110592.0),
                a65 = (float)(253.0 / 4096.0);
constexpr float b1 = (float)(37.0 / 378.0), b3 = (float)(250.0 / 621.0),
                b4 = (float)(125.0 / 594.0), b6 = (float)(512.0 / 1771.0);
constexpr float e1 = (float)(37.0 / 378.0 - 2825.0 / 27648.0),
                e3 = (float)(250.0 / 621.0 - 18575.0 / 48384.0),
                e4 = (float)(125.0 / 594.0 - 13525.0 / 55296.0),
                e5 = (float)(-277.00 / 14336.0), e6 = (float)(512.0 / 1771.0 - 0.25);
// step factors err^-0.25 (reject) and err^-0.2 (accept): stepfactor.h
constexpr float eps = 1.0e-6f, safety = 0.9f, err_min = 1.889568e-4f, scal_min = 0.1f;
// Bound on RK5 attempts per neuron-step.  Finite runs need at most
// (dt/h_min + 1) substeps x ~67 rejections each (h shrinks by >= 1/0.9 per
// rejection down to h_min), i.e. < 70,000 at h_min = dt/1000; the bound only
// ends the loop of a neuron whose state became non-finite.
constexpr int kMaxAttempts = 100000;
}  // namespace ck
using ck::kMaxAttempts;

// The tableau as literals, and as vector registers: a v_fma_f32 takes no
// literal, so literals sit in scalar registers, and a kernel that holds more
// constants, parameters and pointers than its ~100 scalar registers reads
// them back from vector lanes (v_readlane) in every iteration.
struct CkConst {
  static constexpr float a21 = ck::a21, a31 = ck::a31, a32 = ck::a32, a41 = ck::a41;
  static constexpr float a42 = ck::a42, a43 = ck::a43, a51 = ck::a51, a52 = ck::a52;
  static constexpr float a53 = ck::a53, a54 = ck::a54, a61 = ck::a61, a62 = ck::a62;
  static constexpr float a63 = ck::a63, a64 = ck::a64, a65 = ck::a65, b1 = ck::b1;
  static constexpr float b3 = ck::b3, b4 = ck::b4, b6 = ck::b6, e1 = ck::e1;
  static constexpr float e3 = ck::e3, e4 = ck::e4, e5 = ck::e5, e6 = ck::e6;
};
struct CkRegs {
  float a21 = ck::a21, a31 = ck::a31, a32 = ck::a32, a41 = ck::a41;
  float a42 = ck::a42, a43 = ck::a43, a51 = ck::a51, a52 = ck::a52;
  float a53 = ck::a53, a54 = ck::a54, a61 = ck::a61, a62 = ck::a62;
  float a63 = ck::a63, a64 = ck::a64, a65 = ck::a65, b1 = ck::b1;
  float b3 = ck::b3, b4 = ck::b4, b6 = ck::b6, e1 = ck::e1;
  float e3 = ck::e3, e4 = ck::e4, e5 = ck::e5, e6 = ck::e6;
  // values the compiler cannot see through, so they stay where they are
  __device__ inline void hold() {
    asm volatile("" : "+v"(a21), "+v"(a31), "+v"(a32), "+v"(a41), "+v"(a42), "+v"(a43));
    asm volatile("" : "+v"(a51), "+v"(a52), "+v"(a53), "+v"(a54), "+v"(a61), "+v"(a62));
    asm volatile("" : "+v"(a63), "+v"(a64), "+v"(a65), "+v"(b1), "+v"(b3), "+v"(b4));
    asm volatile("" : "+v"(b6), "+v"(e1), "+v"(e3), "+v"(e4), "+v"(e5), "+v"(e6));
  }
};

// ---------------------------------------------------------------------------
// Neuron models (right-hand sides and post-step updates).
// Parameter and variable indices follow the reference's name tables.  Each
// product-plus-sum of the reference's expressions (a*b + c) is one fma: the
// reference's CUDA build contracts by default, though which products its
// compiler fuses is its own choice; this build fixes this pattern (fewer
// instructions on the attempt chain) and the oracle evaluates the same one.
//
// Every division of a right-hand side is by a parameter (M::divisor(j)).
// dv.div(x, p, j) returns x / p[j].  DivIEEE divides.  DivFast, for
// populations whose divisor parameters are uniform with a usable
// reciprocal, multiplies by the double reciprocal (div_recip: the IEEE
// quotient of every dividend, but where the quotient is subnormal, which is
// noted), and rhs() evaluates the whole right-hand side again with DivIEEE
// when a lane of the wave has a nonzero subnormal quotient: one wave-uniform
// branch, normally not taken, per evaluation.
struct DivIEEE {
  __device__ inline float div(float x, const float* p, int j) const { return x / p[j]; }
  __device__ inline float exp_div(float x, const float* p, int j) const { return exp_fma(x / p[j]); }
};
struct DivFast {
  const double* r;
  unsigned int tiny;
  bool far;   // an exponent outside exp_fma_near's range (a subnormal one: exp is 1 either way)
  __device__ inline float div(float x, const float*, int j) { return div_recip(x, r[j], tiny); }
  __device__ inline float exp_div(float x, const float*, int j) {
    const float q = (float)((double)x * r[j]);
    far = !(fabsf(q) <= kExpNear);
    return exp_fma_near(q);
  }
};

// ---------------------------------------------------------------------------
// Right-hand side of a population: with uniform divisor parameters (UNI)
// through DivFast, evaluated again with IEEE divisions when a lane of the
// wave has a subnormal quotient or an exponent out of range.
template <class M, bool UNI>
__device__ inline void rhs(const float* y, float* dy, const float* p, const double* r) {
  if constexpr (UNI) {
    DivFast dv{r, ~0u, false};
    M::deriv(y, dy, p, dv);
    if (__builtin_expect(__any(tiny_noted(dv.tiny) | dv.far), 0)) {
      DivIEEE di;
      M::deriv(y, dy, p, di);
    }
  } else {
    DivIEEE di;
    M::deriv(y, dy, p, di);
  }
}

// err / eps through the double reciprocal (div_recip; a subnormal quotient
// decides nothing: the error ratio is only compared and raised to a power
// when above err_min)
__device__ inline float div_eps(float err) {
  return (float)((double)err * (1.0 / (double)ck::eps));
}

__device__ inline bool lagged_spike(int raw) { return ((unsigned int)raw >> 31) != 0; }

// ---------------------------------------------------------------------------
// One Cash-Karp attempt of step h from (y, k1), src/rk5.h:88-131: the five
// further stages, the 5th-order solution yn and the error ratio
// max_j |h sum_i e_i k_i[j]| / ys[j] (before the division by eps; rel(v, j) is
// v / ys[j]).  Each
// stage's sum_i a_i k_i is accumulated with fma and added to y with one more
// (y + h*(...)), the contracted pattern this build fixes for kernel and oracle.
// C: where the tableau's coefficients are read from (CkConst, CkRegs).
template <class M, class C, class Q, class F>
__device__ inline float rk5_try(const C& c, const float* y, const float* k1, Q&& rel,
                                float h, float* yn, F&& deriv) {
  float k2[M::NV], k3[M::NV], k4[M::NV], k5[M::NV], k6[M::NV];
  const float h21 = h * c.a21;
#pragma unroll
  for (int j = 0; j < M::NV; ++j) yn[j] = fmaf(h21, k1[j], y[j]);
  deriv(yn, k2);
#pragma unroll
  for (int j = 0; j < M::NV; ++j) yn[j] = fmaf(h, fmaf(c.a32, k2[j], c.a31 * k1[j]), y[j]);
  deriv(yn, k3);
#pragma unroll
  for (int j = 0; j < M::NV; ++j) {
    float t = fmaf(c.a42, k2[j], c.a41 * k1[j]);
    t = fmaf(c.a43, k3[j], t);
    yn[j] = fmaf(h, t, y[j]);
  }
  deriv(yn, k4);
#pragma unroll
  for (int j = 0; j < M::NV; ++j) {
    float t = fmaf(c.a52, k2[j], c.a51 * k1[j]);
    t = fmaf(c.a53, k3[j], t);
    t = fmaf(c.a54, k4[j], t);
    yn[j] = fmaf(h, t, y[j]);
  }
  deriv(yn, k5);
#pragma unroll
  for (int j = 0; j < M::NV; ++j) {
    float t = fmaf(c.a62, k2[j], c.a61 * k1[j]);
    t = fmaf(c.a63, k3[j], t);
    t = fmaf(c.a64, k4[j], t);
    t = fmaf(c.a65, k5[j], t);
    yn[j] = fmaf(h, t, y[j]);
  }
  deriv(yn, k6);
  float err = 0.0f;
#pragma unroll
  for (int j = 0; j < M::NV; ++j) {
    float t = fmaf(c.b3, k3[j], c.b1 * k1[j]);
    t = fmaf(c.b4, k4[j], t);
    t = fmaf(c.b6, k6[j], t);
    yn[j] = fmaf(h, t, y[j]);
    float e = fmaf(c.e3, k3[j], c.e1 * k1[j]);
    e = fmaf(c.e4, k4[j], e);
    e = fmaf(c.e5, k5[j], e);
    e = fmaf(c.e6, k6[j], e);
    const float v = rel(h * e, j);
    err = fmaxf(err, fabsf(v));
  }
  return err;
}

// ---------------------------------------------------------------------------
// Adaptive RK5 update of one population, src/rk5.h:69-207: one lane per
// neuron, IEEE divisions (the reference's arithmetic operation by operation).
template <class M>
__global__ void __launch_bounds__(256) rk5_kernel(RK5Args a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = i < a.n;
  unsigned long long n_att = 0, n_rej = 0, n_sub = 0;
  if (active) {
    const int n = a.n;
    float y[M::NV], p[M::NPAR];
#pragma unroll
    for (int j = 0; j < M::NV; ++j) y[j] = a.var[(size_t)j * n + i];
#pragma unroll
    for (int j = 0; j < M::NPAR; ++j)
      p[j] = a.tab.is_per_neuron(j) ? a.param[(size_t)j * n + i] : a.tab.val[j];
    double x = a.x[i];
    float h = a.h[i];
    const double x1 = a.ctx.t1;
    const long long t_idx = a.ctx.t_idx;
    const float h_min = a.h_min;
    const float ref_in = p[M::i_ref];

    bool end_step = false;
    int att_i = 0;
    while (!end_step) {
      const float h_max = (float)(x1 - x);
      // ---- RK5Step ----
      float k1[M::NV];
      float yn[M::NV], ys[M::NV];
      rhs<M, false>(y, k1, p, nullptr);
#pragma unroll
      for (int j = 0; j < M::NV; ++j) ys[j] = fabsf(y[j]) + fabsf(k1[j] * h) + ck::scal_min;
      float err;
      for (;;) {
        if (h > h_max) h = h_max;
        if (h < h_min) h = h_min;
        auto rel = [&](float v, int j) { return v / ys[j]; };
        err = rk5_try<M>(CkConst(), y, k1, rel, h, yn, [&](const float* yy, float* dd) {
          rhs<M, false>(yy, dd, p, nullptr);
        });
        err /= ck::eps;
        ++n_att;
        if (++att_i > kMaxAttempts) {   // non-finite state: end the step (never hit by finite runs)
          x = x1 - h;
          break;
        }
        if (err <= 1.0f || (double)h <= (double)h_min * (1.0 + 1.0e-5)) break;
        ++n_rej;
        const float h_new = h * ck::safety * pow_m025(err);
        h = (float)fmax((double)h_new, 0.1 * (double)h);
      }
      ++n_sub;
      x += h;
      h = (err > ck::err_min) ? h * ck::safety * pow_m02(err) : 5.0f * h;
#pragma unroll
      for (int j = 0; j < M::NV; ++j) y[j] = yn[j];
      // ---- ExternalUpdate ----
      end_step = (x >= x1 - (double)h_min);
      if (y[M::iV] < -1.0e3) {
        y[M::iV] = p[M::i_reset];
        y[M::iw] = 0.0f;
        continue;
      }
      if (y[M::iw] < -1.0e6 || y[M::iw] > 1.0e6) {
        y[M::iV] = p[M::i_reset];
        y[M::iw] = 0.0f;
        continue;
      }
      if (p[M::i_ref] > 0.0f) {
        y[M::iV] = p[M::i_reset];
        if (end_step) p[M::i_ref] -= 1.0f;
      } else if (y[M::iV] >= p[M::i_thr]) {
        emit_spike(a.sl, a.sb, a.ctx.lst, a.i0 + i, i, 1.0f, t_idx, x1);
        y[M::iV] = p[M::i_reset];
        y[M::iw] += p[M::i_jump];
        float r = (float)(int)roundf(p[M::i_tref] / a.dt);
        p[M::i_ref] = r < 0.0f ? 0.0f : r;
      }
    }
#pragma unroll
    for (int j = 0; j < M::NV; ++j) a.var[(size_t)j * n + i] = y[j];
    a.x[i] = x;
    a.h[i] = h;
    if (p[M::i_ref] != ref_in) a.param[(size_t)M::i_ref * n + i] = p[M::i_ref];
  }
  add_wave_counters(a.ctr, (blockIdx.x * blockDim.x + threadIdx.x) / kWave,
                    threadIdx.x & (kWave - 1), n_att, n_rej, n_sub);
}

// ---------------------------------------------------------------------------
// Persistent RK5 update with lane refill (wavefront-ballot compaction).
//
// 99.7% of neuron-steps take a single RK5 attempt, a spiking neuron's step
// ~40.  With one lane per neuron a wave holding one spiking neuron runs ~40
// attempts with 63 idle lanes.  Here each wave owns a contiguous chunk of
// neurons; every iteration is one attempt for all busy lanes (preceded by
// the k1 evaluation for lanes that start a new substep), and lanes whose
// neuron finished the step store it and take the next neurons of the chunk
// (ballot + lane rank; no atomics).  Per neuron the arithmetic is exactly
// that of rk5_kernel.  UNI: every parameter except refractory_step is
// uniform over the population, so parameters come from the kernel-argument
// table and divisions by them use reciprocals (DivFast, bit-identical).
//
// The waves that take the neurons about to spike (the previous launch listed
// them) run the chain form instead of this loop (rk5_chain.h): one neuron
// over a group of lanes.
//
// Step values of one persistent RK5 launch, read where they are used from
// the launch's own kernel arguments (so the compiler reloads them instead of
// holding them in registers): a single-population launch takes them from its
// RK5Args; the multi-population batch kernel from its batch arguments, its
// per-population RK5Args staying in device memory unchanged from step to step.
struct StepFromArgs {
  const RK5Args& a;
  __device__ const StepCtx& ctx() const { return a.ctx; }
  __device__ const StepCtx& pctx() const { return a.pf.ctx; }   // the previous step
  __device__ int prefold() const { return a.prefold; }
  __device__ int defer_cap() const { return a.defer_cap; }
};

// The persistent loop of one wave over its population's share: wave / n_waves
// index the population's waves, ctr_row is the wave's counter row (unique in
// the launch), my_hot / my_spk its LDS buffers of kHotLds / kSpkLds entries,
// s_pred the staged predictor (MODE 2).  Synapses delivered by the wave are
// added to n_dev.
template <class M, bool UNI, int MODE, class SV>
__device__ __attribute__((always_inline)) inline void rk5_persistent_body(
    const RK5Args& a, const SV& sv, const int wave, const int n_waves,
    const int ctr_row, int* my_hot, int* my_spk, PredLDS* s_pred_p, unsigned long long& n_dev) {
  static_assert(MODE == 0 || PredCapable<M>::value, "predictor modes need the AdEx beta model");
  const int lane = threadIdx.x & (kWave - 1);
  const int n = a.n;
  const double x1 = sv.ctx().t1;
  const long long t_idx = sv.ctx().t_idx;
  const int parity = sv.ctx().parity;
  const int lst = sv.ctx().lst;
  // end of the previous step (the end_step_kernel formula one step back): a
  // lagged neuron integrates up to it before starting this step
  const double x1_prev = sv.ctx().t0 + (double)a.dt * (double)sv.ctx().it;
  // the wave's own hot list first (neurons of its chunk that ended the last
  // step about to spike, or split; ~1 per wave, so each takes a lane of its
  // own and the long attempt chains start together in the first iteration),
  // then its chunk, skipping the listed neurons; indices below are relative
  // to the wave's range
  const unsigned char* flag_in = nullptr;
  unsigned char* flag_out = nullptr;
  const int* dense = nullptr;
  int n_hot = 0, q_out = 0;
  constexpr bool kChainOk = MODE != 1 && chain_capable<M>();
  constexpr int kG = chain_lanes(M::NPORT);
  // chain form: wave w < spread takes the hot entries w, w + spread, ... (one
  // per group of lanes), so a launch with few of them gives each a wave of
  // its own (neurons of one wave wait for each other's branches), and the
  // entry is read together with the list's length
  const int spread = kChainOk && a.hot_only ? (a.chain_waves < n_waves / 2 ? a.chain_waves : n_waves / 2) : 0;
  const int my_entry = (lane / kG) * spread + wave;
  int my_node = -1;
  if (a.hot_flag) {
    const int q_in = (int)(t_idx % 3);
    q_out = q_in == 2 ? 0 : q_in + 1;
    const int q_clr = q_out == 2 ? 0 : q_out + 1;   // read by the previous launch
    dense = a.hot_list + (size_t)q_in * n;
    if (wave < spread && my_entry < n) my_node = dense[my_entry];
    n_hot = a.hot_count[q_in];
    if (n_hot > n) n_hot = n;
    flag_in = a.hot_flag + (size_t)parity * n;
    flag_out = a.hot_flag + (size_t)(parity ^ 1) * n;
    if (wave == 0 && lane == 0) a.hot_count[q_clr] = 0;
  }
  // without the chain form wave w takes hot entries [w*hp, w*hp + hp) (one
  // per lane, so the long attempt chains start together in the first
  // iteration, packed into few waves), then its equal share of all neurons
  const bool chain = kChainOk && n_hot > 0 && n_hot <= spread * (kWave / kG);
  int hs = 0, n_hw = 0, w_hot = 0;
  if (chain) {
    w_hot = n_hot < spread ? n_hot : spread;
    n_hw = wave < w_hot ? 1 : 0;   // (the groups' entries are counted by my_entry)
  } else if (n_hot > 0) {
    const int hl = a.hot_lanes < 1 ? 1 : (a.hot_lanes > kWave ? kWave : a.hot_lanes);
    const unsigned int hp =
        n_hot <= n_waves * hl
            ? (unsigned int)hl
            : (((unsigned int)n_hot + n_waves - 1) / n_waves + kWave - 1) & ~(unsigned int)(kWave - 1);
    hs = wave * (int)hp;
    n_hw = hs < n_hot ? (hs + (int)hp < n_hot ? (int)hp : n_hot - hs) : 0;
    w_hot = (int)(((unsigned int)n_hot + hp - 1) / hp);
  }
  // while the hot entries fill less than half the grid, the waves holding
  // them take no share of the bulk (a wave's bulk refills would stall its
  // long chains on memory); the other waves split all neurons, in units of
  // 64, so that no wave has more than one unit more than another (a unit is
  // one iteration: 1e6 neurons over 2,829 waves, 6 iterations in each at
  // equal shares rounded up, 5 in half of them this way)
  const bool hot_only = a.hot_only && w_hot > 0 && 2 * w_hot <= n_waves;
  const int bwave = hot_only ? wave - w_hot : wave;
  int b0 = 0, n_bw = 0;
  if (bwave >= 0) {
    const unsigned int nbw = hot_only ? n_waves - w_hot : n_waves;
    const unsigned int units = ((unsigned int)n + kWave - 1) / kWave;
    const unsigned int per = units / nbw, rem = units - per * nbw;
    const unsigned int u0 = (unsigned int)bwave * per + ((unsigned int)bwave < rem ? bwave : rem);
    const unsigned int u1 = u0 + per + ((unsigned int)bwave < rem ? 1u : 0u);
    b0 = (int)(u0 * kWave);
    const int b1 = (int)(u1 * kWave) < n ? (int)(u1 * kWave) : n;
    n_bw = b1 > b0 ? b1 - b0 : 0;
  }
  int next = 0;
  const int end = n_hw + n_bw;
  // the waves holding the chains issue first; the others fill the free slots
  if (n_hw > 0) __builtin_amdgcn_s_setprio(3);
  // spikes of the wave, appended to the step's list with one atomic when the
  // wave exits (a returning atomic per spike would stall the long chains)
  int scnt = 0;         // spikes of this wave (wave-uniform)
  bool spk = false;     // the lane's neuron spiked in this iteration
  int spk_src = 0;
  int hcnt = 0;         // entries of this wave's hot list for the next step
  int pend = 0;         // bit 0: neuron finished this iteration, bit 1: it is hot
  int pend_i = 0;
  const float h_min = a.h_min;
  float y[M::NV], p[M::NPAR], k1[M::NV], ys[M::NV];
  double x = 0.0;
  double cx1 = 0.0;     // end of the step the lane's neuron is in (x1, or x1_prev if lagged)
  bool lagged = false;
  // Models with many ports fold the previous step's slots in a loop that is not
  // unrolled, over pend_v by selects: unrolled, the loop is too long for the
  // compiler from 8 ports of two variables on, and its arrays went to scratch
  // with it (300,000 neurons: izhikevich_cond_beta, 9 ports, 256 us a step, 203
  // this way; aeif_cond_beta, 12 ports, 446, 354).  With one variable a port
  // that happens from 17 ports on, where scratch costs less than one wave per
  // SIMD would (18 ports: 88, 136 this way); from 13 to 16 ports this form
  // keeps two waves instead of one (16 ports: 108, 81), below it is slower (12
  // ports: 61, 68).
  constexpr bool kCompact =
      M::NPORT > 7 && (M::NV >= 2 + 2 * M::NPORT || (M::NV > 14 && M::NV <= 18));
  // a lagged neuron's stashed input, loaded when the lane takes it, so
  // resuming a split step needs no memory round trip inside the chain
  double pend_v[M::NPORT];
  int rec_k = 0;        // spike-time fill count of the lane's neuron (recording on)
  float h = 0.0f, ref_in = 0.0f;
  int i = -1;
  int att_i = 0;   // attempts of the current neuron in this step
  bool need_k1 = false;
  float el = 1.0f;      // last accepted error ratio (predictor input)
  float h_sub = 0.0f;   // controller proposal at the start of the substep
  bool clip = false;    // accepted attempt was cut by the end of the step
  bool rej_sub = false; // the current substep had a rejected attempt
  unsigned int n_att = 0, n_rej = 0, n_sub = 0, n_split = 0;
#pragma unroll
  for (int j = 0; j < M::NPAR; ++j) p[j] = a.tab.val[j];
  // a spike that found the wave's buffer full: into the list at once
  auto add_now = [&](int src_bits) {
    spike_list_add(a.sl, lst, src_bits, 1.0f);
    if (a.fd.lag_d0_at_exit && lagged_spike(src_bits)) {
      // its d_int = 0 synapses now (the next launch folds their slot)
      const int src = (int)((unsigned int)src_bits & ~kSpikeLagBit);
      n_dev += deliver_segment(a.fd.st, spike_base_slot((unsigned int)src_bits, t_idx, a.fd.st.n_slot),
                               1.0f, a.fd.st.row_ptr[src], a.fd.st.row_ptr[src + 1], 0, 1, 1);
    }
  };
  CkRegs ckr;
  if constexpr (M::NV <= 6) ckr.hold();
  if constexpr (kChainOk) {
    if (chain && n_hw > 0) {
      // the chain's tableau in registers; shared with the loop below, as one
      // set, it cost that loop 24 of them, and from 6 or 7 ports on a kernel
      // then held one wave per SIMD instead of two (1e6 neurons, 7 ports: 70 Hz
      // 254 us a step, 178 this way; 460 Hz 670, 435).  Where both ways fit two
      // waves one set is faster (learned step sizes, 3 ports: 171, 183), and
      // the Izhikevich models, with more neurons hot at once, are with one
      // wave (300,000, 7 ports, 280 Hz: 147, 190)
      constexpr bool kOwn = M::c_mx >= 0 && M::NV > (MODE == 2 ? 10 : UNI ? 12 : 14);
      CkRegs own;
      const CkRegs& ckc = kOwn ? own : ckr;
      if constexpr (kOwn)
        own.hold();
      else if constexpr (M::NV > 6)
        ckr.hold();
      // ---- chain form: one neuron per group of kG lanes (rk5_chain.h) ----
      const int role = lane & (kG - 1), k = role - 1;
      const bool mem = role == 0, port = role >= 1 && role <= M::NPORT;
      const int ia = mem ? M::iV : port ? M::c_ya(k) : -1;
      const int ib = mem ? M::iw : port ? M::c_yb(k) : -1;
      const bool busy0 = my_entry < n_hot;
      bool busy = busy0;
      float ya[2] = {0.0f, 0.0f}, k1a[2] = {0.0f, 0.0f}, ysa[2] = {1.0f, 1.0f};
      ChainDiv d{1.0f, 1.0f, 1.0f, 1.0, 1.0, 1.0};
      double in_add = -0.0;  // the port's stashed input while the neuron is lagged (-0: none)
      float in_wt = 1.0f;    // weight of the port's input
      if (busy0) {
        i = my_node;
        if (ia >= 0) ya[0] = a.var[(size_t)ia * n + i];
        if (ib >= 0) ya[1] = a.var[(size_t)ib * n + i];
        p[M::i_ref] = a.param[(size_t)M::i_ref * n + i];
        if constexpr (!UNI) {
#pragma unroll
          for (int j = 0; j < M::NPAR; ++j)
            if (a.tab.is_per_neuron(j)) p[j] = a.param[(size_t)j * n + i];
        }
        const int ja = mem ? M::c_mv : port ? M::c_da(k) : -1;
        const int jb = mem ? M::c_mw : port ? M::c_db(k) : -1;
        if (ja >= 0) d.da = a.param[(size_t)ja * n + i];
        if (jb >= 0) d.db = a.param[(size_t)jb * n + i];
        if (port && M::in_w(0) >= 0) in_wt = a.param[(size_t)M::in_w(k) * n + i];
        x = a.x[i];
        h = a.h[i];
        lagged = a.lag ? a.lag[i] != 0 : false;
        if (port) {
          const long long lo = (long long)k * n;
          double acc = 0.0;
          if (sv.prefold()) {
            const FoldArgs& f = a.pf;
            double* rp = f.ring + (size_t)sv.pctx().slot * f.n_ch + (size_t)(f.ch_base + lo + i);
            acc = poisson_input<true>(f, lo + i, *rp, sv.pctx().t1, sv.pctx().t_idx,
                                f.pu_b < lo + n && f.pu_e > lo);
            *rp = 0.0;
          } else if (lagged) {
            acc = a.pend[lo + i];
          }
          if (acc != 0.0) {
            constexpr int in = M::in_y(0) == M::c_ya(0) ? 0 : 1;
            if (lagged)
              in_add = acc * (double)in_wt;
            else
              ya[in] = fold_add(ya[in], acc, in_wt);
          }
        }
        if (mem && a.sb.max_rec > 0) rec_k = a.sb.n_rec[i];
        if constexpr (MODE == 2) el = a.err_last[i];
        ref_in = p[M::i_ref];
        if constexpr (M::c_mx >= 0) d.dx = p[M::c_mx < 0 ? 0 : M::c_mx];
        cx1 = lagged ? x1_prev : x1;
        need_k1 = true;
        // the loads complete here, not in the loop
        asm volatile("" ::"v"(ya[0]), "v"(ya[1]), "v"(ref_in), "v"(d.da), "v"(d.db), "v"(in_add),
                     "v"(x), "v"(h), "v"(rec_k), "v"(el));
      }
      d.ra = recip_double(d.da);
      d.rb = recip_double(d.db);
      d.rx = recip_double(d.dx);
      // (uniform populations: the launch checked the divisors)
      const bool ieee = !UNI && __any(!(__builtin_isnormal(d.da) && __builtin_isnormal(d.db) &&
                                        __builtin_isnormal(d.dx)));
#pragma unroll
      for (int j = 0; j < M::NPAR; ++j) asm volatile("" : "+v"(p[j]));
      // controller constants: the largest float h that passes the test
      // (double)h <= (double)h_min * (1 + 1e-5), and the end of the step
      float h_crit;
      {
        const double hc = (double)h_min * (1.0 + 1.0e-5);
        h_crit = (float)hc;
        if ((double)h_crit > hc) h_crit = __uint_as_float(__float_as_uint(h_crit) - 1u);
      }
      double x_end = cx1 - (double)h_min;
      const int cap = sv.defer_cap();
      // i for an address that is to be computed where it is used: hoisted out
      // of the loop such addresses held 24 registers, and the kernel spilled
      auto here = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
      };
      // The arithmetic runs unmasked in all 64 lanes, groups without a (busy)
      // neuron on harmless values, and only what follows from it is selected
      // by `busy`: a wave whose EXEC mask holds fewer than 16 lanes issues
      // these instructions at a half to a third of the rate (measured: one
      // iteration 1,820 cycles with 16 to 64 lanes on, 4,700-5,800 with 4
      // lanes on in each of a compute unit's four waves).
      //
      // k1 of the next attempt is taken from the new state yn beside the error
      // ratio and the step factor, before the attempt is accepted: two serial
      // chains side by side cost little more than one here (8 cycles a
      // dependent instruction, 4-5 an independent one).  It is taken again
      // where an event changed the state.
      auto k1_of = [&](bool sel) {
        float kn[2];
        ChainNote nt{ieee ? 0u : ~0u, 0.0f};
        chain_rhs<M, true>(ya, kn, p, d, mem, nt);
        if (__any(sel & nt.set())) chain_rhs<M, false>(ya, kn, p, d, mem, nt);
        k1a[0] = sel ? kn[0] : k1a[0];
        k1a[1] = sel ? kn[1] : k1a[1];
      };
      k1_of(busy);
      if (__any(busy))
      for (;;) {
        const bool fresh = busy && need_k1;
        if constexpr (MODE == 2) {
          // learned proposal, as in the loop below; the membrane lanes hold
          // the neurons' inputs (columns of the matrix product)
          const bool start = fresh && h < (float)(cx1 - x);
          if (__any(start)) {
            float yy[M::NV], raw[kPI];
            yy[0] = ya[0];
            yy[1] = ya[1];
#pragma unroll
            for (int q = 0; q < M::NPORT; ++q) {
              yy[2 + 2 * q] = chain_from(ya[0], q + 1);
              yy[3 + 2 * q] = chain_from(ya[1], q + 1);
            }
            pred_raw_inputs<M::NPORT>(yy, h, el, a.dt, raw);
#pragma unroll
            for (int q = 0; q < kPI; ++q) raw[q] = busy && mem ? raw[q] : 0.0f;
            const float o = __shfl(pred_infer_wave(*s_pred_p, raw), lane & ~(kG - 1), kWave);
            if (start && o > -60.0f && o < 60.0f)
              h = fminf(h, fmaxf(a.dt * exp2f(o), 2.0f * h_min));
          }
        }
        ChainNote nt{ieee ? 0u : ~0u, 0.0f};
#pragma unroll
        for (int j = 0; j < 2; ++j)
          ysa[j] = fresh ? fabsf(ya[j]) + fabsf(k1a[j] * h) + ck::scal_min : ysa[j];
        const float h_max = (float)(cx1 - x);
        float hh = h;
        if (hh > h_max) hh = h_max;
        if (hh < h_min) hh = h_min;
        const double xn = x + hh;
        float yn[2], kn[2];
        const double rs[2] = {recip_double(ysa[0]), recip_double(ysa[1])};
        // (a subnormal ratio counts only as the learned form's input; a scale
        // of inf gives NaN for 0 here, neither of which changes the maximum)
        auto rel = [&](float v, int j) {
          if constexpr (MODE == 2) return div_recip(v, rs[j], nt.tiny);
          return (float)((double)v * rs[j]);
        };
        float err = rk5_try<ChainNV>(ckc, ya, k1a, rel, hh, yn, [&](const float* yy, float* dd) {
          chain_rhs<M, true>(yy, dd, p, d, mem, nt);
        });
        chain_rhs<M, true>(yn, kn, p, d, mem, nt);
        const float err0 = chain_max<kG>(err);
        err = div_eps(err0);
        bool ok = (err <= 1.0f) | (hh <= h_crit);
        float pw = pow_step_chain(err0, err, ok);
        att_i += busy;
        bool over = false;
        // What is not an ordinary attempt sits behind one branch.  Rare cases:
        // a subnormal quotient (all divisions again by IEEE), the attempt
        // bound of a non-finite state, an error ratio outside the range of
        // the fast step factor.  Events: ExternalUpdate acts on the membrane,
        // the step ends or is split.
        const bool need = !ok | (err > ck::err_min);
        const bool rare = busy & (nt.set() | (att_i > kMaxAttempts) |
                                  (need & !((err >= kPowLo) & (err <= kPowHi))));
        const bool split = (cap > 0) & !lagged & (att_i >= cap);
        const bool ext = mem & ((yn[0] < -1.0e3f) | (yn[0] >= p[M::i_thr]) |
                                (fabsf(yn[1]) > 1.0e6f) | (p[M::i_ref] > 0.0f));
        const bool event = busy & ok & (ext | (xn >= x_end) | split);
        const bool other = __any(rare | event);
        if (__builtin_expect(other, 0) && __any(rare)) {
          if (__any(busy & nt.set())) {
            auto rel = [&](float v, int j) { return v / ysa[j]; };
            err = rk5_try<ChainNV>(ckc, ya, k1a, rel, hh, yn, [&](const float* yy, float* dd) {
              chain_rhs<M, false>(yy, dd, p, d, mem, nt);
            });
            chain_rhs<M, false>(yn, kn, p, d, mem, nt);
            err = div_eps(chain_max<kG>(err));
          }
          if (busy & (att_i > kMaxAttempts)) {   // non-finite state: end the step
            x = cx1;
            err = 0.0f;
            over = true;
          }
          ok = (err <= 1.0f) | (hh <= h_crit);
          pw = pow_step_dev(err, ok, busy & (!ok | (err > ck::err_min)));
        }
        const bool done = busy && ok;   // accepted (src/rk5.h:135-159)
        n_att += busy && mem;
        n_rej += busy && mem && !ok;
        n_sub += done && mem;
        // (float)max of the doubles is the max of the floats
        const float hp = hh * ck::safety * pw;
        const float h_rej = fmaxf(hp, (float)(0.1 * (double)hh));
        const float h_acc = err > ck::err_min ? hp : 5.0f * hh;
        x = done && !over ? xn : x;
        h = busy ? (ok ? h_acc : h_rej) : h;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          ya[j] = done ? yn[j] : ya[j];
          k1a[j] = done ? kn[j] : k1a[j];
        }
        need_k1 = busy ? ok : need_k1;
        if constexpr (MODE == 2) el = done ? err : el;
        if (!other) continue;
        const bool end_step = x >= x_end;
        const bool m = done & mem;
        const bool off = m && (ya[0] < -1.0e3 || ya[1] < -1.0e6 || ya[1] > 1.0e6);
        const bool refr = m && !off && p[M::i_ref] > 0.0f;
        const bool fire = m && !off && !refr && ya[0] >= p[M::i_thr];
        ya[0] = off || refr ? p[M::i_reset] : ya[0];
        ya[1] = off ? 0.0f : ya[1];
        p[M::i_ref] = refr && end_step ? p[M::i_ref] - 1.0f : p[M::i_ref];
        const unsigned long long ms = __ballot(fire);
        if (ms) {
          if (fire) {
            const int v = here(i);
            spike_book(a.sb, a.i0 + v, v, 1.0f, lagged ? t_idx - 1 : t_idx, cx1, &rec_k);
            const int src = lagged ? (int)((unsigned int)(a.i0 + v) | kSpikeLagBit) : a.i0 + v;
            ya[0] = p[M::i_reset];
            ya[1] += p[M::i_jump];
            const float rr = (float)(int)roundf(p[M::i_tref] / a.dt);
            p[M::i_ref] = rr < 0.0f ? 0.0f : rr;
            const int pos = scnt + __popcll(ms & ((1ull << lane) - 1ull));
            if (pos < kSpkLds)
              my_spk[pos] = src;
            else
              add_now(src);
          }
          scnt += __popcll(ms);
        }
        const bool resume = done && end_step && lagged;   // the previous step is complete
        const bool leave = done && !resume && (end_step || split);
        if (__any(resume)) {
          constexpr int in = M::in_y(0) == M::c_ya(0) ? 0 : 1;
          if (resume) {
            if (port) ya[in] = (float)((double)ya[in] + in_add);
            if (mem) a.lag[here(i)] = 0;
            lagged = false;
            cx1 = x1;
            x_end = cx1 - (double)h_min;
            att_i = 0;
          }
        }
        if (__any(leave)) {
          // end of the step, or split: stored; hot again when split or still
          // in the upswing (at most 64 / kG entries per wave)
          bool hot = false;
          if (leave) {
            if (ia >= 0) a.var[(size_t)ia * n + i] = ya[0];
            if (ib >= 0) a.var[(size_t)ib * n + i] = ya[1];
            if (mem) {
              if (!end_step) {
                a.lag[here(i)] = 1;
                ++n_split;
              }
              a.x[i] = x;
              a.h[i] = h;
              if constexpr (MODE == 2) a.err_last[i] = el;
              if (p[M::i_ref] != ref_in) a.param[(size_t)M::i_ref * n + here(i)] = p[M::i_ref];
              hot = !end_step || (p[M::i_ref] <= 0.0f && ya[0] >= M::hot_v(p, a.hot_margin));
              flag_out[i] = hot ? 1 : 0;
            }
            busy = false;
          }
          const unsigned long long mh = __ballot(hot);
          if (hot) my_hot[hcnt + __popcll(mh & ((1ull << lane) - 1ull))] = i;
          hcnt += __popcll(mh);
          if (!__any(busy)) break;
        }
        if (__any(off | refr | fire | resume)) k1_of(done & busy);
      }
      next = end;   // a chain wave takes no share of the bulk
    }
  }
  double r[M::NPAR];
#pragma unroll
  for (int j = 0; j < M::NPAR; ++j) r[j] = UNI && M::divisor(j) ? recip_uniform(p[j]) : 0.0;
  if constexpr (M::NV <= 6 && UNI) {
#pragma unroll
    for (int j = 0; j < M::NPAR; ++j)
      if (M::divisor(j)) asm volatile("" : "+v"(r[j]));
  }
  if (!kChainOk || !(chain && n_hw > 0))
  for (;;) {
    // ---- refill idle lanes from the wave's chunk ----
    const bool want = (i < 0) && next < end;
    const unsigned long long m = __ballot(want);
    if (m) {
      if (want) {
        const int v = next + __popcll(m & ((1ull << lane) - 1ull));
        int cand = -1;
        if (v < end) cand = v < n_hw ? dense[hs + v] : b0 + (v - n_hw);
        int f = 1;
        if (cand >= 0) {
          // every load of the neuron that depends on nothing else goes out
          // together with its hot flag and its ring slots, and a neuron found
          // on the hot list is dropped afterwards: one round trip to memory
          // for a refill, where the flag first, then the state, then each
          // port's slot took three (1e6 AdEx neurons, with the key schedule of
          // poisson_draw_wave: 67.3 -> 66.0 us a step)
          i = cand;
          f = flag_in && v >= n_hw ? (int)flag_in[i] : 0;
#pragma unroll
          for (int j = 0; j < M::NV; ++j) y[j] = a.var[(size_t)j * n + i];
          if (UNI) {
            p[M::i_ref] = a.param[(size_t)M::i_ref * n + i];
          } else {
#pragma unroll
            for (int j = 0; j < M::NPAR; ++j)
              if (a.tab.is_per_neuron(j)) p[j] = a.param[(size_t)j * n + i];
          }
          x = a.x[i];
          h = a.h[i];
          if constexpr (MODE != 0) el = a.err_last[i];
          lagged = a.lag ? a.lag[i] != 0 : false;
          double slot_v[M::NPORT];   // (kCompact: in pend_v)
          const long long slot_0 = (long long)sv.pctx().slot * a.pf.n_ch + a.pf.ch_base + i;
          if (sv.prefold()) {
#pragma unroll
            for (int k = 0; k < M::NPORT; ++k) (kCompact ? pend_v[k] : slot_v[k]) = a.pf.ring[slot_0 + (long long)k * n];
          }
          if (f != 0) i = -1;
          ref_in = p[M::i_ref];
          if (f == 0) {
            if (sv.prefold()) {
              // the previous step's fold of this neuron's channels (the fold
              // kernel's arithmetic): added to the input variables, or kept
              // as the stashed input of a neuron still inside that step
              const FoldArgs& pf = a.pf;
              auto fold = [&](int k, double slot) {
                const long long lo = (long long)k * n;
                const double acc = poisson_input<true>(pf, lo + i, slot, sv.pctx().t1,
                                                       sv.pctx().t_idx,
                                                       pf.pu_b < lo + n && pf.pu_e > lo);
                pf.ring[slot_0 + lo] = 0.0;
                return acc;
              };
              if constexpr (kCompact) {
#pragma unroll 1
                for (int k = 0; k < M::NPORT; ++k) {
                  double v = 0.0;
#pragma unroll
                  for (int j = 0; j < M::NPORT; ++j) v = j == k ? pend_v[j] : v;
                  v = fold(k, v);
#pragma unroll
                  for (int j = 0; j < M::NPORT; ++j) pend_v[j] = j == k ? v : pend_v[j];
                }
              }
#pragma unroll
              for (int k = 0; k < M::NPORT; ++k) {
                const double acc = kCompact ? pend_v[k] : fold(k, slot_v[k]);
                if (lagged) {
                  pend_v[k] = acc;
                } else if (acc != 0.0) {
                  const int wj = M::in_w(k);
                  const float w = wj >= 0 ? p[wj < 0 ? 0 : wj] : 1.0f;
                  y[M::in_y(k)] = fold_add(y[M::in_y(k)], acc, w);
                }
              }
            } else if (lagged) {
#pragma unroll
              for (int k = 0; k < M::NPORT; ++k) pend_v[k] = a.pend[(size_t)k * n + i];
            }
            if (a.sb.max_rec > 0) rec_k = a.sb.n_rec[i];
            cx1 = lagged ? x1_prev : x1;
            need_k1 = true;
            att_i = 0;
            // the loads complete here: left pending, the compiler waits for them
            // where the paths join (the k1 evaluation of every later
            // iteration), and that wait, counting stores too, would hold the
            // chain on the stores of finished neurons
#pragma unroll
            for (int j = 0; j < M::NV; ++j) asm volatile("" ::"v"(y[j]));
            if (UNI) {
              asm volatile("" ::"v"(p[M::i_ref]));
            } else {
#pragma unroll
              for (int j = 0; j < M::NPAR; ++j)
                if (a.tab.is_per_neuron(j)) asm volatile("" ::"v"(p[j]));
            }
            asm volatile("" ::"v"(x), "v"(h));
            if constexpr (MODE != 0) asm volatile("" ::"v"(el));
            if (lagged) {
#pragma unroll
              for (int k = 0; k < M::NPORT; ++k) asm volatile("" ::"v"(pend_v[k]));
            }
            if (a.sb.max_rec > 0) asm volatile("" ::"v"(rec_k));
          }
        }
      }
      next += __popcll(m);
    }
    // all lanes idle with the chunk not exhausted (every candidate was on
    // the hot list): the masked iteration below does nothing, refill again
    if (!__any(i >= 0) && next >= end) break;
    if constexpr (MODE == 2) {
      // learned proposal for every lane starting a substep whose controller
      // proposal ends inside the step (one cut by the step end, the quiet
      // neuron's usual single substep, is left alone); whole wave on the
      // matrix cores, lanes without a neuron feed zeros
      const bool start = (i >= 0) && need_k1 && h < (float)(cx1 - x);
      if (__any(start)) {
        float raw[kPI];
        if (i >= 0) {
          pred_raw_inputs<M::NPORT>(y, h, el, a.dt, raw);
        } else {
#pragma unroll
          for (int k = 0; k < kPI; ++k) raw[k] = 0.0f;
        }
        const float o = pred_infer_wave(*s_pred_p, raw);
        // the learned proposal only shortens the controller's (the error
        // scale |y| + |k1 h| + 0.1 grows with h, so a longer step than the
        // controller's could pass the test less accurately); floored at
        // 2 h_min, since a step at h_min is accepted whatever its error
        if (start && o > -60.0f && o < 60.0f)
          h = fminf(h, fmaxf(a.dt * exp2f(o), 2.0f * h_min));
      }
    }
    if (i >= 0) {
      // ---- start of a substep: k1 and the error scale (src/rk5.h:83-86) ----
      if (need_k1) {
        if constexpr (MODE == 1) {
          h_sub = h;
          rej_sub = false;
        }
        rhs<M, UNI>(y, k1, p, r);
#pragma unroll
        for (int j = 0; j < M::NV; ++j) ys[j] = fabsf(y[j]) + fabsf(k1[j] * h) + ck::scal_min;
        need_k1 = false;
      }
      // ---- one attempt (src/rk5.h:88-131) ----
      const float h_max = (float)(cx1 - x);
      clip = false;
      if (h > h_max) {
        h = h_max;
        clip = true;
      }
      if (h < h_min) h = h_min;
      float yn[M::NV];
      auto rel = [&](float v, int j) { return v / ys[j]; };
      float err = rk5_try<M>(ckr, y, k1, rel, h, yn, [&](const float* yy, float* dd) {
        rhs<M, UNI>(yy, dd, p, r);
      });
      err = div_eps(err);
      ++n_att;
      if (++att_i > kMaxAttempts) {   // non-finite state: end the step (never hit by finite runs)
        x = cx1;
        err = 0.0f;
      }
      const bool ok = err <= 1.0f || (double)h <= (double)h_min * (1.0 + 1.0e-5);
      const float pw = pow_step_dev(err, ok, !ok || err > ck::err_min);
      if (!ok) {
        ++n_rej;   // rejected: shrink h, retry with the same k1 and scale
        if constexpr (MODE == 1) rej_sub = true;
        const float h_new = h * ck::safety * pw;
        h = (float)fmax((double)h_new, 0.1 * (double)h);
      } else {
        ++n_sub;   // accepted (src/rk5.h:135-159), then ExternalUpdate
        if constexpr (MODE == 1) {
          if (i % a.log_stride == 0) {
            float raw[kPI];
            pred_raw_inputs<M::NPORT>(y, h_sub, el, a.dt, raw);
            const unsigned long long pos = atomicAdd(a.log_count, 1ull);
            if (pos < (unsigned long long)a.log_cap) {
              float* rec = a.log_buf + pos * kLogCols;
#pragma unroll
              for (int k = 0; k < kPI; ++k) rec[k] = raw[k];
              rec[kPI] = __log2f(h / a.dt);
              // lower bound only (censored): h cut by the end of the step,
              // or accepted at the first try (a longer step might have
              // passed too); exact after a rejection, where the controller
              // overshot and the accepted h is what should have been proposed
              rec[kPI + 1] = (clip || !rej_sub) ? 1.0f : 0.0f;
            }
          }
        }
        if constexpr (MODE != 0) el = err;
        if (att_i <= kMaxAttempts) x += h;
        h = (err > ck::err_min) ? h * ck::safety * pw : 5.0f * h;
#pragma unroll
        for (int j = 0; j < M::NV; ++j) y[j] = yn[j];
        need_k1 = true;
        const bool end_step = (x >= cx1 - (double)h_min);
        if (y[M::iV] < -1.0e3 || y[M::iw] < -1.0e6 || y[M::iw] > 1.0e6) {
          y[M::iV] = p[M::i_reset];
          y[M::iw] = 0.0f;
        } else if (p[M::i_ref] > 0.0f) {
          y[M::iV] = p[M::i_reset];
          if (end_step) p[M::i_ref] -= 1.0f;
        } else if (y[M::iV] >= p[M::i_thr]) {
          spike_book(a.sb, a.i0 + i, i, 1.0f, lagged ? t_idx - 1 : t_idx, cx1, &rec_k);
          spk = true;
          spk_src = lagged ? (int)((unsigned int)(a.i0 + i) | kSpikeLagBit) : a.i0 + i;
          y[M::iV] = p[M::i_reset];
          y[M::iw] += p[M::i_jump];
          const float rr = (float)(int)roundf(p[M::i_tref] / a.dt);
          p[M::i_ref] = rr < 0.0f ? 0.0f : rr;
        }
        if (end_step && lagged) {
          // the previous step is complete: add its input (computed when the
          // lane took the neuron, or stashed by that step's fold launch; the
          // fold's arithmetic), then go on with this step
#pragma unroll
          for (int k = 0; k < M::NPORT; ++k) {
            const double acc = pend_v[k];
            if (acc != 0.0) {
              const int wj = M::in_w(k);
              const float w = wj >= 0 ? p[wj < 0 ? 0 : wj] : 1.0f;
              y[M::in_y(k)] = fold_add(y[M::in_y(k)], acc, w);
            }
          }
          a.lag[i] = 0;
          lagged = false;
          cx1 = x1;
          att_i = 0;
        } else if (end_step || (sv.defer_cap() > 0 && !lagged && att_i >= sv.defer_cap())) {
          // end of the step, or split: the neuron is stored mid-step with
          // lag = 1 (and listed hot, so the next launch resumes it first)
          if (!end_step) {
            a.lag[i] = 1;
            ++n_split;
          }
#pragma unroll
          for (int j = 0; j < M::NV; ++j) a.var[(size_t)j * n + i] = y[j];
          a.x[i] = x;
          a.h[i] = h;
          if constexpr (MODE != 0) a.err_last[i] = el;
          if (p[M::i_ref] != ref_in) a.param[(size_t)M::i_ref * n + i] = p[M::i_ref];
          pend = 1 | ((!end_step || (p[M::i_ref] <= 0.0f && y[M::iV] >= M::hot_v(p, a.hot_margin))) ? 2 : 0);
          pend_i = i;
          i = -1;
        }
      }
    }
    // spikes of this iteration into the wave's buffer (the list itself when
    // the buffer is full)
    {
      const unsigned long long ms = __ballot(spk);
      if (spk) {
        const int pos = scnt + __popcll(ms & ((1ull << lane) - 1ull));
        if (pos < kSpkLds) {
          my_spk[pos] = spk_src;
        } else {
          add_now(spk_src);
        }
        spk = false;
      }
      scnt += __popcll(ms);
    }
    // neurons that finished the step: next step's hot list and flags
    if (a.hot_flag) {
      const unsigned long long mh = __ballot(pend == 3);
      if (pend) {
        bool listed = false;
        if (pend == 3) {
          const int pos = hcnt + __popcll(mh & ((1ull << lane) - 1ull));
          if (pos < kHotLds) {
            my_hot[pos] = pend_i;
            listed = true;
          }
        }
        flag_out[pend_i] = listed ? 1 : 0;
        pend = 0;
      }
      hcnt += __popcll(mh);
    }
  }
  {
    // the wave's spikes into the step's list and its hot entries into the
    // next step's (one atomic each; the order within a list does not matter:
    // delivery sums exactly, scheduling changes no arithmetic).  Both atomics
    // and the lagged spikes' segment bounds are in flight together.
    const int n_spk = scnt < kSpkLds ? scnt : kSpkLds;
    const int n_list = hcnt < kHotLds ? hcnt : kHotLds;
    int spk_base = 0, hot_base = 0;
    if (lane == 0) {
      if (n_spk > 0) spk_base = atomicAdd(a.sl.count + lst, n_spk);
      if (n_list > 0) hot_base = atomicAdd(a.hot_count + q_out, n_list);
    }
    // the d_int = 0 synapses of the wave's lagged spikes: their slot (t_idx)
    // is folded by the next launch; the other synapses are delivered with the
    // list by the next launch's idle waves
    if (a.fd.lag_d0_at_exit && n_spk > 0)
      n_dev += deliver_lagged_d0(a.fd.st, my_spk, n_spk, t_idx, lane);
    if (n_spk > 0) {
      const int pos = __builtin_amdgcn_readfirstlane(spk_base) + lane;   // kSpkLds entries: one per lane
      if (lane < n_spk) {
        if (pos < a.sl.cap) {
          a.sl.src[(size_t)lst * a.sl.cap + pos] = my_spk[lane];
          a.sl.height[(size_t)lst * a.sl.cap + pos] = 1.0f;
        } else {
          atomicAdd(a.sl.overflow, 1);
        }
      }
    }
    if (n_list > 0) {
      int* out = a.hot_list + (size_t)q_out * n + __builtin_amdgcn_readfirstlane(hot_base);
      for (int e = lane; e < n_list; e += kWave) out[e] = my_hot[e];
    }
    if (a.ctr) {
      // (no value is read back, so the wave does not wait)
      const unsigned int c[5] = {wave_sum32(n_att), wave_sum32(n_rej), wave_sum32(n_sub),
                                 (unsigned int)n_list, wave_sum32(n_split)};
      unsigned long long* row = a.ctr + (size_t)ctr_row * kCtrCols;
#pragma unroll
      for (int k = 0; k < 5; ++k)
        if (lane == 0 && c[k]) atomicAdd(row + (k < 3 ? k : k + 1), (unsigned long long)c[k]);
    }
  }
}
static_assert(kSpkLds <= kWave, "one spike entry per lane when the wave's buffer is written out");

// Fused delivery: the previous step's spike list, taken from the last wave of
// the launch down so that the first waves (the hot ones, which end last) take
// none while there are fewer spikes than waves.  Few spikes with long segments
// are shared by up to 2^parts_log2 waves each (the last half of the launch's
// waves), so a segment takes one round of record loads instead of several one
// after the other.  Returns the synapses delivered by the lane.
// n_prev: the list's length, read when the launch began.
__device__ inline unsigned long long deliver_prev_list(const FusedDeliver& fd, const SpikeList& sl,
                                                       int n_prev, int wave, int n_waves, int lane) {
  unsigned long long n_dev = 0;
  const int pl = fd.prev_lst;
  if (n_prev > sl.cap) n_prev = sl.cap;
  const int* srcs = sl.src + (size_t)pl * sl.cap;
  const float* hts = sl.height + (size_t)pl * sl.cap;
  int lg = 0;   // log2 of the parts
  while (lg < fd.parts_log2 && ((long long)n_prev << (lg + 2)) <= n_waves) ++lg;
  for (int it = n_waves - 1 - wave; it < n_prev << lg; it += n_waves) {
    const int sp = it >> lg, part = it & ((1 << lg) - 1);
    const unsigned int raw = (unsigned int)srcs[sp];
    const int src = (int)(raw & ~kSpikeLagBit);
    const int mode = (fd.skip_lagged_d0 && (raw >> 31)) ? 2 : 0;
    n_dev += deliver_segment(fd.st, spike_base_slot(raw, fd.prev_t_idx, fd.st.n_slot), hts[sp],
                             fd.st.row_ptr[src], fd.st.row_ptr[src + 1], part * kWave + lane,
                             kWave << lg, mode);
  }
  if (wave == 0 && lane == 0 && fd.spikes && n_prev) atomicAdd(fd.spikes, (unsigned long long)n_prev);
  return n_dev;
}

// Clears the count of the spike list the next step writes (with fused
// delivery no delivery launch does: it held the list of step t_idx - 2,
// delivered by the previous launch).
__device__ inline void clear_next_spike_list(const SpikeList& sl, int lst) {
  sl.count[lst == kSpikeLists - 1 ? 0 : lst + 1] = 0;
}

// Register budget of a small model's kernel (at most 6 state variables): 168
// VGPRs, 3 waves per SIMD.  The chain form keeps the tableau and the
// parameters in vector registers; held to 128 VGPRs (4 waves) it spilled 51
// of them, and the bulk of a launch runs as fast with 3 waves as with 4.
// Models of 17 and 18 state variables (8 ports of two each) are held to 256, 2
// waves: without, some need a few more (300,000 neurons, 8 ports, per-neuron C_m:
// one wave 274 us a step, two 194).  With 20 and more two waves spill: 300,000
// neurons, 10 ports, 70 Hz, one wave 223, two 274.
template <class M, bool UNI, int MODE>
__global__ void __launch_bounds__(kRK5Block)
__attribute__((amdgpu_waves_per_eu(MODE == 1 || M::NV > 18 ? 1 : M::NV > 16 ? 2 : M::NV > 6 ? 1 : MODE == 2 ? 2 : 3)))
rk5_persistent_kernel(RK5Args a) {
  __shared__ int s_hot[kRK5Block / kWave][kHotLds];
  __shared__ int s_spk[kRK5Block / kWave][kSpkLds];
  __shared__ PredLDS s_pred;
  if constexpr (MODE == 2) {
    pred_stage(s_pred, a.pred_params);
    __syncthreads();
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wave = blockIdx.x * (blockDim.x / kWave) + wib;
  const int n_waves = gridDim.x * (blockDim.x / kWave);
  if (a.clear_next_list && blockIdx.x == 0 && threadIdx.x == 0) clear_next_spike_list(a.sl, a.ctx.lst);
  const StepFromArgs sv{a};
  const int n_prev = a.fd.enable ? a.sl.count[a.fd.prev_lst] : 0;
  unsigned long long n_dev = 0;   // synapses delivered by this lane (fused delivery)
  rk5_persistent_body<M, UNI, MODE>(a, sv, wave, n_waves, wave, s_hot[wib],
                                    s_spk[wib], &s_pred, n_dev);
  if (a.fd.enable) n_dev += deliver_prev_list(a.fd, a.sl, n_prev, wave, n_waves, lane);
  if (a.ctr) {
    const unsigned int ev = wave_sum32((unsigned int)n_dev);
    if (lane == 0 && ev) atomicAdd(a.ctr + (size_t)wave * kCtrCols + 3, (unsigned long long)ev);
  }
}

inline int persistent_grid(int n, int max_blocks) {
  const int waves_needed = (n + kWave - 1) / kWave;
  int grid = (waves_needed + kRK5Block / kWave - 1) / (kRK5Block / kWave);
  if (max_blocks > 0 && grid > max_blocks) grid = max_blocks;
  return grid;
}


// Blocks of one persistent RK5 instantiation that are resident on the device
// at once (its register and LDS use decide; every block must be resident,
// since each wave owns a static chunk of the population).
template <class M, bool UNI, int MODE>
static int resident_blocks() {
  static int blocks = 0;
  if (blocks == 0) {
    int per_cu = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, rk5_persistent_kernel<M, UNI, MODE>,
                                                     kRK5Block, 0) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        per_cu <= 0 || cus <= 0)
      throw std::runtime_error("cannot query the occupancy of the persistent RK5 kernel");
    blocks = per_cu * cus;
  }
  return blocks;
}

template <class M, bool UNI, int MODE>
static void launch_persistent(const RK5Args& a, hipStream_t s) {
  // enough waves to fill the GPU with every block resident, at most one
  // lane per neuron
  int cap = resident_blocks<M, UNI, MODE>();
  if (a.max_blocks > 0 && a.max_blocks < cap) cap = a.max_blocks;
  const int grid = persistent_grid(a.n, cap);
  hipLaunchKernelGGL((rk5_persistent_kernel<M, UNI, MODE>), dim3(grid), dim3(kRK5Block), 0, s, a);
}

template <class M>
static void launch_rk5_t(const RK5Args& a, hipStream_t s) {
  const int block = kRK5Block;
  if (a.persistent) {
    if constexpr (M::NPORT > kFastPort) {
      // many ports: one persistent variant (parameters per lane, IEEE
      // divisions), the same arithmetic as the others
      launch_persistent<M, false, 0>(a, s);
      return;
    } else {
    const uint64_t rest = a.tab.per_neuron[0] & ~(1ull << M::i_ref);
    bool uni = rest == 0 && a.tab.per_neuron[1] == 0;
    for (int j = 0; j < M::NPAR && uni; ++j)
      if (M::divisor(j) && recip_rn(a.tab.val[j]) == 0.0f) uni = false;
    if constexpr (PredCapable<M>::value) {
      if (uni && a.pred_mode == 1) {
        launch_persistent<M, true, 1>(a, s);
        return;
      }
      if (uni && a.pred_mode == 2) {
        launch_persistent<M, true, 2>(a, s);
        return;
      }
    }
    if (uni)
      launch_persistent<M, true, 0>(a, s);
    else
      launch_persistent<M, false, 0>(a, s);
    return;
    }
  }
  const int grid = (a.n + block - 1) / block;
  hipLaunchKernelGGL(rk5_kernel<M>, dim3(grid), dim3(block), 0, s, a);
}

// Launch for a model templated on its port count, NP = 1..kMaxPort.
template <template <int> class M, int NP = 1>
inline void dispatch_ports(int n_port, const RK5Args& a, hipStream_t s) {
  if constexpr (NP <= kMaxPort) {
    if (n_port == NP) {
      launch_rk5_t<M<NP>>(a, s);
      return;
    }
    dispatch_ports<M, NP + 1>(n_port, a, s);
  } else {
    throw std::runtime_error("RK5: port count " + std::to_string(n_port) + " out of range");
  }
}

// Whether the compile-time input layout of model M (input variable and
// weight parameter of each port) is the fold's layout.
template <class M>
inline bool fold_layout_is(int in_var, int in_stride, int w_param, int w_stride) {
  for (int k = 0; k < M::NPORT; ++k) {
    if (M::in_y(k) != in_var + k * in_stride) return false;
    if (M::in_w(k) != (w_param >= 0 ? w_param + k * w_stride : -1)) return false;
  }
  return true;
}

template <template <int> class M, int NP = 1>
inline bool fold_layout_ports(int n_port, int iv, int is, int wp, int ws) {
  if constexpr (NP <= kMaxPort) {
    if (n_port == NP) return fold_layout_is<M<NP>>(iv, is, wp, ws);
    return fold_layout_ports<M, NP + 1>(n_port, iv, is, wp, ws);
  } else {
    return false;
  }
}

}  // namespace ngpu
