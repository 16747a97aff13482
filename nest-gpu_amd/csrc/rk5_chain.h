// Chain form of the RK5 update: one neuron spread over a group of lanes.
//
// A spiking neuron's step is a serial chain of ~46 dependent attempts, and
// the waves holding such neurons run almost alone on their SIMDs, so the
// launch lasts as long as one chain: a wave issues one instruction at a time
// (4-5 cycles each when independent, 8 when dependent), and what counts is
// the number of instructions from one attempt to the next.  Here a group of
// G = 2, 4 or 8 lanes holds one neuron: the membrane lane (V, w) and one lane
// per receptor port (its conductance or current and the rise variable), so
// the stage sums, the error estimate and the divisions of all variables are
// done side by side in the same instructions.  The membrane lane reads the
// ports' variables with DPP row shifts, the error ratio is the maximum over
// the group by DPP.  Every variable goes through exactly the operations of
// M::deriv, rk5_try and the persistent loop, so results are the same bits.
//
// Bound: the latency of one attempt's dependent instructions, ~2,300 cycles
// from one attempt to the next, 23 of them in a launch.  Measured (MI355X,
// time of a 0.1 ms step, one lane per neuron -> this form): 1e6 AdEx neurons
// with 100 synapses each, 13.9 Hz, 134 -> 66 us; 60,000 with 1,000 synapses
// 120 -> 37.6 us; 1,000 neurons 65 -> 28.9 us; 2,000 with plastic synapses (no
// split steps, so the whole chain in one launch) 105 -> 52.5 us; the
// six-population batch of 50,330 neurons 127 -> 39.7 us.  Of these k1 taken
// beside the error ratio, and the shorter right-hand side (ChainNote below,
// the error ratio by reciprocal), gave 39.6 -> 37.6, 30.6 -> 28.9,
// 55.7 -> 52.5 and 41.1 -> 39.7 us.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"
#include "device_common.h"
#include "kernels.h"
#include "rk5_models.h"

namespace ngpu {

// lanes per neuron: the membrane lane and one per port, a power of two
constexpr int chain_lanes(int n_port) { return n_port < 2 ? 2 : n_port < 4 ? 4 : 8; }

// models and port counts the chain form serves
template <class M>
constexpr bool chain_capable() { return M::kChain && M::NPORT <= 7; }

// v of the lane k places up (within the group's row of 16 lanes)
__device__ inline float chain_from(float v, int k) {
  int x = __float_as_int(v);
  switch (k) {
    case 1: x = __builtin_amdgcn_update_dpp(0, x, 0x101, 0xf, 0xf, true); break;
    case 2: x = __builtin_amdgcn_update_dpp(0, x, 0x102, 0xf, 0xf, true); break;
    case 3: x = __builtin_amdgcn_update_dpp(0, x, 0x103, 0xf, 0xf, true); break;
    case 4: x = __builtin_amdgcn_update_dpp(0, x, 0x104, 0xf, 0xf, true); break;
    case 5: x = __builtin_amdgcn_update_dpp(0, x, 0x105, 0xf, 0xf, true); break;
    case 6: x = __builtin_amdgcn_update_dpp(0, x, 0x106, 0xf, 0xf, true); break;
    case 7: x = __builtin_amdgcn_update_dpp(0, x, 0x107, 0xf, 0xf, true); break;
    default: break;
  }
  return __int_as_float(x);
}

// maximum over the group of a value >= 0 and not NaN (so its bits order as
// integers): quad permutations xor 1 and xor 2, then the half-row mirror
template <int G>
__device__ inline float chain_max(float v) {
  unsigned int u = __float_as_uint(v);
  u = max(u, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)u, 0xB1, 0xf, 0xf, true));
  if constexpr (G >= 4)
    u = max(u, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)u, 0x4E, 0xf, 0xf, true));
  if constexpr (G >= 8)
    u = max(u, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)u, 0x141, 0xf, 0xf, true));
  return __uint_as_float(u);
}

// the divisors of a lane: of its variables a and b, and of the membrane
// lane's inner division (x), with their double reciprocals
struct ChainDiv {
  float da, db, dx;
  double ra, rb, rx;
};

struct ChainNV {
  static constexpr int NV = 2;   // variables per lane, as rk5_try counts them
};

// What a lane's fast divisions and exponentials met that needs the IEEE form:
// the smallest subnormal quotient (div_recip) and the largest exponent.
struct ChainNote {
  unsigned int tiny;
  float big;
  __device__ bool set() const { return tiny_noted(tiny) | !(big <= kExpNear); }
};

// d(a, b)/dt of the lane's variables.  FAST, on an attempt's serial path:
// divisions by reciprocal; the potential's clamp as one median of three (a
// NaN becomes -inf, which is noted); the exponential without its clamps, whose
// argument is noted where these act beyond kExpNear (a subnormal argument
// needs no note: exp is 1 either way); signs and the refractory zero as one
// fma with the lane's sign and addend (1, -0: exact).  Else the IEEE form.
template <class M, bool FAST>
__device__ inline void chain_rhs(const float* y, float* dy, const float* p, const ChainDiv& d,
                                 bool mem, ChainNote& note) {
  constexpr bool kB = M::c_yb(0) >= 0;   // the ports have a rise variable
  auto quot = [&](float x, double r, float den) {
    if constexpr (FAST) {
      return div_recip(x, r, note.tiny);
    } else {
      return x / den;
    }
  };
  const bool refr = p[M::i_ref] > 0.0f;
  struct {
    const ChainDiv& d;
    ChainNote& note;
    float lo, hi;
    __device__ float v(const float* q, float V) const {
      if constexpr (FAST) return __builtin_amdgcn_fmed3f(V, lo, hi);
      return adex_v(q, V);
    }
    __device__ float expx(float x) const {
      if constexpr (!FAST) return exp_fma(x / d.dx);
      const float q = (float)((double)x * d.rx);
      note.big = fmaxf(note.big, fabsf(q));
      return exp_fma_near(q);
    }
  } fx{d, note, refr ? p[M::i_reset] : -__builtin_inff(), refr ? p[M::i_reset] : p[M::i_thr]};
  float nv, nw;
  M::c_mem(p, y[0], y[1], [&](int k) { return chain_from(y[0], k + 1); }, fx, &nv, &nw);
  float qb = 0.0f;
  if constexpr (kB || M::c_mw >= 0) qb = quot(M::c_mw >= 0 && mem ? nw : y[1], d.rb, d.db);
  dy[1] = mem ? (M::c_mw >= 0 ? qb : nw) : kB ? -qb : 0.0f;
  if constexpr (FAST && M::c_mv >= 0) {
    const bool move = mem && !refr;
    const float ya = mem && refr ? 0.0f : y[0];
    const float add = mem ? (refr ? 0.0f : -0.0f) : kB ? y[1] : -0.0f;
    dy[0] = fmaf(mem ? 1.0f : -1.0f, quot(move ? nv : ya, d.ra, d.da), add);
  } else {
    const float qa = quot(M::c_mv >= 0 && mem ? nv : y[0], d.ra, d.da);
    dy[0] = mem ? (refr ? 0.0f : (M::c_mv >= 0 ? qa : nv)) : kB ? y[1] - qa : -qa;
  }
}

}  // namespace ngpu
