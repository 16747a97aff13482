// Philox4x32-10 (Salmon et al., SC'11) and the Poisson sampler used for
// poisson_generator input, usable on host and device.
//
// The reference draws Poisson counts with cuRAND (src/poiss_gen.cu:74);
// this build uses the published Philox construction with a Knuth
// multiplication sampler (TAOCP 3.4.1) evaluated as a chain of IEEE double
// products, so every draw is reproducible bit for bit off the GPU.
//   stream  = index of the connection in the source-major connection table
//   counter = {block, t_idx lo, t_idx hi, stream}, key = 64-bit kernel seed
// The mean is split in `chunks` equal parts with threshold exp(-lambda/chunks)
// computed on the host, keeping the products inside the double range.
#pragma once
#include <cstdint>

#ifndef __HIPCC__
#define NGPU_HD
#else
#define NGPU_HD __host__ __device__
#endif

namespace ngpu {

struct U32x4 { uint32_t x, y, z, w; };

NGPU_HD inline U32x4 philox4x32_10(U32x4 c, uint32_t k0, uint32_t k1) {
#ifdef __clang__
#pragma unroll
#endif
  for (int r = 0; r < 10; ++r) {
    uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    U32x4 n;
    n.x = (uint32_t)(p1 >> 32) ^ c.y ^ k0;
    n.y = (uint32_t)p1;
    n.z = (uint32_t)(p0 >> 32) ^ c.w ^ k1;
    n.w = (uint32_t)p0;
    c = n;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

NGPU_HD inline uint32_t pick(const U32x4& r, int i) {
  return i == 0 ? r.x : (i == 1 ? r.y : (i == 2 ? r.z : r.w));
}

// Chunk count for a Poisson mean (16 per chunk).
inline int poisson_chunks_host(double lambda) {
  if (!(lambda > 0.0)) return 0;
  int m = (int)(lambda / 16.0);
  if ((double)m * 16.0 < lambda) ++m;
  return m;
}

NGPU_HD inline int poisson_draw(uint64_t seed, uint32_t stream, long long t_idx,
                                int chunks, double exp_chunk) {
  if (chunks <= 0) return 0;
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  U32x4 ctr{0u, (uint32_t)(uint64_t)t_idx, (uint32_t)((uint64_t)t_idx >> 32), stream};
  U32x4 r = philox4x32_10(ctr, k0, k1);
  int used = 0, n = 0;
  for (int c = 0; c < chunks; ++c) {
    double p = 1.0;
    for (;;) {
      if (used == 4) {
        ctr.x += 1u;
        r = philox4x32_10(ctr, k0, k1);
        used = 0;
      }
      double u = ((double)pick(r, used++) + 0.5) * (1.0 / 4294967296.0);
      p *= u;
      if (p <= exp_chunk) break;
      ++n;
    }
  }
  return n;
}

#ifdef __HIPCC__
// poisson_draw for all lanes of a wave together (lanes of a partly masked wave
// too), the same counts.  With one chunk the count is the number of prefix
// products that stay above the threshold (they only fall), so the uniforms of
// a Philox block are taken without a branch: four multiplications, four
// comparisons.  Blocks are wave-uniform, so the first rounds' products of the
// counter's uniform words are scalar, and a wave goes on to the next block
// while any lane is above its threshold (a mean of 2, 20 kHz at 0.1 ms: two
// blocks).  The per-lane loop it replaces ran 7-9 rounds with ever fewer
// lanes on, ~20 instructions each, and two to three Philox calls.
// kRekey: the key schedule is computed at each block, by the scalar unit.
// For the RK5 kernels, where it would be hoisted out of the refill loop: its
// 20 keys and first products then hold the scalar registers, and spilling
// others costs more vector instructions than the schedule (1e6 AdEx neurons,
// 67.3 -> 66.0 us a step together with the refill's single round trip).  The
// iaf_psc_exp kernels have the registers (re-keyed, 77,169 neurons: 15.7 ->
// 16.0 us).
template <bool kRekey = false>
__device__ inline int poisson_draw_wave(uint64_t seed, uint32_t stream, long long t_idx, int chunks,
                                        double exp_chunk) {
  if (__any(chunks > 1)) return poisson_draw(seed, stream, t_idx, chunks, exp_chunk);
  auto word = [](uint64_t v) {
    if constexpr (kRekey) return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    return (uint32_t)v;
  };
  uint32_t k0 = word(seed), k1 = word(seed >> 32);
  uint32_t t_lo = word((uint64_t)t_idx), t_hi = word((uint64_t)t_idx >> 32);
  double p = chunks > 0 ? 1.0 : 0.0;
  const double e = chunks > 0 ? exp_chunk : 1.0;
  int n = 0;
  for (uint32_t blk = 0; __any(p > e); ++blk) {
    if constexpr (kRekey) asm volatile("" : "+s"(k0), "+s"(k1), "+s"(t_lo), "+s"(t_hi));
    const U32x4 r = philox4x32_10(U32x4{blk, t_lo, t_hi, stream}, k0, k1);
    // ((double)r + 0.5) 2^-32, exact
    p *= fma((double)r.x, 0x1p-32, 0x1p-33);
    n += p > e;
    p *= fma((double)r.y, 0x1p-32, 0x1p-33);
    n += p > e;
    p *= fma((double)r.z, 0x1p-32, 0x1p-33);
    n += p > e;
    p *= fma((double)r.w, 0x1p-32, 0x1p-33);
    n += p > e;
  }
  return n;
}
#endif

}  // namespace ngpu
