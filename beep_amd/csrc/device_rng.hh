// Counter-based random numbers and the Poisson / binomial samplers used by
// the tau-leap kernels.
//
// Streams.  Every draw is a pure function of
//   (seed, stream, instance key, step, cell = area*G + dp, transition order)
// so a trajectory is the same whichever batch, slot or launch shape computes
// it.  Philox-4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers:
// as easy as 1, 2, 3", SC'11) maps a 128-bit counter and 64-bit key to 128
// random bits:
//   key     = seed
//   counter = (step | stream << 16, cell, block, instance key)
// The uniforms of one (step, cell) form a pool read in order by the draws of
// its transitions, taken in transition order; block counts the 4-word Philox
// blocks the pool has used.
//
// Samplers (the reference draws with libstdc++ std::poisson_distribution and
// std::binomial_distribution, src/utils.cc:148-180; the device draws the same
// distributions with these published methods):
//   Poisson, mean < 10:  sequential-search inversion of the CDF;
//   Poisson, mean >= 10: PTRS, transformed rejection with squeeze
//                        (W. Hormann, "The transformed rejection method for
//                        generating Poisson random variables", Insurance:
//                        Mathematics and Economics 12 (1993) 39-45);
//   binomial, n*min(p,1-p) < 10: inversion (BINV, Kachitvichyanukul &
//                        Schmeiser, CACM 31 (1988) 216-222);
//   binomial otherwise:  BTRD (W. Hormann, "The generation of binomial random
//                        variates", J. Statist. Comput. Simul. 46 (1993) 101-110).
// All arithmetic is FP32: the rejection tests use C. Loader's saddle-point
// log-pmf, candidates are formed as floor(mean) + floor(frac(mean) + x) so they
// are exact integers, means of 2^23 and above are drawn as sums of Poisson
// variates (superposition) and binomials of 2^23 trials and above as sums of
// binomials over chunks of the trials, both exact in distribution.
#pragma once
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#include <stdint.h>
#else
// Run-time compilation provides the fixed-width types in its own namespace.
typedef __hip_internal::uint8_t uint8_t;
typedef __hip_internal::uint16_t uint16_t;
typedef __hip_internal::uint32_t uint32_t;
typedef __hip_internal::uint64_t uint64_t;
#endif

namespace beepdev {

struct u4 { uint32_t x, y, z, w; };

__device__ __host__ inline uint32_t mulhi32(uint32_t a, uint32_t b) {
  return (uint32_t)(((uint64_t)a * (uint64_t)b) >> 32);
}

// 16 to 20 quarter-rate 32x32->64 products per block; the two exclusive ors of
// a word are one three-input v_bitop3_b32 (20 instructions fewer per block:
// spatial simulation kernel 14.35 -> 13.65 ms).
__device__ inline u4 philox4x32_10(u4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int i = 0; i < 10; i++) {
    // One 32x32->64 product gives both halves (v_mad_u64_u32).
    uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    u4 o;
    o.x = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c.y, k0, 0x96);
    o.y = (uint32_t)p1;
    o.z = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c.w, k1, 0x96);
    o.w = (uint32_t)p0;
    c = o;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

// Uniform on the open interval (0,1) from 32 random bits, FP64.
__device__ inline double u01d(uint32_t x) { return ((double)x + 0.5) * 2.3283064365386963e-10; }
// Uniform on (0,1) from the top 24 bits, FP32.
__device__ inline float u01f(uint32_t x) { return ((float)(x >> 8) + 0.5f) * 5.9604644775390625e-08f; }

// The uniform pool of one (step, cell).
struct CellRng {
  uint32_t k0, k1, c0, c1, c3;
  uint32_t block;
  int idx;
  u4 buf;
  __device__ inline void init(uint32_t kk0, uint32_t kk1, uint32_t cc0, uint32_t cc1, uint32_t cc3) {
    k0 = kk0; k1 = kk1; c0 = cc0; c1 = cc1; c3 = cc3; block = 0; idx = 4;
  }
  __device__ inline uint32_t bits() {
    if (idx >= 4) {
      buf = philox4x32_10(u4{c0, c1, block, c3}, k0, k1);
      block++;
      idx = 0;
    }
    // The block is consumed from .x and shifted down: no per-lane index into
    // it, which the compiler would otherwise lower to a stack array.
    uint32_t x = buf.x;
    buf.x = buf.y; buf.y = buf.z; buf.z = buf.w;
    idx++;
    return x;
  }
  __device__ inline float next() { return u01f(bits()); }
  // Fills the first block now (the same block the first bits() would make):
  // where the lanes of a wavefront make their first draw at different places
  // of an unrolled loop, this runs the generator once, converged.
  __device__ inline void prime() {
    buf = philox4x32_10(u4{c0, c1, block, c3}, k0, k1);
    block++;
    idx = 0;
  }
};
typedef CellRng ExtraUniforms;

#define BEEP_MAX_EXTRA_BLOCKS 4096u

// Blocks a pool has used: the low 22 bits of its block word.  A cell-step's
// pool counts from 0; a large draw's own stream from 0x80000000 | tr << 22
// (draw_item_body), so the transition bits above must not count.  The
// rejection loops stop at BEEP_MAX_EXTRA_BLOCKS blocks (a bound on the loop,
// reached with probability far below 1e-100).
__device__ inline uint32_t blocks_used(const CellRng& r) { return r.block & 0x3FFFFFu; }

// ---- log-pmf pieces in FP32 (C. Loader, "Fast and accurate computation of
// binomial probabilities", 2000): log n! = (n+1/2) log n - n + log(2 pi)/2 +
// stirlerr(n), and bd0(x, m) = x log(x/m) + m - x evaluated without
// cancellation, so log Pois(k; m) = -log(2 pi k)/2 - stirlerr(k) - bd0(k, m).

__device__ inline float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

// stirlerr(0..16) from lgamma (entry 0 unused).
__constant__ float kStirlerr[17] = {0.0f, 8.106146680e-02f, 4.134069596e-02f, 2.767792568e-02f, 2.079067210e-02f,
                                    1.664469119e-02f, 1.387612882e-02f, 1.189670995e-02f, 1.041126526e-02f,
                                    9.255462183e-03f, 8.330563433e-03f, 7.573675488e-03f, 6.942840107e-03f,
                                    6.408994188e-03f, 5.951370113e-03f, 5.554733552e-03f, 5.207655920e-03f};

__device__ inline float stirlerr_f(float n) {
  // The table below 17, the asymptotic series above.
  if (n <= 16.f) return kStirlerr[(int)n];
  const float S0 = 1.f / 12.f, S1 = 1.f / 360.f, S2 = 1.f / 1260.f, S3 = 1.f / 1680.f;
  float in = __builtin_amdgcn_rcpf(n), inn = in * in;
  if (n > 80.f) return (S0 - (S1 - S2 * inn) * inn) * in;
  return (S0 - (S1 - (S2 - S3 * inn) * inn) * inn) * in;
}

__device__ inline float bd0_f(float x, float m) {
  float d = x - m;
  if (fabsf(d) < 0.1f * (x + m)) {
    // 2 x sum_{j>=1} v^(2j+1)/(2j+1) with v = d/(x+m): |v| < 0.1, so 8 terms
    // reach FP32 precision.
    const float inv_odd[9] = {0.f, 1.f / 3.f, 1.f / 5.f, 1.f / 7.f, 1.f / 9.f, 1.f / 11.f, 1.f / 13.f, 1.f / 15.f,
                              1.f / 17.f};
    float v = fdiv(d, x + m);
    float s = d * v;
    float ej = 2.f * x * v;
    v = v * v;
#pragma unroll
    for (int j = 1; j < 9; j++) {
      ej *= v;
      s += ej * inv_odd[j];
    }
    return s;
  }
  return x * logf(x / m) + m - x;
}

// log Pois(k; lam), k >= 1.
__device__ inline float log_pois_f(float k, float lam) {
  return -0.5f * __logf(6.2831853071795865f * k) - stirlerr_f(k) - bd0_f(k, lam);
}

// Whether any active lane of the wavefront holds c.
__device__ inline bool wave_any(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0; }

// Where the running sum of the inversion search first stops growing (or 64):
// the search's result when FP32 rounding leaves u above that sum, a tail event
// of probability ~1e-7, hence one compact loop.  1 / k up to 16 is the
// correctly rounded reciprocal: a Newton step from any value within one ulp
// of 1 / k gives it for these k.
__device__ inline int poisson_stall(float lam, float p) {
  float F = p;
  int k = 0;
#pragma unroll 1
  while (k < 64) {
    k++;
    float r = __builtin_amdgcn_rcpf((float)k);
    if (k <= 16) r = __builtin_fmaf(__builtin_fmaf(-(float)k, r, 1.f), r, r);
    const float l = lam * r, Fn = __builtin_fmaf(l, p, F);
    p *= l;
    if (Fn == F) return k;
    F = Fn;
  }
  return k;
}

// One term of the search: F_k = F_{k-1} + p_k with p_k = p_{k-1} lam / k.
#define BEEP_INV_TERM(K)                           \
  {                                                \
    const float l = lam * (1.0f / (K));            \
    F = __builtin_fmaf(l, p, F);                   \
    p = l * p;                                     \
    k += u > F;                                    \
  }
#define BEEP_INV_BLOCK(K0) BEEP_INV_TERM(K0 + 1) BEEP_INV_TERM(K0 + 2) BEEP_INV_TERM(K0 + 3) BEEP_INV_TERM(K0 + 4)

// Poisson(lam) with first uniform u (FP32, lam < 10): sequential inversion,
// the first k at which the CDF F_k reaches u or stops growing.
//
// The F_k of a lane never fall, so k is the number of them below u: a compare
// and an add with carry per term, with no lane masked off, and the wavefront
// goes on, four terms at a time, while any lane's u is above its sum (a lane
// that is done counts nothing more).  Below mean 10 a sum that has stopped
// growing never grows again, so u at or below the last sum was reached before
// any stop; a lane still above its sum at the end has stopped
// (poisson_stall).  Terms 1-16 have their reciprocals as constants.
// The search with its first-of-four selection and masked exits cost 32
// instructions per block of four terms and lane-mask work between blocks, this
// one 20: spatial simulation of 4096 x 400 cells x 200 steps 15.8 -> 14.35 ms.
__device__ inline int poisson_inversion(float lam, float u) {
  const float p0 = __expf(-lam);
  float p = p0, F = p0;
  int k = u > F;
  if (!wave_any(u > F)) return k;
  BEEP_INV_BLOCK(0)
  if (wave_any(u > F)) {
    BEEP_INV_BLOCK(4)
    if (wave_any(u > F)) {
      BEEP_INV_BLOCK(8)
      if (wave_any(u > F)) {
        BEEP_INV_BLOCK(12)
        float Fp = -1.f;
        for (int t = 17; t <= 64 && wave_any(u > F && F != Fp); t++) {
          const float l = lam * __builtin_amdgcn_rcpf((float)t);
          Fp = F;
          F = __builtin_fmaf(l, p, F);
          p *= l;
          k += u > F;
        }
        if (u > F) k = poisson_stall(lam, p0);
      }
    }
  }
  return k;
}
#undef BEEP_INV_BLOCK
#undef BEEP_INV_TERM

// PTRS (Hormann 1993) for 10 <= lam < 2^23: the squeeze accepts most
// candidates; the exact test compares with the saddle-point log-pmf.
__device__ inline int poisson_ptrs(float lam, float ufirst, ExtraUniforms& r) {
  const float slam = __builtin_amdgcn_sqrtf(lam);
  const float b = 0.931f + 2.53f * slam;
  const float a = -0.059f + 0.02483f * b;
  const float vr = 0.9277f - fdiv(3.6224f, b - 2.f);
  const float lfl = floorf(lam), lfr = lam - lfl;
  float Uraw = ufirst;
  for (;;) {
    float U = Uraw - 0.5f;
    float V = r.next();
    float us = 0.5f - fabsf(U);
    float k = lfl + floorf((fdiv(2.f * a, us) + b) * U + (lfr + 0.43f));
    if (us >= 0.07f && V <= vr) return (int)k;
    if (!(k < 0.f || (us < 0.013f && V > us))) {
      float lhs = __logf(V * (1.1239f + fdiv(1.1328f, b - 3.4f))) - __logf(fdiv(a, us * us) + b);
      float rhs = k == 0.f ? -lam : log_pois_f(k, lam);
      if (lhs <= rhs) return (int)k;
    }
    if (blocks_used(r) >= BEEP_MAX_EXTRA_BLOCKS) return (int)lfl;   // unreachable in practice
    Uraw = r.next();
  }
}

#define BEEP_SPLIT (8388608.0f)   // 2^23

__device__ inline int poisson_draw(float lam, float ufirst, ExtraUniforms& r) {
  if (lam < 10.0f) return poisson_inversion(lam, ufirst);
  if (lam < BEEP_SPLIT) return poisson_ptrs(lam, ufirst, r);
  // Superposition: Pois(lam) = sum of m independent Pois(lam / m).
  int m = (int)ceilf(lam / BEEP_SPLIT);
  float part = lam / (float)m;
  int n = 0;
  for (int i = 0; i < m; i++) n += poisson_ptrs(part, i == 0 ? ufirst : r.next(), r);
  return n;
}

// Inversion from k = 0 (BINV), FP32, for n * p < 10 with p <= 1/2: u loses the
// masses r_0, r_1, ... until it is at or below the next one; k counts the
// masses passed.  The wavefront steps through k together, four masses to a
// branch, with no lane masked off: a search that is over (u <= r) stays over,
// since u - r <= 0 and the next mass, clamped at 0, is no smaller.  A search
// that passes more than n masses (or 110) has run out of mass by rounding, or
// far into the tail, and draws again.  The clamp does not touch a search in
// progress: r_k / r_(k-1) = a / k - s is positive up to k = n.  A search lane
// by lane took a branch per mass; coupled proposals of 24 instances with 30%
// masks went from 1990 to 1815 us (kernel), uneven batches from 11.75 to 10.95 ms.
__device__ inline int binomial_inversion(int n, float p, float ufirst, ExtraUniforms& r) {
  const float q = 1.f - p, s = fdiv(p, q), a = (float)(n + 1) * s;
  const float r0 = __expf((float)n * log1pf(-p));
  const int last = n < 110 ? n : 110;
  float u = ufirst;
  for (;;) {
    float rr = r0;
    int k = u > rr;
    for (int t = 1; t <= 111 && wave_any(u > rr && k <= last); t += 4) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float x = fmaxf(__builtin_fmaf(a, __builtin_amdgcn_rcpf((float)(t + j)), -s), 0.f);
        u -= rr;
        rr *= x;
        asm("" : "+v"(rr));        // rounded: the next u - rr is no fused u - rr * x
        k += u > rr;
      }
    }
    if (k <= last) return k;
    if (blocks_used(r) >= BEEP_MAX_EXTRA_BLOCKS) return (int)floorf(n * p);   // unreachable in practice
    u = (float)r.next();
  }
}

// BTRD (Hormann 1993) in FP32 for n * p >= 10, p <= 1/2, n < 2^24;
// fc(k) = stirlerr(k + 1).
__device__ inline int binomial_btrd(int n, float p, float ufirst, ExtraUniforms& r) {
  const float q = 1.f - p;
  const float nf = (float)n;
  const float m = floorf((nf + 1.f) * p);
  const float rr = fdiv(p, q), nr = (nf + 1.f) * rr, npq = nf * p * q;
  const float snpq = __builtin_amdgcn_sqrtf(npq);
  const float b = 1.15f + 2.53f * snpq;
  const float a = -0.0873f + 0.0248f * b + 0.01f * p;
  const float c = nf * p + 0.5f;
  const float alpha = (2.83f + fdiv(5.1f, b)) * snpq;
  const float vr = 0.92f - fdiv(4.2f, b);
  const float urvr = 0.86f * vr;
  float v = ufirst;
  for (;;) {
    float u;
    if (v <= urvr) {
      u = fdiv(v, vr) - 0.43f;
      return (int)floorf((fdiv(2.f * a, 0.5f - fabsf(u)) + b) * u + c);
    }
    if (v >= vr) {
      u = (float)r.next() - 0.5f;
    } else {
      u = fdiv(v, vr) - 0.93f;
      u = (u < 0.f ? -0.5f : 0.5f) - u;
      v = (float)r.next() * vr;
    }
    float us = 0.5f - fabsf(u);
    float k = floorf((fdiv(2.f * a, us) + b) * u + c);
    bool accept = false;
    if (k >= 0.f && k <= nf) {
      v = v * fdiv(alpha, fdiv(a, us * us) + b);
      float km = fabsf(k - m);
      if (km <= 15.f) {
        float f = 1.f;
        if (m < k) {
          for (float i = m + 1.f; i <= k; i += 1.f) f *= (fdiv(nr, i) - rr);
        } else if (m > k) {
          for (float i = k + 1.f; i <= m; i += 1.f) v *= (fdiv(nr, i) - rr);
        }
        accept = (v <= f);
      } else {
        float lv = __logf(v);
        float inpq = __builtin_amdgcn_rcpf(npq);
        float rho = (km * inpq) * (((km * (1.f / 3.f) + 0.625f) * km + 1.f / 6.f) * inpq + 0.5f);
        float t = -km * km * 0.5f * inpq;
        if (lv < t - rho) accept = true;
        else if (lv <= t + rho) {
          float nm = nf - m + 1.f;
          float h = (m + 0.5f) * logf((m + 1.f) / (rr * nm)) + stirlerr_f(m + 1.f) + stirlerr_f(nf - m + 1.f);
          float nk = nf - k + 1.f;
          accept = lv <= h + (nf + 1.f) * logf(nm / nk) + (k + 0.5f) * logf(nk * rr / (k + 1.f)) -
                             stirlerr_f(k + 1.f) - stirlerr_f(nf - k + 1.f);
        }
      }
    }
    if (accept) return (int)k;
    if (blocks_used(r) >= BEEP_MAX_EXTRA_BLOCKS) return (int)floorf(n * p);   // unreachable in practice
    v = (float)r.next();
  }
}

__device__ inline int binomial_chunk(int n, float p, float ufirst, ExtraUniforms& r) {
  if ((float)n * p < 10.f) return binomial_inversion(n, p, ufirst, r);
  return binomial_btrd(n, p, ufirst, r);
}

// Binomial(n, p) for 0 < p < 1.
__device__ inline int binomial_draw(int n, float p, float ufirst, ExtraUniforms& r) {
  if (n <= 0) return 0;
  bool flip = p > 0.5f;
  float pp = flip ? 1.f - p : p;
  int k = 0;
  const int chunk = 1 << 23;
  int left = n;
  bool first = true;
  while (left > 0) {          // Bin(n, p) = sum of Bin(chunk, p) over chunks of the trials
    int c = left < chunk ? left : chunk;
    k += binomial_chunk(c, pp, first ? ufirst : r.next(), r);
    first = false;
    left -= c;
  }
  return flip ? n - k : k;
}

// binomial_draw where n * min(p, 1 - p) < 10 is known: every chunk then takes
// the inversion branch, so this is the same function of (n, p, uniforms)
// without the BTRD code, for call sites inlined in the transition loop.
__device__ inline int binomial_draw_small(int n, float p, float ufirst, ExtraUniforms& r) {
  if (n <= 0) return 0;
  bool flip = p > 0.5f;
  float pp = flip ? 1.f - p : p;
  int k = 0;
  const int chunk = 1 << 23;
  int left = n;
  bool first = true;
  while (left > 0) {
    int c = left < chunk ? left : chunk;
    k += binomial_inversion(c, pp, first ? ufirst : r.next(), r);
    first = false;
    left -= c;
  }
  return flip ? n - k : k;
}

}  // namespace beepdev
