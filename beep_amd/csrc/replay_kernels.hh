// State::initialise_from_particle (src/state.cc:294-322) for a trajectory of
// transition counts: the populations of every step are prefix sums of the
// counts, and given them each step's means depend on nothing else, so the steps
// are computed side by side instead of one after the other (one instance of
// 400 cells x 8 transitions x 200 steps: 376 us step by step, 56 + 11 us here).  The FP32 expressions
// are the simulation kernels', with the same roundings.  For models without
// strains on the fused path; strains (populations pooled step by step) and the
// step-wise path replay through their simulation kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fused_common.hh"

namespace beepdev {

// Populations at the start of every step, pop[s][c][cell], and the current
// state, from the counts tn[s][tr][cell].  One thread per (compartment, cell),
// the counts of BEEP_REPLAY_AHEAD steps loaded together: what bounds it is the
// chain of loads over the steps, (steps / AHEAD) memory latencies.
#define BEEP_REPLAY_AHEAD 16
__global__ void __launch_bounds__(64) k_replay_pops(const TopoDev* __restrict__ topo, const int* __restrict__ tn,
                                                    int* __restrict__ pop, int* __restrict__ state) {
  ctopo* tp = (ctopo*)topo;
  const int AG = tp->AG, T = tp->T, C = tp->C, S = tp->S;
  const int cell = blockIdx.x * 64 + threadIdx.x, c = blockIdx.y;
  if (cell >= AG) return;
  const size_t TAG = (size_t)T * AG, CAG = (size_t)C * AG;
  gcint* n = gptr(tn) + cell;
  int v = gptr(tp->pop_init)[c * AG + cell];
  gint* out = (gint*)pop + (size_t)c * AG + cell;
  for (int s0 = 0; s0 < S; s0 += BEEP_REPLAY_AHEAD) {
    const int ns = min(BEEP_REPLAY_AHEAD, S - s0);
    int d[BEEP_REPLAY_AHEAD];
#pragma unroll
    for (int k = 0; k < BEEP_REPLAY_AHEAD; k++) d[k] = 0;
    for (int tr = 0; tr < T; tr++) {
      const int sign = (gptr(tp->to)[tr] == c) - (gptr(tp->from)[tr] == c);
      if (sign == 0) continue;
#pragma unroll
      for (int k = 0; k < BEEP_REPLAY_AHEAD; k++)
        d[k] += sign * n[(size_t)(s0 + min(k, ns - 1)) * TAG + (size_t)tr * AG];
    }
#pragma unroll
    for (int k = 0; k < BEEP_REPLAY_AHEAD; k++)
      if (k < ns) {
        out[(size_t)(s0 + k) * CAG] = v;
        if (s0 + k < S - 1) v += d[k];       // the last step is not applied (src/state.cc:634)
      }
  }
  ((gint*)state)[c * AG + cell] = v;
}

// The means of step blockIdx.x: infectivity of every cell, area mixing, age
// mixing, transition means.  One workgroup per step; LDS: infectivity and mixed
// infectivity, 2 AG floats.
__global__ void __launch_bounds__(512) k_replay_means(const TopoDev* __restrict__ topo, const float* __restrict__ tab_,
                                                      const int* __restrict__ pop, float* __restrict__ tm,
                                                      int* __restrict__ err) {
  extern __shared__ float rsm[];
  ctopo* tp = (ctopo*)topo;
  const int A = tp->A, G = tp->G, C = tp->C, T = tp->T, AG = tp->AG, s = blockIdx.x;
  const int tid = threadIdx.x, nt = blockDim.x;
  float* sdinf = rsm;
  float* sI = rsm + AG;
  gcfloat* tab = gptr(tab_);
  gcint* p = gptr(pop) + (size_t)s * C * AG;
  for (int cell = tid; cell < AG; cell += nt) {
    float d = 0.f;
    for (int c = 0; c < C; c++) {
      const float w = tab[tp->off_inf + c];
      if (w != 0.f) d = __builtin_fmaf(w, (float)p[c * AG + cell], d);
    }
    sdinf[cell] = d;
  }
  __syncthreads();
  mix_cells(gptr(tp->diag), gptr(tp->fac), gptr(tp->in_ptr), gptr(tp->in_src), gptr(tp->in_w), gptr(tp->mix_order), sdinf,
            sI, tab[tp->off_geo + s], G, AG, tid, nt);
  __syncthreads();
  const size_t offN = tp->off_N + (tp->N_tv ? (size_t)s * G * G : 0);
  gcfloat* af_s = af_row(tp, tab, s);
  gfloat* tm_s = tm ? (gfloat*)tm + (size_t)s * T * AG : nullptr;
  const float dt = tp->dt;
  int bad = 0;
  for (int cell = tid; cell < AG; cell += nt) {
    const int j = cell / G, g = cell - j * G;
    float nmi = 0.f;
    for (int gg = 0; gg < G; gg++) nmi = __builtin_fmaf(tab[offN + g * G + gg], sI[j * G + gg], nmi);
    if (nmi < 0.f) nmi = 0.f;
    float bet, ef, agc;
    foi_groups(tp, tab, s, j, g, G, bet, ef, agc);
    float afc = af_s[j];
    mod_foi_factors(tp, s, cell, afc, agc);
    const float foi = foi_mean(bet, afc, nmi, ef, agc);
    for (int tr = 0; tr < T; tr++) {
      const float popu = (float)p[gptr(tp->from)[tr] * AG + cell];
      float lp = 0.f;
      if (popu > 0.f)
        lp = tr == tp->inf_tr ? dt * popu * tab[tp->off_sus + g] * foi : dt * popu * tab[tp->off_rate + tr * G + g];
      lp = mod_mean(tp, s, tr, cell, lp);
      if (lp != lp) { bad |= 1; lp = 0.f; }
      else if (lp > 1e9f) { bad |= 2; lp = 0.f; }
      if (tm_s) tm_s[tr * AG + cell] = lp;
    }
  }
  if (bad) atomicOr(err, bad);
}

}  // namespace beepdev
