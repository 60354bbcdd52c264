// Structure-specialised transition kernel of the step-wise path, compiled at
// run time together with fused_spec.hh (same prelude: namespace beepspec).
// It computes exactly what k_step_trans (step_kernels.hh) computes -- same
// FP32 expressions and order, same uniforms in the same order.  As in the fused
// kernel: all means first without a branch, kept arrays written through slabs,
// one queue reservation per wavefront for the draws made cooperatively, and
// the populations, at compile-time indices, in LDS only while those draws land.
// Populations pass from step to step through the kept trajectory, which a step
// would write anyway; the state is written by the run's last step alone.
//
// Bound by instruction issue (about 1,330 vector instructions per wavefront, 73%
// of the vector cycles) next to 240 MB of traffic a step for 512 instances x
// 2,853 cells: 74 us in the median step of an epidemic (79 on average, 119 at its
// height), where the copy rate would take 50.  Reading and writing the state each
// step and reserving per transition took 13 us more.
#pragma once

namespace beepdev {

template <int MODE>
__device__ inline void step_spec_body(const Job* __restrict__ jobs, const float* __restrict__ Ibuf,
                                      float* __restrict__ D, int Apad, int s, const uint64_t* __restrict__ rngp) {
  using namespace beepspec;
  const uint64_t seed = rngp[0];
  const uint32_t stream = (uint32_t)rngp[1];
  const int b = blockIdx.x;
  const Job jb = jobs[b];
  ctopo* __restrict__ tp = (ctopo*)jb.topo;
  const int A = tp->A, S = tp->S, AG = tp->AG;
  const float dt = tp->dt;
  const int tid = threadIdx.x;
  const int cell = blockIdx.y * BEEP_STEP_BLOCK + tid;
  const bool valid = cell < AG && s >= jb.t0 && s < jb.t1;

  __shared__ int spop[CP][BEEP_STEP_BLOCK];          // populations after the step's own-lane draws
  __shared__ uint16_t qcode[T * BEEP_STEP_BLOCK];          // cell of the workgroup * T + transition, T <= 64
  __shared__ float qval[T * BEEP_STEP_BLOCK];
  __shared__ int qcount;
  __shared__ float srate[T * G], sN[G * G], ssus[G], sinf[C];
  gcfloat* tab = gptr(jb.tab);
  for (int i = tid; i < T * G; i += BEEP_STEP_BLOCK) srate[i] = tab[tp->off_rate + i];
  const size_t offN = tp->off_N + (N_TV ? (size_t)s * G * G : 0);   // a time-varying age matrix: step s's
  for (int i = tid; i < G * G; i += BEEP_STEP_BLOCK) sN[i] = tab[offN + i];
  for (int i = tid; i < G; i += BEEP_STEP_BLOCK) ssus[i] = tab[tp->off_sus + i];
  for (int i = tid; i < C; i += BEEP_STEP_BLOCK) sinf[i] = tab[tp->off_inf + i];
  if (tid == 0) qcount = 0;
  __syncthreads();

  const uint32_t TAG = (uint32_t)(T * AG), CAG = (uint32_t)(C * AG);
  gcint* itn = MODE == MODE_MBP ? gptr(jb.init_tn) + (size_t)s * TAG : nullptr;
  gcfloat* itm = MODE == MODE_MBP ? gptr(jb.init_tm) + (size_t)s * TAG : nullptr;
  gcint* tn_r = MODE == MODE_REPLAY ? gptr(jb.tn) + (size_t)s * TAG : nullptr;
  // Populations: of step s from the kept trajectory, where the step before (or
  // the run's start) left them, and of step s + 1 to it; the run's last step
  // leaves them in the state.  Without a kept trajectory the state holds them
  // throughout.
  const bool last = s + 1 >= jb.t1;
  gcint* pop_in = KEEP_PT ? gptr(jb.pt) + (size_t)s * CAG : gptr(jb.state);
  const rsrc_t pop_out = slab(KEEP_PT && !last ? jb.pt + (size_t)(s + 1) * CAG : jb.state, CAG * 4);
  rsrc_t tn_b, tm_b;
  if constexpr (KEEP_TN) tn_b = slab(jb.tn + (size_t)s * TAG, TAG * 4);
  if constexpr (KEEP_TM) tm_b = slab(jb.tm + (size_t)s * TAG, TAG * 4);
  const int upd = s < S - 1 ? -1 : 0;
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const uint32_t c0 = (uint32_t)s | (stream << 16);
  const uint32_t off = 4u * (uint32_t)cell;
  int j = 0, g = 0;
  if (valid) {
    j = cell / G;
    g = cell - j * G;
    // Every load before the first store.
    int p[CP];
#pragma unroll
    for (int c = 0; c < CP; c++) p[c] = c < C ? pop_in[c * AG + cell] : 0;
    int nini[T];
    float lini[T];
    if constexpr (MODE == MODE_MBP) {
#pragma unroll
      for (int tr = 0; tr < T; tr++) {
        nini[tr] = itn[tr * AG + cell];
        lini[tr] = itm[tr * AG + cell];
      }
    }
    if constexpr (MODE == MODE_REPLAY) {
#pragma unroll
      for (int tr = 0; tr < T; tr++) nini[tr] = tn_r[tr * AG + cell];
    }
    gcfloat* Ib = gptr(Ibuf) + (size_t)b * G * Apad;
    float nmi = 0.f;
#pragma unroll
    for (int gg = 0; gg < G; gg++) nmi += sN[g * G + gg] * Ib[(size_t)gg * Apad + j];
    if (nmi < 0.f) nmi = 0.f;
    float bet, ef, agc;
    foi_groups(tp, tab, s, j, g, DPM, bet, ef, agc);
    float afc = af_row(tp, tab, s)[j];
    if constexpr (MODS) mod_foi_factors(tp, s, cell, afc, agc);
    const float foi = foi_mean(bet, afc, nmi, ef, agc);
    const bool simu = MODE == MODE_MBP ? (jb.simu ? gptr(jb.simu)[(size_t)s * A + j] != 0 : false) : true;
    // All means first, without a branch.
    float lp[T];
    int bad = 0;
#pragma unroll
    for (int tr = 0; tr < T; tr++) {
      const float popu = (float)p[FROM[tr]];
      const float mean = tr == INF_TR ? dt * popu * ssus[g] * foi : dt * popu * srate[tr * G + g];
      lp[tr] = popu > 0.f ? mean : 0.f;
    }
    if constexpr (MODS) {
#pragma unroll
      for (int tr = 0; tr < T; tr++) lp[tr] = mod_mean(tp, s, tr, cell, lp[tr]);
    }
#pragma unroll
    for (int tr = 0; tr < T; tr++) {
      bad |= lp[tr] != lp[tr] ? 1 : lp[tr] > 1e9f ? 2 : 0;
      lp[tr] = lp[tr] <= 1e9f ? lp[tr] : 0.f;
    }
    if (wave_any(bad != 0)) {
      if (bad) atomicOr(jb.err, bad);
    }
    if constexpr (KEEP_TM) {
#pragma unroll
      for (int tr = 0; tr < T; tr++) st_slab(tm_b, __float_as_int(lp[tr]), off, (uint32_t)(4 * tr * AG));
    }
    int q[CP];
#pragma unroll
    for (int c = 0; c < CP; c++) q[c] = p[c];
    if constexpr (MODE == MODE_REPLAY) {
#pragma unroll
      for (int tr = 0; tr < T; tr++) {
        q[FROM[tr]] -= nini[tr] & upd;
        q[TO[tr]] += nini[tr] & upd;
      }
    } else {
      CellRng rng;
      rng.init(k0, k1, c0, (uint32_t)cell, jb.key);
      rng.prime();
      // qv[tr] != 0: queued, a value of the fused kernel's three kinds.
      float qv[T];
#pragma unroll
      for (int tr = 0; tr < T; tr++) {
        float lam = lp[tr];
        int base = 0;
        bool bino = false;
        float pr = 0.f;
        qv[tr] = lam >= BEEP_POIS_INLINE ? lam : 0.f;
        if constexpr (MODE == MODE_MBP) {
          const int ni = nini[tr];
          const float li = lini[tr];
          const bool coupled = !simu && lam > 0.f;
          const bool down = coupled && !(lam > li) && !(lam == li);
          const float dl = lam > li ? lam - li : 0.f;
          if (coupled) {
            base = ni;
            qv[tr] = dl >= BEEP_POIS_INLINE ? -dl : 0.f;
            lam = dl;
          }
          if (down) {
            pr = lp[tr] / li;
            const float pp = pr > 0.5f ? 1.f - pr : pr;
            bino = (float)ni * pp < 10.f;
            qv[tr] = bino ? 0.f : pr;
          }
        }
        int n = base;
        if ((lam > 0.f && qv[tr] == 0.f && !bino) || bino) {
          const float u = rng.next();
          if (!bino) n = base + poisson_inversion(lam, u);
          else n = binomial_draw_small(nini[tr], pr, u, rng);
        }
        n = qv[tr] != 0.f ? 0 : n;
        if constexpr (KEEP_TN) st_slab(tn_b, n, qv[tr] != 0.f ? 0x80000000u : off, (uint32_t)(4 * tr * AG));
        q[FROM[tr]] -= n & upd;
        q[TO[tr]] += n & upd;
      }
      int total = 0;
#pragma unroll
      for (int tr = 0; tr < T; tr++) total += __popcll(__builtin_amdgcn_ballot_w64(qv[tr] != 0.f));
      if (total) {
        const int lane = (int)__lane_id();
        const int leader = __ffsll((long long)__builtin_amdgcn_ballot_w64(true)) - 1;
        int slot0 = 0;
        if (lane == leader) slot0 = atomicAdd(&qcount, total);
        slot0 = __builtin_amdgcn_readlane(slot0, leader);
#pragma unroll
        for (int tr = 0; tr < T; tr++) {
          const unsigned long long qm = __builtin_amdgcn_ballot_w64(qv[tr] != 0.f);
          if (qv[tr] != 0.f) {
            const int slot = slot0 + __popcll(qm & ((1ull << lane) - 1ull));
            qcode[slot] = (uint16_t)(tid * T + tr);
            qval[slot] = qv[tr];
          }
          slot0 += __popcll(qm);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < CP; c++) spop[c][tid] = q[c];
  }
  __syncthreads();
  const int nq = qcount;
  for (int i = tid; i < nq; i += BEEP_STEP_BLOCK) {
    const uint32_t code = qcode[i];
    const int t2 = (int)(code / T), tr = (int)(code - (uint32_t)t2 * T);
    const int c2 = blockIdx.y * BEEP_STEP_BLOCK + t2;
    const float v = qval[i];
    int n;
    if constexpr (MODE == MODE_SIM) {
      n = draw_large_poisson(v, k0, k1, c0, (uint32_t)c2, (uint32_t)tr, jb.key);
    } else {
      const int kind = v < 0.f ? ITEM_POIS_ADD : (v < 1.f ? ITEM_BINOM : ITEM_POIS);
      const int ni = MODE == MODE_MBP ? itn[tr * AG + c2] : 0;
      n = draw_item_inline(kind, fabsf(v), ni, k0, k1, c0, (uint32_t)c2, (uint32_t)tr, jb.key);
    }
    if constexpr (KEEP_TN) st_slab(tn_b, n, 4u * (uint32_t)(tr * AG + c2), 0);
    if (upd && n != 0) {
      int fr = 0, to = 0;
#pragma unroll
      for (int k = 0; k < T; k++)
        if (k == tr) { fr = FROM[k]; to = TO[k]; }
      atomicSub(&spop[fr][t2], n);
      atomicAdd(&spop[to][t2], n);
    }
  }
  __syncthreads();
  if (valid) {
    float d = 0.f;
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int v = spop[c][tid];
      __builtin_amdgcn_raw_buffer_store_b32(v, pop_out, (int)off, 4 * c * AG, 0);
      if (INFC[c]) {
        const float w = sinf[c];
        if (w != 0.f) d += w * (float)v;
      }
    }
    ((gfloat*)D)[frag_at(b * G + g, j, Apad)] = d;
  }
}

}  // namespace beepdev

#ifdef BEEP_SPEC_STEP
extern "C" __global__ void __launch_bounds__(BEEP_STEP_BLOCK, beepspec::STEP_WAVES)
    beep_step_spec_sim(const beepdev::Job* jobs, const float* I, float* D, int Apad, int s, const uint64_t* rngp) {
  beepdev::step_spec_body<beepdev::MODE_SIM>(jobs, I, D, Apad, s, rngp);
}
extern "C" __global__ void __launch_bounds__(BEEP_STEP_BLOCK, beepspec::STEP_WAVES)
    beep_step_spec_mbp(const beepdev::Job* jobs, const float* I, float* D, int Apad, int s, const uint64_t* rngp) {
  beepdev::step_spec_body<beepdev::MODE_MBP>(jobs, I, D, Apad, s, rngp);
}
extern "C" __global__ void __launch_bounds__(BEEP_STEP_BLOCK, beepspec::STEP_WAVES)
    beep_step_spec_replay(const beepdev::Job* jobs, const float* I, float* D, int Apad, int s, const uint64_t* rngp) {
  beepdev::step_spec_body<beepdev::MODE_REPLAY>(jobs, I, D, Apad, s, rngp);
}
#endif
