// Structure-specialised fused simulation kernel, compiled at run time for one
// compartment structure (hiprtc).  The text compiled is a prelude defining
// namespace beepspec, then device_rng.hh, fused_common.hh and this file.  The
// prelude fixes:
//   constexpr int C, T, G, CP;        compartments, transitions, age groups,
//                                     C rounded up to a multiple of 4
//   constexpr int INF_TR;             the infection transition
//   constexpr int FROM[T], TO[T];     transition source / destination
//   constexpr bool INFC[C];           compartments with an infectivity weight
//   constexpr int NSTRAIN, DPM;       strains, and groups per strain (G = NSTRAIN * DPM)
//   constexpr bool GROUPED, N_TV, MODS, AF_STATIC;   R or external-force groups, a time-varying age matrix,
//                                     prediction-mode modifications, an area factor that does not vary
//   constexpr bool STAGED, Q16;       the mixing CSR staged in LDS, 16-bit queue indices
//   constexpr bool KEEP_TN, KEEP_TM, KEEP_PT;   the trajectories kept
//
// It computes exactly what k_fused (kernels.hh) computes -- the same FP32
// expressions in the same order and the same uniforms consumed in the same
// order -- so trajectories are bit-identical to the generic kernel and to the
// step-wise path for the same keys.  What the specialisation buys: a cell's
// populations sit in registers through the step with compile-time source and
// destination indices, the transition loop is unrolled, divisions by G are by
// a constant, and populations are single-buffered in LDS in 16-byte chunks of
// four compartments so one cell's compartments load and store as vectors.
//
// Per step: (B) area mixing, (C) means, small draws, updates of the cell's own
// populations and its infectivity for the next step, large draws queued; where
// some draw was queued, (D) the queued draws by all lanes, applied with LDS
// atomics, (E) the infectivities again.
//
// Few instances leave a compute unit with one or two wavefronts per SIMD, and
// a step is then a serial chain of latencies.  What keeps it short:
//  - loads and stores share one counter, so a load issued after a step's
//    trajectory stores waits for them too.  The step's scalars (beta, external
//    force, m) are held 64 steps to a register, one lane each; the area factor
//    is staged once when it does not vary; a cell's means are all formed before
//    its first store;
//  - a taken branch refetches instructions: stores go through slabs whose range
//    check drops a lane's store (st_slab), a cell's queued draws take one LDS
//    atomic together, errors are tested once per cell;
//  - steps that queue nothing have neither (D) nor (E): two barriers.
// Replaced: a branch per transition for each null check, error check, queue
// push and masked store, and four global loads per step behind the stores
// (92 branches per step of a single-cell instance, half of a wavefront's time in
// waits).  Proposals of 256 x 400 cells x 200 steps: 2.87 -> 1.96 ms, and 1.75
// with the context's choices at compile time and binomials drawn by counting; one
// single-cell instance, 100 steps: 0.395 -> 0.32 -> 0.235 ms.
#pragma once

namespace beepdev {

static_assert(beepspec::CP % 4 == 0 && beepspec::CP >= beepspec::C, "CP");

// Populations in LDS: compartment c of a cell in 16-byte chunk c / 4 of the
// cell; chunk k of all cells is contiguous, so one wavefront's 16-byte
// accesses to its cells' chunk are consecutive in LDS.
__device__ inline int pidx(int c, int cell, int AG) { return ((c >> 2) * AG + cell) * 4 + (c & 3); }

// Infectivity of a cell, dinf = sum_c inf_c * pop_c (State::set_I_from_pop),
// from its populations in registers or in LDS.
__device__ inline float infectivity(const int (&p)[beepspec::CP], const float* sinf) {
  float d = 0.f;
#pragma unroll
  for (int c = 0; c < beepspec::C; c++)
    if (beepspec::INFC[c]) {
      const float w = sinf[c];
      if (w != 0.f) d += w * (float)p[c];
    }
  return d;
}
__device__ inline float cell_infectivity(const int* pop, int cell, int AG, const float* sinf) {
  const int4* pv = (const int4*)pop;
  int p[beepspec::CP];
#pragma unroll
  for (int c4 = 0; c4 < beepspec::CP / 4; c4++) {
    const int4 v = pv[c4 * AG + cell];
    p[4 * c4] = v.x; p[4 * c4 + 1] = v.y; p[4 * c4 + 2] = v.z; p[4 * c4 + 3] = v.w;
  }
  return infectivity(p, sinf);
}

// Strains: for each strain-0 cell, the susceptibles of its dp summed over
// the strains (reads pop only; the caller's barrier publishes spool).
__device__ inline void pool_susceptibles(const int* pop, int* spool, int AG, int tid, int nt) {
  if constexpr (beepspec::NSTRAIN > 1) {
    constexpr int G = beepspec::G, DPM = beepspec::DPM, SUS = beepspec::FROM[beepspec::INF_TR];
    for (int cell = tid; cell < AG; cell += nt) {
      const int j = cell / G, g = cell - j * G;
      if (g < DPM) {
        int sum = 0;
#pragma unroll
        for (int st = 0; st < beepspec::NSTRAIN; st++) sum += pop[pidx(SUS, j * G + st * DPM + g, AG)];
        spool[cell] = sum;
      }
    }
  }
}

template <int MODE>
__device__ inline void fused_spec_body(const Job* __restrict__ jobs, uint64_t seed, uint32_t stream) {
  using namespace beepspec;
  const Job jb = jobs[blockIdx.x];
  constexpr int mode = MODE;
  ctopo* __restrict__ tpp = (ctopo*)jb.topo;
  const int A = tpp->A, S = tpp->S, AG = tpp->AG;
  const int nt = blockDim.x, tid = threadIdx.x;
  const float dt = tpp->dt;
  const int qcap = T * AG;                             // every (cell, transition): never full
  constexpr bool q16 = Q16;

  extern __shared__ int smem[];
  int* pop = smem;                                     // [CP/4][AG] chunks of 4 compartments
  float* sdinf = (float*)(pop + (size_t)AG * CP);      // [AG]
  float* sI = sdinf + AG;                              // [AG]
  float* qval = sI + AG;                               // [qcap] value; negative: ITEM_POIS_ADD
  int* qcount = (int*)(qval + qcap);                   // [4]
  float* srate = (float*)(qcount + 4);                 // [T][G]
  float* sN = srate + T * G;                           // [G][G]
  float* ssus = sN + G * G;                            // [G]
  float* sinf = ssus + G;                              // [C]
  gcfloat* diag = gptr(tpp->diag);
  gcfloat* fac = gptr(tpp->fac);
  gcint* in_ptr = gptr(tpp->in_ptr);
  gcint* in_src = gptr(tpp->in_src);
  gcfloat* in_w = gptr(tpp->in_w);
  gcint* order = gptr(tpp->mix_order);
  constexpr bool staged = STAGED;
  // This step's area factor and the external force's age weights, read by
  // every cell in (C): from LDS, so that no global load there waits behind the
  // trajectory stores still in flight (loads and stores share one counter).
  float* saf = sinf + C;                               // [A]
  constexpr bool grouped = GROUPED;
  const int nE = grouped ? tpp->nE : 1;
  float* sage = saf + A;                               // [nE][G] age weights of each external-force group
  // With R or external-force groups: this step's beta of every area and
  // external force of every (strain, area), and each (strain, area)'s group.
  float* sbeta = sage + (size_t)nE * G;                // [A]
  float* sefoi = sbeta + (grouped ? A : 0);            // [NSTRAIN][A]
  int* segrp = (int*)(sefoi + (grouped ? NSTRAIN * A : 0));   // [NSTRAIN][A]
  float* sdiag = (float*)(segrp + (grouped ? NSTRAIN * A : 0));
  float* sfac = sdiag + A;
  int* sptr = (int*)(sfac + A);
  int* ssrc = sptr + A + 1;
  float* sw = (float*)(ssrc + tpp->nnz);
  int* sord = (int*)(sw + tpp->nnz);
  // The queue's item indices (cell * T + tr), after the tables and, when
  // staged, the mixing CSR: 16 bits each when they fit.
  void* qidx = staged ? (void*)(sord + A) : (void*)sdiag;
  uint16_t* qidx16 = (uint16_t*)qidx;
  uint32_t* qidx32 = (uint32_t*)qidx;
  // Strains: each strain-0 cell's susceptibles pooled over the strains of its
  // dp (src/state.cc:395-404), after the queue's indices.
  int* spool = (int*)((char*)qidx + ((size_t)qcap * (q16 ? 2 : 4) + 3) / 4 * 4);
  if constexpr (staged) {
    for (int i = tid; i < A; i += nt) { sdiag[i] = diag[i]; sfac[i] = fac[i]; sord[i] = order[i]; }
    for (int i = tid; i <= A; i += nt) sptr[i] = in_ptr[i];
    for (int i = tid; i < tpp->nnz; i += nt) { ssrc[i] = in_src[i]; sw[i] = in_w[i]; }
  }

  gcfloat* __restrict__ tab = gptr(jb.tab);
  {
    gcint* src = gptr(jb.from_init ? tpp->pop_init : jb.state);
    for (int cell = tid; cell < AG; cell += nt) {
#pragma unroll
      for (int c = 0; c < CP; c++) pop[pidx(c, cell, AG)] = c < C ? src[c * AG + cell] : 0;
    }
    for (int i = tid; i < T * G; i += nt) srate[i] = tab[tpp->off_rate + i];
    for (int i = tid; i < G * G; i += nt) sN[i] = tab[tpp->off_N + i];
    for (int i = tid; i < G; i += nt) ssus[i] = tab[tpp->off_sus + i];
    for (int i = tid; i < C; i += nt) sinf[i] = tab[tpp->off_inf + i];
    for (int i = tid; i < nE * G; i += nt) sage[i] = gptr(tpp->agedist)[i];
    if constexpr (grouped)
      for (int i = tid; i < NSTRAIN * A; i += nt) segrp[i] = tpp->nE > 1 ? gptr(tpp->egrp)[i] : 0;
    if (tid == 0) qcount[0] = 0;
  }
  constexpr bool af_static = AF_STATIC;
  if constexpr (af_static) {
    gcfloat* af0 = af_row(tpp, tab, 0);
    for (int i = tid; i < A; i += nt) saf[i] = af0[i];
  }
  __syncthreads();

  // (E) for the first step.
  for (int cell = tid; cell < AG; cell += nt) sdinf[cell] = cell_infectivity(pop, cell, AG, sinf);
  pool_susceptibles(pop, spool, AG, tid, nt);
  __syncthreads();

  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const uint32_t TAG = (uint32_t)(T * AG), CAG = (uint32_t)(C * AG);

  const int lane64 = tid & 63;
  float vbeta = 0.f, vefoi = 0.f, vgeo = 0.f;          // this lane's step of the current 64
  gcfloat* tbeta = tab + tpp->off_beta;
  gcfloat* tefoi = tab + tpp->off_efoi;
  gcfloat* tgeo = tab + tpp->off_geo;
  const int t0 = jb.t0, spd = tpp->spd;

  for (int s = t0; s < jb.t1; s++) {
    const int s64 = (s - t0) & 63;
    if (s64 == 0) {
      const int sl = min(s + lane64, S - 1);
      vbeta = tbeta[sl];
      vefoi = tefoi[sl];
      vgeo = tgeo[sl];
    }
    auto of_step = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), s64)); };
    const float beta_s = of_step(vbeta), efoi_s = of_step(vefoi), m = of_step(vgeo);
    // The area factor's row where it varies: loaded here, written to LDS after
    // the mixing.  Read in (C) after the barrier that ends (B); step s-1's
    // reads ended at the barrier of (C).
    gcfloat* af_s = af_static ? nullptr : af_row(tpp, tab, s);
    const bool newrow = !af_static && (s == t0 || s % spd == 0);
    float afr = 0.f;
    if (newrow && tid < A) afr = af_s[tid];
    if constexpr (grouped) {
      const int nR = tpp->nR;
      for (int i = tid; i < A; i += nt) sbeta[i] = tab[tpp->off_beta + (size_t)s * nR + (nR > 1 ? gptr(tpp->rgrp)[i] : 0)];
      for (int i = tid; i < NSTRAIN * A; i += nt) sefoi[i] = tab[tpp->off_efoi + (size_t)s * nE + segrp[i]];
    }
    // A time-varying age matrix: this step's.  Step s-1's reads of sN in (C)
    // ended at the barrier after (C); these writes are seen after (B)'s.
    if constexpr (N_TV) {
      for (int i = tid; i < G * G; i += nt) sN[i] = tab[tpp->off_N + (size_t)s * G * G + i];
    }
    gcint* itn = mode == MODE_MBP ? gptr(jb.init_tn) + (size_t)s * TAG : nullptr;
    gcfloat* itm = mode == MODE_MBP ? gptr(jb.init_tm) + (size_t)s * TAG : nullptr;
    gcint* tn_r = mode == MODE_REPLAY ? gptr(jb.tn) + (size_t)s * TAG : nullptr;
    gcbyte* simu_s = mode == MODE_MBP && jb.simu ? gptr(jb.simu) + (size_t)s * A : nullptr;
    // A cell's global reads, issued before its first store.
    bool simu = mode != MODE_MBP;
    int nrep[T], nini[T];
    float lini[T];
    auto read_cell = [&](int cell) {
      if (mode == MODE_REPLAY) {
#pragma unroll
        for (int tr = 0; tr < T; tr++) nrep[tr] = tn_r[tr * AG + cell];
      }
      if (mode == MODE_MBP) {
        simu = simu_s ? simu_s[cell / G] != 0 : false;
#pragma unroll
        for (int tr = 0; tr < T; tr++) {
          nini[tr] = itn[tr * AG + cell];
          lini[tr] = itm[tr * AG + cell];
        }
      }
    };
    // (B) area mixing, from LDS when the CSR is staged there.
    if constexpr (staged)
      mix_cells((lcfloat*)sdiag, (lcfloat*)sfac, (lcint*)sptr, (lcint*)ssrc, (lcfloat*)sw, (lcint*)sord, sdinf, sI, m,
                G, AG, tid, nt);
    else
      mix_cells(diag, fac, in_ptr, in_src, in_w, order, sdinf, sI, m, G, AG, tid, nt);
    if (newrow) {
      if (tid < A) saf[tid] = afr;
      for (int i = tid + nt; i < A; i += nt) saf[i] = af_s[i];
    }
    __syncthreads();
    // (C) means, small draws, own-cell updates; large draws queued.
    const bool update = s < S - 1;           // the last step is not applied (src/state.cc:634)
    const int upd = update ? -1 : 0;
    const uint32_t c0 = (uint32_t)s | (stream << 16);
    rsrc_t tn_b, tm_b, pt_b;                 // this step's slabs
    if constexpr (KEEP_TN) tn_b = slab(jb.tn + (size_t)s * TAG, TAG * 4);
    if constexpr (KEEP_TM) tm_b = slab(jb.tm + (size_t)s * TAG, TAG * 4);
    if constexpr (KEEP_PT) pt_b = slab(jb.pt + (size_t)s * CAG, CAG * 4);
    for (int cell = tid; cell < AG; cell += nt) {
      const int j = cell / G, g = cell - j * G;
      const uint32_t off = 4u * (uint32_t)cell;
      read_cell(cell);
      int p[CP];
      {
        const int4* pv = (const int4*)pop;
#pragma unroll
        for (int c4 = 0; c4 < CP / 4; c4++) {
          int4 v = pv[c4 * AG + cell];
          p[4 * c4] = v.x; p[4 * c4 + 1] = v.y; p[4 * c4 + 2] = v.z; p[4 * c4 + 3] = v.w;
        }
      }
      int pool = 0;
      if constexpr (NSTRAIN > 1) {
        // Strain st's infections draw on the pooled susceptibles, which the
        // reference keeps in strain 0's dp (src/state.cc:395-425).
        const int st = g / DPM;
        pool = spool[j * G + (g - st * DPM)];
        p[FROM[INF_TR]] = st == 0 ? pool : 0;
      }
      float nmi = 0.f;
#pragma unroll
      for (int gg = 0; gg < G; gg++) nmi += sN[g * G + gg] * sI[j * G + gg];
      if (nmi < 0.f) nmi = 0.f;
      float afc = saf[j], agc, bet = beta_s, ef = efoi_s;
      if constexpr (grouped) {
        const int k = (g / DPM) * A + j;
        bet = sbeta[j];
        ef = sefoi[k];
        agc = sage[segrp[k] * G + g];
      } else {
        agc = sage[g];
      }
      if constexpr (MODS) mod_foi_factors(tpp, s, cell, afc, agc);
      const float foi = foi_mean(bet, afc, nmi, ef, agc);
      // All means first, without a branch.
      float lp[T];
      int bad = 0;
#pragma unroll
      for (int tr = 0; tr < T; tr++) {
        float popu = (float)p[FROM[tr]];
        if constexpr (NSTRAIN > 1) {
          if (tr == INF_TR) popu = (float)pool;
        }
        const float mean = tr == INF_TR ? dt * popu * ssus[g] * foi : dt * popu * srate[tr * G + g];
        lp[tr] = popu > 0.f ? mean : 0.f;
      }
      if constexpr (MODS) {
#pragma unroll
        for (int tr = 0; tr < T; tr++) lp[tr] = mod_mean(tpp, s, tr, cell, lp[tr]);
      }
      // src/state.cc:429 (NaN mean) and src/utils.cc:150 (mean > 1e9) stop the reference.
#pragma unroll
      for (int tr = 0; tr < T; tr++) {
        bad |= lp[tr] != lp[tr] ? 1 : lp[tr] > 1e9f ? 2 : 0;
        lp[tr] = lp[tr] <= 1e9f ? lp[tr] : 0.f;
      }
      if (wave_any(bad != 0)) {
        if (bad) atomicOr(jb.err, bad);
      }
      if constexpr (KEEP_PT) {
#pragma unroll
        for (int c = 0; c < C; c++) st_slab(pt_b, p[c], off, (uint32_t)(4 * c * AG));
      }
      if constexpr (KEEP_TM) {
#pragma unroll
        for (int tr = 0; tr < T; tr++) st_slab(tm_b, __float_as_int(lp[tr]), off, (uint32_t)(4 * tr * AG));
      }
      // Draws in transition order: n[tr] events now, or qv[tr] != 0 queued for
      // (D): a Poisson mean (>= 10), minus the mean of a proposal's additional
      // events (<= -10), or a binomial probability in (0, 1).
      int q[CP];
#pragma unroll
      for (int c = 0; c < CP; c++) q[c] = p[c];
      float qv[T];
      if constexpr (MODE == MODE_REPLAY) {
#pragma unroll
        for (int tr = 0; tr < T; tr++) {
          q[FROM[tr]] -= nrep[tr] & upd;
          q[TO[tr]] += nrep[tr] & upd;
        }
      } else {
        CellRng rng;
        rng.init(k0, k1, c0, (uint32_t)cell, jb.key);
        rng.prime();
#pragma unroll
        for (int tr = 0; tr < T; tr++) {
          float lam = lp[tr];                // mean of the Poisson part
          int base = 0;                      // events carried over from the current trajectory
          bool bino = false;
          float pr = 0.f;
          qv[tr] = lam >= BEEP_POIS_INLINE ? lam : 0.f;
          if constexpr (MODE == MODE_MBP) {
            // Coupled proposal (src/mbp.cc:286-311).
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
          const bool pois = lam > 0.f && qv[tr] == 0.f && !bino;
          int n = base;
          if (pois || bino) {
            const float u = rng.next();
            if (!bino) n = base + poisson_inversion(lam, u);
            else n = binomial_draw_small(nini[tr], pr, u, rng);
          }
          n = qv[tr] != 0.f ? 0 : n;
          // Lanes that queue have the store dropped by the slab's range check.
          if constexpr (KEEP_TN) st_slab(tn_b, n, qv[tr] != 0.f ? 0x80000000u : off, (uint32_t)(4 * tr * AG));
          q[FROM[tr]] -= n & upd;
          q[TO[tr]] += n & upd;
        }
        // The wavefront's queued draws take consecutive slots from one LDS
        // atomic (they are keyed by cell and transition, so the slots' order
        // is immaterial).
        int total = 0;
#pragma unroll
        for (int tr = 0; tr < T; tr++) total += __popcll(__builtin_amdgcn_ballot_w64(qv[tr] != 0.f));
        if (total) {
          const int lane = (int)__lane_id();
          const int leader = __ffsll((long long)__builtin_amdgcn_ballot_w64(true)) - 1;
          int base = 0;
          if (lane == leader) base = atomicAdd(qcount, total);
          base = __builtin_amdgcn_readlane(base, leader);
#pragma unroll
          for (int tr = 0; tr < T; tr++) {
            const unsigned long long qm = __builtin_amdgcn_ballot_w64(qv[tr] != 0.f);
            if (qv[tr] != 0.f) {
              const int slot = base + __popcll(qm & ((1ull << lane) - 1ull));
              const uint32_t idx = (uint32_t)cell * T + tr;
              if (q16) qidx16[slot] = (uint16_t)idx;
              else qidx32[slot] = idx;
              qval[slot] = qv[tr];
            }
            base += __popcll(qm);
          }
        }
      }
      {
        int4* pv = (int4*)pop;
#pragma unroll
        for (int c4 = 0; c4 < CP / 4; c4++)
          pv[c4 * AG + cell] = make_int4(q[4 * c4], q[4 * c4 + 1], q[4 * c4 + 2], q[4 * c4 + 3]);
      }
      if constexpr (NSTRAIN == 1) sdinf[cell] = infectivity(q, sinf);
    }
    __syncthreads();
    // (D) the queued large draws (PTRS / BTRD), every lane busy.
    int nq = 0;
    if constexpr (MODE != MODE_REPLAY) {
      nq = qcount[0];
      if (nq > 0) {
        for (int i = tid; i < nq; i += nt) {
          const uint32_t idx = q16 ? (uint32_t)qidx16[i] : qidx32[i];
          const int cell = (int)(idx / T), tr = (int)(idx - (uint32_t)cell * T);
          const float v = qval[i];
          int n;
          if constexpr (MODE == MODE_SIM) {
            n = draw_large_poisson(v, k0, k1, c0, (uint32_t)cell, (uint32_t)tr, jb.key);
          } else {
            const int kind = v < 0.f ? ITEM_POIS_ADD : (v < 1.f ? ITEM_BINOM : ITEM_POIS);
            n = draw_item_inline(kind, fabsf(v), itn[tr * AG + cell], k0, k1, c0, (uint32_t)cell, (uint32_t)tr, jb.key);
          }
          if constexpr (KEEP_TN) st_slab(tn_b, n, 4u * (uint32_t)(tr * AG + cell), 0);
          if (update && n != 0) {
            int fr = 0, to = 0;
#pragma unroll
            for (int k = 0; k < T; k++)
              if (k == tr) { fr = FROM[k]; to = TO[k]; }
            atomicSub(&pop[pidx(fr, cell, AG)], n);
            atomicAdd(&pop[pidx(to, cell, AG)], n);
          }
        }
        __syncthreads();
        if (tid == 0) qcount[0] = 0;
      }
    }
    // (E) infectivity for the next step, where (D) or the pooling over strains
    // changed what (C) wrote.
    if (NSTRAIN > 1 || nq > 0) {
      for (int cell = tid; cell < AG; cell += nt) sdinf[cell] = cell_infectivity(pop, cell, AG, sinf);
      pool_susceptibles(pop, spool, AG, tid, nt);
      __syncthreads();
    }
  }
  for (int cell = tid; cell < AG; cell += nt) {
#pragma unroll
    for (int c = 0; c < C; c++) ((gint*)jb.state)[c * AG + cell] = pop[pidx(c, cell, AG)];
  }
}

}  // namespace beepdev

#ifdef BEEP_SPEC_FUSED
extern "C" __global__ void __launch_bounds__(BEEP_SPEC_MAX_BLOCK, beepspec::MIN_WAVES)
    beep_fused_spec_sim(const beepdev::Job* jobs, uint64_t seed, uint32_t stream) {
  beepdev::fused_spec_body<beepdev::MODE_SIM>(jobs, seed, stream);
}
// The coupled proposal needs more registers than a simulation: at most five
// resident wavefronts per SIMD (96 registers) keep its spills small.
extern "C" __global__ void __launch_bounds__(BEEP_SPEC_MAX_BLOCK, beepspec::MIN_WAVES < 5 ? beepspec::MIN_WAVES : 5)
    beep_fused_spec_mbp(const beepdev::Job* jobs, uint64_t seed, uint32_t stream) {
  beepdev::fused_spec_body<beepdev::MODE_MBP>(jobs, seed, stream);
}
#ifdef BEEP_SPEC_REPLAY
extern "C" __global__ void __launch_bounds__(BEEP_SPEC_MAX_BLOCK, beepspec::MIN_WAVES)
    beep_fused_spec_replay(const beepdev::Job* jobs, uint64_t seed, uint32_t stream) {
  beepdev::fused_spec_body<beepdev::MODE_REPLAY>(jobs, seed, stream);
}
#endif
#endif
