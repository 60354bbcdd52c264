// Particle-filter kernels of the PMCMC likelihood estimate: the bootstrap
// resampling step, the state moves between sections and the gather of one
// sampled trajectory from its ancestors.  Weights and the log-mean-exp are
// FP64.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_rng.hh"
#include "fused_common.hh"

namespace beepdev {

#define BEEP_BOOT_BLOCK 1024
#define BEEP_BOOT_LDS 2048
#define BEEP_BOOT_UNSET 0x7FFFFFFF

// Exclusive prefix sum of one int per thread over the workgroup; returns the
// total in *total (all threads).  red holds BEEP_BOOT_BLOCK/64 ints.
__device__ inline int block_excl_scan(int v, int* red, int* total) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int x = v;
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o);
    if (l >= o) x += y;
  }
  __syncthreads();
  if (l == 63) red[w] = x;
  __syncthreads();
  int before = 0, all = 0;
  for (int k = 0; k < nw; k++) {
    if (k < w) before += red[k];
    all += red[k];
  }
  *total = all;
  return before + x - v;
}

__device__ inline double block_max_d(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  double t = red[0];
  for (int k = 1; k < nw; k++) t = fmax(t, red[k]);
  return t;
}

// PMCMC::bootstrap (src/pmcmc.cc:211-268) for one section, one workgroup of
// BEEP_BOOT_BLOCK threads over n particles.  L_p = L[p] + L[n + p] + ... over the
// nchunk chunks of the section's observations is particle p's log-likelihood.
//   w_p = exp(invT (L_p - Lmax)),  wsum_p = sum_{q<=p} w_q,
//   obprob += invT Lmax + log(wsum_{n-1} / n)                 (224-236)
//   draw j: z = u_j wsum_{n-1}; pp = first p with z <= wsum_p  (245-248)
//   the first draw of each pp keeps it in place (bp[pp] = pp); later draws of
//   the same pp are "extras", handed out last-first to the particles no draw
//   chose, in increasing particle order                          (249-260)
// The linear search of the reference and the binary search here return the
// same index on the nondecreasing wsum.  Thread t owns the contiguous chunk
// [t*cs, (t+1)*cs) of particles and of draws, so the scans below keep draw
// order.  LDS: the work arrays are in LDS (n <= BEEP_BOOT_LDS), else in the
// scratch arrays wsum[n] double, first[n], draw[n], extra[n] int: the kernel is
// one chain of dependent steps, and each of the binary search's is a load (500
// particles: 13.5 us with them in memory, 7.4 in LDS; 512 particles of five
// chunks 18 and 12).
template <bool LDS>
__global__ void __launch_bounds__(BEEP_BOOT_BLOCK) k_bootstrap(int n, const double* __restrict__ L, int nchunk,
                                                             double invT, uint64_t seed, uint32_t stream, int sec,
                                                             int* __restrict__ bp, double* __restrict__ g_wsum,
                                                             int* __restrict__ g_first, int* __restrict__ g_draw,
                                                             int* __restrict__ g_extra, double* __restrict__ obprob,
                                                             int* __restrict__ err) {
  constexpr int N = LDS ? BEEP_BOOT_LDS : 1;
  __shared__ double l_wsum[N];
  __shared__ int l_first[N], l_draw[N], l_extra[N];
  auto wsum = [&](int p) -> double& { if constexpr (LDS) return l_wsum[p]; else return g_wsum[p]; };
  auto first = [&](int p) -> int& { if constexpr (LDS) return l_first[p]; else return g_first[p]; };
  auto draw = [&](int p) -> int& { if constexpr (LDS) return l_draw[p]; else return g_draw[p]; };
  auto extra = [&](int p) -> int& { if constexpr (LDS) return l_extra[p]; else return g_extra[p]; };
  __shared__ double redd[BEEP_BOOT_BLOCK / 64];
  __shared__ int redi[BEEP_BOOT_BLOCK / 64];
  __shared__ double s_sum;
  const int t = threadIdx.x;
  const int cs = (n + blockDim.x - 1) / blockDim.x;
  const int lo = min(n, t * cs), hi = min(n, lo + cs);

  // Lmax; a NaN anywhere makes the estimate NaN (reference: emsgEC("PMCMC",1)).
  double mx = -INFINITY;
  int bad = 0;
  for (int p = lo; p < hi; p++) {
    double v = L[p];
    for (int c = 1; c < nchunk; c++) v += L[(size_t)c * n + p];
    if (v != v) bad = 1;
    mx = fmax(mx, v);
    wsum(p) = v;
    first(p) = BEEP_BOOT_UNSET;
  }
  const double Lmax = block_max_d(mx, redd);

  // Inclusive prefix sum of the weights: chunk sums, then a scan over chunks.
  double loc = 0;
  for (int p = lo; p < hi; p++) {
    loc += exp(invT * (wsum(p) - Lmax));
    wsum(p) = loc;
  }
  // A place of padding every 16: wavefront 0's threads read runs of 16.
  __shared__ double chunk[BEEP_BOOT_BLOCK + BEEP_BOOT_BLOCK / 16];
  chunk[t + (t >> 4)] = loc;
  __syncthreads();
  if (t < 64) {                      // wavefront 0 scans the chunk sums
    constexpr int per = BEEP_BOOT_BLOCK / 64;
    static_assert(per == 16, "one place of padding per run");
    double v[per];
#pragma unroll
    for (int k = 0; k < per; k++) v[k] = chunk[t * (per + 1) + k];
    double a = 0;
#pragma unroll
    for (int k = 0; k < per; k++) a += v[k];
    double x = a;
    for (int o = 1; o < 64; o <<= 1) {
      double y = __shfl_up(x, o);
      if (t >= o) x += y;
    }
    double base = x - a;
#pragma unroll
    for (int k = 0; k < per; k++) {
      chunk[t * (per + 1) + k] = base;
      base += v[k];
    }
  }
  __syncthreads();
  const double off = chunk[t + (t >> 4)];
  for (int p = lo; p < hi; p++) wsum(p) += off;
  __syncthreads();
  if (t == 0) s_sum = wsum(n - 1);
  __syncthreads();
  const double sum = s_sum;         // z = u * sum <= wsum[n-1] for u < 1
  if (t == 0) {
    double ob = invT * Lmax + log(sum / n);
    if (bad || !(ob == ob) || isinf(ob)) atomicOr(err, 4);
    else obprob[0] += ob;
  }
  __syncthreads();

  // Draws; first[pp] = the earliest draw that chose pp.
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  for (int j = lo; j < hi; j++) {
    u4 r = philox4x32_10(u4{0xFFFEu | (stream << 16), (uint32_t)j, (uint32_t)sec, 0x7FFFFFFEu}, k0, k1);
    double z = u01d(r.x) * sum;
    int a = 0, b = n;                // first index with z <= wsum[index], n if none
    while (a < b) {
      int m = (a + b) >> 1;
      if (z <= wsum(m)) b = m;
      else a = m + 1;
    }
    if (a == n) {                    // reference: emsgEC("PMCMC",2)
      atomicOr(err, 4);
      a = n - 1;
    }
    draw(j) = a;
    atomicMin(&first(a), j);
  }
  __syncthreads();

  // Extras in draw order.
  int ne = 0;
  for (int j = lo; j < hi; j++) ne += first(draw(j)) != j;
  int tot_e;
  int pos = block_excl_scan(ne, redi, &tot_e);
  for (int j = lo; j < hi; j++)
    if (first(draw(j)) != j) extra(pos++) = draw(j);
  __syncthreads();

  // Unchosen particles, in increasing order, take extras from the back.
  int nu = 0;
  for (int p = lo; p < hi; p++) nu += first(p) == BEEP_BOOT_UNSET;
  int tot_u;
  int r = block_excl_scan(nu, redi, &tot_u);
  for (int p = lo; p < hi; p++) {
    if (first(p) != BEEP_BOOT_UNSET) {
      bp[p] = p;
    } else {
      int k = tot_e - 1 - r;
      r++;
      bp[p] = k >= 0 ? extra(k) : p;
    }
  }
  if (t == 0 && tot_e != tot_u) atomicOr(err, 4);   // reference: emsgEC("PMCMC",3)
}

// A particle filter's jobs of section k >= 1: those of section 0 over the steps
// of section k, which start from the state.  Grid (ceil(n / 256), nsec - 1).
// 500 particles x 8 sections: made and copied on the host 170 us a call, here 5.
__global__ void __launch_bounds__(256) k_section_jobs(Job* __restrict__ jobs, int n, const int* __restrict__ sec_ti,
                                                      const int* __restrict__ sec_tf) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, k = (int)blockIdx.y + 1;
  if (i >= n) return;
  Job j = jobs[i];
  j.t0 = sec_ti[k];
  j.t1 = sec_tf[k];
  j.from_init = j.t0 == 0 ? 1 : 0;
  jobs[(size_t)k * n + i] = j;
}

// Mpi::end_sec_swap (src/mpi.cc:215-327) on one device: particle p takes the
// current populations of particle bp[p].  Grid (n, chunks).  Sources are particles that kept
// their own state (bp[src] == src), so no source is overwritten.
__global__ void k_move_states(const int* __restrict__ inst, const int* __restrict__ bp, int* __restrict__ state,
                              size_t state_sz) {
  const int p = blockIdx.x;
  const int src = bp[p];
  if (src == p) return;
  const int* s_ = state + (size_t)inst[src] * state_sz;
  int* d_ = state + (size_t)inst[p] * state_sz;
  for (size_t k = blockIdx.y * blockDim.x + threadIdx.x; k < state_sz; k += (size_t)gridDim.y * blockDim.x)
    d_[k] = s_[k];
}

// Mpi::particle_sample (src/mpi.cc:331-385): the trajectory of the particle
// drawn first by the last bootstrap, traced back through the ancestry, is
// gathered section by section into instance dst.  bp holds nsec+1 rows of n
// (row k+1 written by the bootstrap of section k).  One workgroup row per
// section; the per-step trajectory slabs are tn/tm [T*AG], pt [C*AG].
__global__ void k_particle_sample(int n, int nsec, const int* __restrict__ sec_ti, const int* __restrict__ sec_tf,
                                  const int* __restrict__ bp, const int* __restrict__ inst, int dst,
                                  int* __restrict__ tn, float* __restrict__ tm, int* __restrict__ pt, size_t traj_sz,
                                  size_t pop_traj_sz, int TAG, int CAG) {
  const int sec = blockIdx.y;
  int p = bp[(size_t)nsec * n];
  for (int s = nsec - 1; s > sec; s--) p = bp[(size_t)s * n + p];
  const int src = inst[p];
  if (src == dst) return;
  const size_t t0 = sec_ti[sec], t1 = sec_tf[sec];
  const size_t a = t0 * TAG, b = t1 * TAG;
  for (size_t k = a + blockIdx.x * blockDim.x + threadIdx.x; k < b; k += (size_t)gridDim.x * blockDim.x) {
    if (tn) tn[(size_t)dst * traj_sz + k] = tn[(size_t)src * traj_sz + k];
    if (tm) tm[(size_t)dst * traj_sz + k] = tm[(size_t)src * traj_sz + k];
  }
  if (pt) {
    const size_t pa = t0 * CAG, pb = t1 * CAG;
    for (size_t k = pa + blockIdx.x * blockDim.x + threadIdx.x; k < pb; k += (size_t)gridDim.x * blockDim.x)
      pt[(size_t)dst * pop_traj_sz + k] = pt[(size_t)src * pop_traj_sz + k];
  }
}

}  // namespace beepdev

namespace beepdev {

#define BEEP_ABC_BLOCK 256
#define BEEP_ABC_J 2                // previous particles a thread works on at a time (4: 253 registers, two wavefronts per SIMD)
#define BEEP_ABC_WGS 2048           // workgroups aimed at: eight per CU

typedef const __attribute__((address_space(4))) double cdouble;

// ABCSMC::calculate_particle_weight (src/abcsmc.cc:260-271) for n_new
// proposals at once, FP64:
//   den[i] = sum_j w[j] exp(MVN::probability(theta_i, prev_j)),
//   MVN::probability(a, b) = -0.5 sum_{v1} sum_{v2} ((a-b)_v1 / size) invM[v1][v2] ((a-b)_v2 / size)
//                                                         (src/mvn.cc:185-195)
//   out[i] = exp(logprior[i]) / den[i].
// The quadratic form of any matrix is that of its upper triangle with the
// mirrored entries added, so a pair costs NV (NV + 1) / 2 + NV FMAs: U holds
// that triangle over size^2, row after row, NV being nvar rounded up to an
// even number and the padding zero.  The differences
// are formed per pair, so nothing cancels that did not before.
//
// Bound: FP64 FMA issue (253 + 22 per pair at 22 variables, plus the exp).  A
// thread keeps its proposal and the differences of BEEP_ABC_J previous
// particles in registers; U and the previous particles are the same for the
// whole wavefront and come as scalar operands, each entry of U feeding
// BEEP_ABC_J FMAs, so the loop has no LDS and no vector loads.  The previous
// generation is split over workgroups (grid: blocks of proposals x splits of
// jper previous particles), one partial sum per (split, proposal).
// 4096 x 4096 x 22: 0.20 ms, 5.0 G FMAs at 0.69 of the FP64 product rate; one
// thread per proposal with the matrix and the differences in LDS, on 32
// workgroups, took 92 ms.
// Blocks of eight entries of the triangle of NV variables (at least two).
__host__ __device__ constexpr int abc_blocks(int NV) {
  const int n = (NV * (NV + 1) / 2 + 7) / 8;
  return n < 2 ? 2 : n;
}

// Rows V and up of the triangle (compile-time recursion over rows, the row
// unrolled: every index below is a constant): q = the form so far, for J pairs.
template <int NV, int J, int V>
__device__ inline __attribute__((always_inline)) void abc_rows(cdouble*& Up, double (&u)[3][8], const double (&d)[J][NV],
                                                               double (&q)[J]) {
  if constexpr (V < NV) {
    constexpr int E0 = V * NV - V * (V - 1) / 2;       // the row's first entry
    double a[J];
#pragma unroll
    for (int k = 0; k < J; k++) a[k] = 0.0;
#pragma unroll
    for (int x = V; x < NV; x++) {
      const int E = E0 + x - V, c = E / 8;
      if (E % 8 == 0 && c + 2 < abc_blocks(NV)) {
        if (c > 0) asm volatile("" : "+s"(Up), "+v"(a[0]));
#pragma unroll
        for (int e = 0; e < 8; e++) u[(c + 2) % 3][e] = Up[(c + 2) * 8 + e];
      }
#pragma unroll
      for (int k = 0; k < J; k++)
        a[k] = x == V ? u[c % 3][E % 8] * d[k][x] : __builtin_fma(u[c % 3][E % 8], d[k][x], a[k]);
    }
#pragma unroll
    for (int k = 0; k < J; k++) q[k] = __builtin_fma(a[k], d[k][V], q[k]);
    abc_rows<NV, J, V + 1>(Up, u, d, q);
  }
}

template <int NV>
__global__ void __launch_bounds__(BEEP_ABC_BLOCK, 2)
    k_abcsmc_partial(int n_prev, int jper, const double* prev_, const double* w_, int n_new,
                     const double* __restrict__ theta, const double* U_, double* __restrict__ partial) {
  constexpr int J = BEEP_ABC_J;
  cdouble* prev = (cdouble*)prev_;
  cdouble* w = (cdouble*)w_;
  cdouble* U = (cdouble*)U_;
  const int i = blockIdx.x * BEEP_ABC_BLOCK + threadIdx.x;
  const int ic = min(i, n_new - 1);
  double th[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) th[v] = theta[(size_t)ic * NV + v];
  const int j0 = blockIdx.y * jper, j1 = min(n_prev, j0 + jper);
  double den = 0.0;
  for (int j = j0; j < j1; j += J) {
    double d[J][NV], q[J];
#pragma unroll
    for (int k = 0; k < J; k++) {
      cdouble* pj = prev + (size_t)min(j + k, n_prev - 1) * NV;
      if (k > 0) asm volatile("" : "+s"(pj), "+v"(d[k - 1][NV - 1]));
      q[k] = 0.0;
#pragma unroll
      for (int v = 0; v < NV; v++) d[k][v] = th[v] - pj[v];
    }
    // The triangle in order, eight entries (one 64-byte scalar load) at a
    // time, two loads ahead.  The empty asm ties each load's address to a
    // value of the block before: hoisted to the top or out of the loop, the
    // loads would spill the whole triangle.
    cdouble* Up = U;
    asm volatile("" : "+s"(Up), "+v"(d[J - 1][NV - 1]));
    double u[3][8];
#pragma unroll
    for (int e = 0; e < 8; e++) u[0][e] = Up[e];
#pragma unroll
    for (int e = 0; e < 8; e++) u[1][e] = Up[8 + e];
    abc_rows<NV, J, 0>(Up, u, d, q);
    // All J forms are done here: sunk into the conditions below, the FMAs of
    // the later pairs would keep the whole triangle alive.
#pragma unroll
    for (int k = 0; k < J; k++) asm volatile("" : "+v"(q[k]));
#pragma unroll
    for (int k = 0; k < J; k++)
      if (j + k < j1) den += w[j + k] * exp(-0.5 * q[k]);
  }
  if (i < n_new) partial[(size_t)blockIdx.y * n_new + i] = den;
}

// The splits' sums in order, and the weight.
__global__ void __launch_bounds__(BEEP_ABC_BLOCK) k_abcsmc_finish(int n_new, int nsplit,
                                                                const double* __restrict__ partial,
                                                                const double* __restrict__ logprior,
                                                                double* __restrict__ out) {
  const int i = blockIdx.x * BEEP_ABC_BLOCK + threadIdx.x;
  if (i >= n_new) return;
  double den = 0.0;
#pragma unroll 8
  for (int s = 0; s < nsplit; s++) den += partial[(size_t)s * n_new + i];
  out[i] = exp(logprior[i]) / den;
}

// MC3::swap_states (src/mc3.cc:153-215) for the chains of one launch, each
// group of chains sharing a run swapped among themselves: five sweeps over
// neighbouring pairs (i, i+1) with the same run, accepting with probability
//   al = exp(0.5 (invT_i - invT_{i+1}) (EF_i - EF_{i+1}))
// and swapping the chain labels (order) and EF.  One thread per launch, as
// the sweeps are sequential; draw k uses the Philox counter
// {0xFFFD | stream << 16, k, 0, 0x7FFFFFFD}.
// The five sweeps of neighbour swaps over one ladder of n chains (EF already
// gathered); the uniforms are Philox blocks (0xFFFD | stream << 16, draw,
// ladder, 0x7FFFFFFD), draw counting the ladder's swap trials.
__device__ inline void mc3_sweeps(int n, const int* __restrict__ run, const double* __restrict__ invT,
                                  double* __restrict__ EF, int* __restrict__ order, int* __restrict__ ntr,
                                  int* __restrict__ nac, uint64_t seed, uint32_t stream, uint32_t ladder) {
  for (int i = 0; i < n; i++) {
    order[i] = i;
    ntr[i] = 0;
    nac[i] = 0;
  }
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  uint32_t draw = 0;
  for (int loop = 0; loop < 5; loop++) {
    for (int i = 0; i + 1 < n; i++) {
      if (run[i] != run[i + 1]) continue;
      const double al = exp(0.5 * (invT[i] - invT[i + 1]) * (EF[i] - EF[i + 1]));
      ntr[i]++;
      u4 r = philox4x32_10(u4{0xFFFDu | (stream << 16), draw++, ladder, 0x7FFFFFFDu}, k0, k1);
      if (u01d(r.x) < al) {
        nac[i]++;
        int to = order[i];
        order[i] = order[i + 1];
        order[i + 1] = to;
        double te = EF[i];
        EF[i] = EF[i + 1];
        EF[i + 1] = te;
      }
    }
  }
}

__global__ void k_mc3_swap(int n, const int* __restrict__ run, const double* __restrict__ invT,
                           const double* __restrict__ EFall, const int* __restrict__ inst, double* __restrict__ EF,
                           int* __restrict__ order, int* __restrict__ ntr, int* __restrict__ nac, uint64_t seed,
                           uint32_t stream) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  for (int i = 0; i < n; i++) EF[i] = EFall[inst[i]];
  mc3_sweeps(n, run, invT, EF, order, ntr, nac, seed, stream, 0u);
}

// Many ladders at once, one thread each: ladder l holds the chains
// ptr[l] .. ptr[l+1]-1, whose EF are read through per-chain pointers (their
// contexts' EF arrays); order is local to the ladder.
__global__ void k_mc3_swap_ladders(int nladder, const int* __restrict__ ptr, const int* __restrict__ run,
                                   const double* __restrict__ invT, const double* const* __restrict__ efp,
                                   double* __restrict__ EF, int* __restrict__ order, int* __restrict__ ntr,
                                   int* __restrict__ nac, uint64_t seed, uint32_t stream) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= nladder) return;
  const int b = ptr[l], e = ptr[l + 1];
  for (int i = b; i < e; i++) EF[i] = *efp[i];
  mc3_sweeps(e - b, run + b, invT + b, EF + b, order + b, ntr + b, nac + b, seed, stream, (uint32_t)l);
}

}  // namespace beepdev
