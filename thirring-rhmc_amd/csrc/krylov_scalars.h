// Scalar recurrences of the reference-order Krylov solvers, device side.
//
// Each step runs in one block of BLK threads on the sum (in every thread) of the
// operator's partial dot products.  It runs as a kernel of its own (k_scalar and others in
// solvers.hip) or in an extra block of the operator launch that follows
// (DslashLaunch::scal), where it overlaps with that launch's field work: every
// other block derives the one scalar it needs from the same sum.
#pragma once
#include "solvers.h"

namespace thr {

// iterations per block of the blocked shift updates (k_ms_flush)
constexpr int MSR = 32;

// CG state (measure_module.F90:41-120); lam: |r|^2 of the last two iterations
// by parity, so that a step never writes what its launch's other blocks read
struct CgState {
  double alpha, alphan, betacg, lam[2];
  float resid;
  int niterc, nx, itercg, stop, iterations;
};

// multishift state (multishift_module.F90:71-282); dl: delta of the last two
// iterations by parity
struct MsState {
  double delta, alpha, lambda, omega, omega_save, minus_omega, gammag, dl[2];
  double zeta_i[MAXSHIFT], zeta_ii[MAXSHIFT], zeta_iii[MAXSHIFT], omegas[MAXSHIFT],
      gammas[MAXSHIFT], corr[MAXSHIFT], aden[MAXSHIFT];
  int flags[MAXSHIFT], cg_returns[MAXSHIFT];
  int n, mini, maxi, umin, umax, cg_return, maxcg, stop, done, plain;
  int nonfinite;  // a dot product came out NaN/Inf: the solve stopped there
  float res;
  double resd;  // threshold used by the convergence test
  // blocked shift updates: the scalars of iteration j of the block for every
  // shift updated in it, how many iterations of the block updated shift i,
  // and the block's iterations so far
  double rec_om[MSR][MAXSHIFT], rec_ga[MSR][MAXSHIFT], rec_ze[MSR][MAXSHIFT];
  int cnt[MAXSHIFT], jcount;
  // the block's coefficients for its flush: p_i = ca P_i + sum cb R,
  // x_i = X_i + cc P_i + sum cd R
  double ca[MAXSHIFT], cc[MAXSHIFT], cb[MAXSHIFT][MSR], cd[MAXSHIFT][MSR];
  int fcnt[MAXSHIFT], fact[MAXSHIFT], fjc;
};

namespace {

// sum: the dot product, called after the state's loads are issued, so that the
// step waits once for both (see scalar_block)

// alpha of a CG iteration from |M p|^2
template <class F> __device__ inline void cg_alpha_step(CgState *st, F sum) {
  const int nx = st->nx, itercg = st->itercg;
  const double alphan = st->alphan;
  asm volatile("" ::: "memory");
  const double alphad = sum();
  if (threadIdx.x == 0) {
    st->nx = nx + 1;
    st->itercg = itercg + 1;
    st->alpha = alphan / alphad;
    // a non-finite |M p|^2 (NaN or Inf in the source, the guess or the links)
    // can never meet the stopping rule: end the solve here instead of at
    // niterc, with x as the iteration before left it (the field blocks of a
    // launch that carries this step test the same two values)
    if (!isfinite(alphad) || !isfinite(alphan / alphad)) {
      st->stop = 3;
      st->iterations = nx + 1;
    }
  }
}

// beta and the stopping rule from |r|^2; slot: where lam of this iteration goes
template <class F> __device__ inline void cg_beta_step(CgState *st, double *slot, F sum) {
  const int nx = st->nx, niterc = st->niterc;
  const double alphan = st->alphan;
  const float resid = st->resid;
  asm volatile("" ::: "memory");
  const double bn = sum();
  if (threadIdx.x == 0) {
    st->betacg = nx == 1 ? 0.0 : bn / alphan;
    st->alphan = bn;
    *slot = bn;
    if (!isfinite(bn)) {
      st->stop = 3;
      st->iterations = nx;
    } else if (bn < (double)resid) {
      st->stop = 1;
      st->iterations = nx;
    } else if (nx >= niterc) {
      // the Fortran loop ends with nx = niterc + 1
      st->iterations = niterc + 1;
      st->stop = 2;
    }
  }
}

// The shift recurrences take one thread per shift (MAXSHIFT <= 64: all in
// wave 0); each shift's arithmetic is the serial loop's.  One thread walking
// 25 shifts took 5.9 (alpha) and 11.7 us (lambda) per launch at 16^3 x 48,
// most of it the memory latency of one shift after another; so 2.6 and 3.4.
template <class F> __device__ inline void ms_alpha_step(MsState *st, F sum) {
  const int i = threadIdx.x, ic = min(i, MAXSHIFT - 1), mini = st->mini, maxi = st->maxi,
            cg = st->cg_return;
  const double os = st->omega, gg = st->gammag, delta = st->delta;
  const double z1 = st->zeta_i[ic], z2 = st->zeta_ii[ic], aden = st->aden[ic];
  asm volatile("" ::: "memory");
  const double al = sum(), om = -delta / al;
  const bool ok = isfinite(om);
  if (ok && i >= mini - 1 && i < maxi) {
    const double z3 = (z1 * z2 * os) / (om * gg * (z1 - z2) + z1 * os * (1.0 - aden * om));
    st->zeta_iii[i] = z3;
    st->omegas[i] = om * z3 / z2;
  }
  __syncthreads();  // every thread has read the scalars before thread 0 writes them
  if (threadIdx.x == 0) {
    st->cg_return = cg + 1;
    st->alpha = al;
    st->omega_save = os;
    st->omega = om;
    st->minus_omega = -om;
    if (!ok) {
      // nothing downstream of a non-finite omega is meaningful: stop before
      // any shift is updated.  Field blocks of a launch that carries this step
      // may still write their part of r, into a ring slot that no flush reads:
      // the iteration is not counted in jcount.
      st->nonfinite = 1;
      st->stop = 1;
      st->done = 1;
    }
  }
}

// REC: record the iteration's shift scalars for the block's flush; slot: where
// the next iteration's delta goes beside the state's
template <bool REC, class F>
__device__ inline void ms_lambda_step(MsState *st, double *slot, F sum) {
  __shared__ int s_nmin, s_nmax;
  const int i = threadIdx.x, ic = min(i, MAXSHIFT - 1), mini = st->mini, maxi = st->maxi,
            n = st->n, j = st->jcount, cg = st->cg_return, maxcg = st->maxcg, flag = st->flags[ic];
  const double delta = st->delta, om = st->omega, resd = st->resd;
  const double zeta2 = st->zeta_ii[ic], zeta3 = st->zeta_iii[ic], omi = st->omegas[ic],
               corr = st->corr[ic];
  asm volatile("" ::: "memory");
  const double lam = sum();
  if (!isfinite(lam)) {
    if (threadIdx.x == 0) {
      st->nonfinite = 1;
      st->stop = 1;
      st->done = 1;
    }
    return;
  }
  const double gg = lam / delta;
  if (i < 64) {  // wave 0: the ballot spans every shift
    const bool mine = i >= mini - 1 && i < maxi;
    double z2 = 0.0, z3 = 0.0;
    bool on = false;
    if (i < n) {
      z2 = zeta2;
      if (mine) {
        z3 = zeta3;
        const double ga = gg * z3 * omi / (z2 * om);
        st->gammas[i] = ga;
        st->cg_returns[i] = cg;
        if constexpr (REC) {
          st->rec_om[j][i] = omi;
          st->rec_ga[j][i] = ga;
          st->rec_ze[j][i] = z3;
          st->cnt[i] = j + 1;
        }
      }
      on = flag && !(sqrt(delta * z2 * z2) * corr < resd);
      if (!on) st->flags[i] = 0;
    }
    const unsigned long long live = __ballot(on);
    const int nmax = live ? 64 - __clzll(live) : 0, nmin = live ? __ffsll((long long)live) : n + 1;
    // the window only shrinks, so its shifts have their zeta in registers
    if (i >= nmin - 1 && i < nmax) {
      st->zeta_i[i] = z2;
      st->zeta_ii[i] = z3;
    }
    if (i == 0) {
      s_nmin = nmin;
      s_nmax = nmax;
    }
  }
  __syncthreads();  // also: every thread has read the scalars
  if (threadIdx.x == 0) {
    st->lambda = lam;
    st->gammag = gg;
    st->umin = mini;
    st->umax = maxi;
    st->mini = s_nmin;
    st->maxi = s_nmax;
    st->delta = lam;
    if (REC) {
      *slot = lam;
      st->jcount = j + 1;
    }
    if (!(s_nmax > s_nmin - 1 && cg < maxcg)) st->stop = 1;
  }
}

// the step that DslashLaunch::scal names
__device__ inline const int *scalar_stop(int kind, const void *st) {
  return kind <= SCAL_MS_LAMBDA ? &((const MsState *)st)->stop : &((const CgState *)st)->stop;
}
template <class F> __device__ inline void scalar_step(int kind, void *st, double *slot, F sum) {
  if (kind == SCAL_MS_ALPHA)
    ms_alpha_step((MsState *)st, sum);
  else if (kind == SCAL_MS_LAMBDA)
    ms_lambda_step<true>((MsState *)st, slot, sum);
  else if (kind == SCAL_CG_ALPHA)
    cg_alpha_step((CgState *)st, sum);
  else
    cg_beta_step((CgState *)st, slot, sum);
}

// The blocks in front of a launch's field blocks when it carries a scalar step.
// The step is a chain of waits, so its block is the launch's first and waits
// for the sum and the state together: as the last block it started when the
// field blocks made room, and the multishift at 16^3 x 48 (768 field blocks)
// took 9.73 ms against 9.33.  SCAL_LEAD of them, so that field block b still
// runs on XCD b % 8.
__device__ inline void scalar_block(const DslashLaunch &L) {
  if (blockIdx.x) return;
  constexpr int NP = 4;
  double part[NP];
  const int dn = L.done ? *L.done : 0;
#pragma unroll
  for (int k = 0; k < NP; k++) part[k] = L.fsum[min((int)threadIdx.x + k * BLK, L.fsum_n - 1)];
  if (dn) return;
  scalar_step(L.scal, L.sst, L.sslot, [&] {
    double v = 0.0;  // the field blocks' order of summation
#pragma unroll
    for (int k = 0; k < NP; k++)
      if ((int)threadIdx.x + k * BLK < L.fsum_n) v += part[k];
    for (int k = (int)threadIdx.x + NP * BLK; k < L.fsum_n; k += BLK) v += L.fsum[k];
    return block_sum_once<BLK, 3>(v);
  });
}

}  // namespace
}  // namespace thr
