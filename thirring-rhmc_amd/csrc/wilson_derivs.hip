// Wilson-kernel domain-wall operator (secondary generation kernel) and the
// Shamir fermion force.
//
// Wilson kernel, dirac.F90:226-299 (M) and 538-625 (M^dagger).  The reference
// builds it from 4-D Wilson applications on s-slices; with D_W that slice
// operator and the s-couplings collected into one field it reads
//   M  R = D_W (R + Q) + (R - Q),
//        Q(s) = P+ R(s-1) + P- R(s+1)       (interior s)
//             + c1 P+ R(Ls) at s=1, c2 P- R(1) at s=Ls
//   M^+R = T + R + P- cA (T - R)(s_A) + P+ cB (T - R)(s_B),  T = D_W^+ R
// so each application is one 4-D stencil pass: the s-couplings come by wave
// shuffles where an s-line fits one wave (Ls <= 64, k_wilson), and as two local
// passes around the Dslash kernel's 4-D form above that.
//
// Force, derivs_module.F90:99-196: for every link (x, mu) the sum over s and
// spin of the Wilson and Dirac parts of d/dtheta Re<R, M^(+) X2>, with the
// float32 coefficient tzi_real = 2*real(anum).
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "dslash_site.h"
#include "krylov_scalars.h"

namespace thr {

namespace {

__device__ inline void ld_spinor(const double2 *__restrict__ p, unsigned v5, unsigned site,
                                 cx<double> v[4]) {
#pragma unroll
  for (int a = 0; a < 4; a++) v[a] = ldc(p, (long)a * v5 + site);
}

// The Wilson kernel's s-couplings of a spinor held one site per lane, an
// s-line per segment of lanes: q = Q v with
//   (Q v)(s) = P+ v(s-1) + P- v(s+1),  P+ the spins 1, 2 and P- the spins 3, 4,
// and the wall terms c1 P+ v(Ls) at s = 1, c2 P- v(1) at s = Ls.  DAG: P+ and P-
// trade places (c1 goes with s - 1 and c2 with s + 1 as before).  lane0: the
// segment's first lane.  Every lane of the wave takes part.
struct WallCoef {
  double c1r, c1i, c2r, c2i;
};
template <bool DAG>
__device__ inline void couplings(const cx<double> v[4], cx<double> q[4], unsigned s, unsigned ls,
                                 unsigned lane0, const WallCoef &w) {
  const int dn = (int)(lane0 + (s == 0 ? ls - 1 : s - 1)), up = (int)(lane0 + (s + 1 < ls ? s + 1 : 0));
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const bool below = (a < 2) != DAG;
    const int src = below ? dn : up;
    const cx<double> n{__shfl(v[a].r, src, 64), __shfl(v[a].i, src, 64)};
    const bool wall = below ? s == 0 : s + 1 == ls;
    const cx<double> c = below ? cx<double>{w.c1r, w.c1i} : cx<double>{w.c2r, w.c2i};
    q[a] = wall ? cmul(c, n) : n;
  }
}
__device__ inline void add_couplings(cx<double> v[4], unsigned s, unsigned ls, unsigned lane0,
                                     const WallCoef &w) {
  cx<double> q[4];
  couplings<false>(v, q, s, ls, lane0, w);
#pragma unroll
  for (int a = 0; a < 4; a++) v[a] = v[a] + q[a];
}

// One side of a 4-D hop of M (half_hop) on the P+ part of v (spins 1, 2) and
// on its P- part (spins 3, 4) apart: A -= 1/2 (1 + SIG gamma_mu) U P+ v, B the
// same of P- v.
template <int MU, int SIG>
__device__ inline void half_hop_split(cx<double> A[4], cx<double> B[4], cx<double> u,
                                      const Site<P64> &S) {
  constexpr int p0 = kGamP[MU][0], p1 = kGamP[MU][1];
  constexpr double h = 0.5, hs = SIG > 0 ? 0.5 : -0.5;
  const cx<double> w0 = cmul(u, S.v[0]), w1 = cmul(u, S.v[1]);
  A[0] = A[0] - h * w0;
  A[1] = A[1] - h * w1;
  A[p0] = A[p0] - hs * phase<kGamE[MU][p0]>(w0);
  A[p1] = A[p1] - hs * phase<kGamE[MU][p1]>(w1);
  const cx<double> z0 = cmul(u, phase<kGamE[MU][0]>(S.v[p0])), z1 = cmul(u, phase<kGamE[MU][1]>(S.v[p1]));
  B[0] = B[0] - hs * z0;
  B[1] = B[1] - hs * z1;
  B[p0] = B[p0] - h * phase<kGamE[MU][p0]>(z0);
  B[p1] = B[p1] - h * phase<kGamE[MU][p1]>(z1);
}

// value of v at the segment's lane `src`, times c where it crossed the wall
__device__ inline cx<double> from_line(cx<double> v, int src, bool wall, cx<double> c) {
  const cx<double> n{__shfl(v.r, src, 64), __shfl(v.i, src, 64)};
  return wall ? cmul(c, n) : n;
}

// smallest power of two >= ls (ls <= 64): lanes per s-line
inline unsigned segment(int ls) {
  unsigned w = 1;
  while (w < (unsigned)ls) w <<= 1;
  return w;
}

// Wilson-kernel M or M^+ with the epilogues of the Dslash kernel, FP64, Ls <=
// 64: an s-line per lane segment, one site per lane, one t step per thread.
//   M:   out = A + B + R + (A - P+ R)(s-1) + (B - P- R)(s+1) with A = D_W P+ R
//        and B = D_W P- R (D_W is diagonal in s, so the shift along s may
//        follow it: 8 shuffled numbers per site instead of 28 when Y = R + Q R
//        is formed on each of the 7 loaded sites, and 11.3 us)
//   M^+: out = T + R + Q^+ (T - R),  T = D_W^+ R
// Bound by latency on the lattices this kernel is generated on (14^2 x 18 x
// 20: 4.5 MB fields), so everything is one pass with all loads issued
// together.  The passes it replaces took 16.5 us for M (couplings, stencil,
// combination) and 18.4 for M^+ (stencil, couplings, epilogue) there; this one
// takes 9.9 with its epilogue, and 7.8.
template <bool DAG, int MODE>
__global__ __launch_bounds__(BLK, 2) void k_wilson(const DslashLaunch L, unsigned wseg,
                                                   const WallCoef wall) {
  const int rhs = blockIdx.y;
  // one batch of argument loads (see k_dslash_site)
  asm volatile("" ::"s"(L.done), "s"(L.fsum), "s"(L.fdelta), "s"(L.b_ptr), "s"(L.r), "s"(L.in),
               "s"(L.out), "s"(L.links), "s"(L.partial), "s"(L.d.lx), "s"(L.am3), "s"(wseg));
  const int done = L.done ? L.done[(long)rhs * L.done_stride] : 0;
  const unsigned lx = L.d.lx, ly = L.d.ly, lt = L.d.lt, ls = L.d.ls;
  const unsigned v2 = lx * ly, v3 = v2 * ls, v4 = v2 * lt, v5 = v4 * ls;
  const unsigned nl = BLK / wseg, nb2 = (v2 + nl - 1) / nl;  // lines per block, blocks per t
  constexpr bool HREC = MODE == EPI_HREC || MODE == EPI_HPREC;
  constexpr bool SUM = MODE == EPI_CG || HREC;
  // the launch's field blocks, after those of a scalar step
  const unsigned lead = SUM && L.scal ? SCAL_LEAD : 0;
  if constexpr (SUM) {
    if (blockIdx.x < lead) {
      scalar_block(L);
      return;
    }
  }
  const unsigned bid = blockIdx.x - lead, nbl = nb2 * lt;
  const unsigned t = bid / nb2, lb = bid - t * nb2;
  const unsigned line = threadIdx.x / wseg, s = threadIdx.x - line * wseg;
  const unsigned col = lb * nl + line;  // 2-D site x + lx y
  const bool valid = s < ls && col < v2;
  const unsigned lane0 = (threadIdx.x & 63) - s;
  const long off = (long)rhs * 4 * v5;
  const bool fsum = SUM && L.fsum;
  const unsigned i = s + ls * col + v3 * t;
  Site<P64> c{}, f[3]{}, b[3]{}, old{}, pold{};  // old: the epilogue's h or r
  cx<double> uf[3]{}, ub[3]{};
  // the epilogue's scalars: delta of a fused one, else a (EPI_CG) or b; the
  // partial sums of a fused one
  const double *sp = fsum ? L.fdelta : MODE == EPI_CG ? L.a_ptr : L.b_ptr;
  const double *bp = MODE == EPI_CG && L.b_ptr ? L.b_ptr : sp;
  const bool first = MODE == EPI_HPREC && !L.b_ptr;  // b = 0
  constexpr int NP = 4;
  double part[NP] = {}, sc = 0.0, sb = 0.0;
  if constexpr (SUM) {
    if (sp) {
      sc = sp[(long)rhs * L.sc_stride];
      sb = bp[(long)rhs * L.sc_stride];
    }
    if (fsum) {
#pragma unroll
      for (int k = 0; k < NP; k++)
        part[k] = L.fsum[min((int)threadIdx.x + k * BLK, L.fsum_n - 1)];
    }
  }
  if (valid) {
    const double2 *in = (const double2 *)L.in + off, *u = (const double2 *)L.links;
    const unsigned x = col % lx, y = col / lx;
    const unsigned xf = x + 1 == lx ? 0 : x + 1, xb = x == 0 ? lx - 1 : x - 1;
    const unsigned yf = y + 1 == ly ? 0 : y + 1, yb = y == 0 ? ly - 1 : y - 1;
    const unsigned tf = t + 1 == lt ? 0 : t + 1, tb = t == 0 ? lt - 1 : t - 1;
    ld_spinor(in, v5, i, c.v);
    ld_spinor(in, v5, s + ls * (xf + lx * y) + v3 * t, f[0].v);
    ld_spinor(in, v5, s + ls * (xb + lx * y) + v3 * t, b[0].v);
    ld_spinor(in, v5, s + ls * (x + lx * yf) + v3 * t, f[1].v);
    ld_spinor(in, v5, s + ls * (x + lx * yb) + v3 * t, b[1].v);
    ld_spinor(in, v5, s + ls * col + v3 * tf, f[2].v);
    ld_spinor(in, v5, s + ls * col + v3 * tb, b[2].v);
    uf[0] = ldc(u, col + v2 * t);
    ub[0] = conj(ldc(u, xb + lx * y + v2 * t));
    uf[1] = ldc(u, v4 + col + v2 * t);
    ub[1] = conj(ldc(u, v4 + x + lx * yb + v2 * t));
    uf[2] = ldc(u, 2 * v4 + col + v2 * t);
    ub[2] = conj(ldc(u, 2 * v4 + col + v2 * tb));
    if constexpr (HREC) ld_spinor((const double2 *)L.out + off, v5, i, old.v);
    if constexpr (MODE == EPI_HPREC) ld_spinor((const double2 *)L.x + off, v5, i, pold.v);
    if constexpr (MODE == EPI_CG) ld_spinor((const double2 *)L.r + off, v5, i, old.v);
  }
  asm volatile("" ::: "memory");  // the loads stay above the branch and the barriers
  if (done) return;
  // a fused alpha that stops the solve (cg_alpha_step) must leave x as it is
  bool xgo = MODE == EPI_CG && L.b_ptr;
  if constexpr (SUM) {
    if (fsum) {  // the order of partial_sum
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < NP; k++)
        if ((int)threadIdx.x + k * BLK < L.fsum_n) v += part[k];
      for (int k = (int)threadIdx.x + NP * BLK; k < L.fsum_n; k += BLK) v += L.fsum[k];
      v = block_sum_once<BLK, 1>(v);
      sc = MODE == EPI_CG ? sc / v : v / sc;  // alpha = delta / |h|^2, gamma = lambda / delta
      xgo = xgo && isfinite(v) && isfinite(sc);
    }
  }
  const double ea = sc, eb = MODE == EPI_CG ? (fsum ? sc : sb) : first ? 0.0 : sc;
  const double diag = (double)(3.0f + (-L.am3));
  cx<double> o[4];
  if constexpr (!DAG) {
    cx<double> A[4]{}, B[4]{};
    A[0] = diag * c.v[0];
    A[1] = diag * c.v[1];
    B[2] = diag * c.v[2];
    B[3] = diag * c.v[3];
    half_hop_split<0, -1>(A, B, uf[0], f[0]);
    half_hop_split<0, 1>(A, B, ub[0], b[0]);
    half_hop_split<1, -1>(A, B, uf[1], f[1]);
    half_hop_split<1, 1>(A, B, ub[1], b[1]);
    half_hop_split<2, -1>(A, B, uf[2], f[2]);
    half_hop_split<2, 1>(A, B, ub[2], b[2]);
    const int dn = (int)(lane0 + (s == 0 ? ls - 1 : s - 1));
    const int up = (int)(lane0 + (s + 1 < ls ? s + 1 : 0));
#pragma unroll
    for (int a = 0; a < 4; a++) {
      o[a] = A[a] + B[a] + c.v[a];
      if (a < 2)
        A[a] = A[a] - c.v[a];
      else
        B[a] = B[a] - c.v[a];
      o[a] = o[a] + from_line(A[a], dn, s == 0, {wall.c1r, wall.c1i});
      o[a] = o[a] + from_line(B[a], up, s + 1 == ls, {wall.c2r, wall.c2i});
    }
  } else {
    centre(o, diag, c);
    hop<0, DAG>(o, uf[0], f[0], ub[0], b[0]);
    hop<1, DAG>(o, uf[1], f[1], ub[1], b[1]);
    hop<2, DAG>(o, uf[2], f[2], ub[2], b[2]);
    cx<double> w[4], q[4];
#pragma unroll
    for (int a = 0; a < 4; a++) w[a] = o[a] - c.v[a];
    couplings<true>(w, q, s, ls, lane0, wall);
#pragma unroll
    for (int a = 0; a < 4; a++) o[a] = o[a] + c.v[a] + q[a];
  }
  double red = 0.0;
  if (valid) {
    double2 *out = (double2 *)L.out + off;
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const long e = (long)a * v5 + i;
      if constexpr (MODE == EPI_CG) {
        const cx<double> rv = old.v[a] - ea * o[a];
        st((double2 *)(L.r_out ? L.r_out : L.r) + off, e, rv);
        red += norm2(rv);
        if (xgo) {
          double2 *xo = (double2 *)L.x + off;
          st(xo, e, ldc(xo, e) + eb * ldc((const double2 *)L.p + off, e));
        }
      } else {
        if constexpr (HREC) o[a] = o[a] + eb * old.v[a];
        st(out, e, o[a]);
        if constexpr (MODE == EPI_HPREC)
          st((double2 *)L.x + off, e, first ? c.v[a] : c.v[a] + eb * pold.v[a]);
        if constexpr (MODE == EPI_NORM || HREC) red += norm2(o[a]);
        if constexpr (MODE == EPI_DOTW) {
          const cx<double> wv = ldc((const double2 *)L.w + off, e);
          red += wv.r * o[a].r + wv.i * o[a].i;
        }
      }
    }
  }
  if constexpr (MODE != EPI_STORE) {
    const double tot = block_sum_once<BLK, 2>(red);
    if (threadIdx.x == 0) L.partial[(long)rhs * nbl + bid] = tot;
  }
}

// Y = R + Q  (M) ; coefficients c1, c2 multiply the wall terms
__global__ __launch_bounds__(BLK) void k_wk_pre(const Dims d, int nrhs, const double2 *R,
                                                double2 *Y, double2 c1, double2 c2) {
  const long v5 = d.v5();
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= v5 * nrhs) return;
  const long rhs = i / v5, site = i % v5;
  const int s = (int)(site % d.ls);
  const long col = site - s;
  const double2 *r = R + rhs * 4 * v5;
  double2 *y = Y + rhs * 4 * v5;
  for (int a = 0; a < 4; a++) {
    cx<double> v = ldc(r, a * v5 + site);
    if (a < 2) {  // P+ from s-1
      if (s > 0) v = v + ldc(r, a * v5 + site - 1);
      if (s == 0) v = v + cmul(cx<double>{c1.x, c1.y}, ldc(r, a * v5 + col + d.ls - 1));
    } else {  // P- from s+1
      if (s + 1 < d.ls) v = v + ldc(r, a * v5 + site + 1);
      if (s == d.ls - 1) v = v + cmul(cx<double>{c2.x, c2.y}, ldc(r, a * v5 + col));
    }
    st(y, a * v5 + site, v);
  }
}

// Phi += 2R - Y
__global__ __launch_bounds__(BLK) void k_wk_post(long n, const double2 *R, const double2 *Y,
                                                 double2 *Phi) {
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= n) return;
  const double2 r = R[i], y = Y[i], p = Phi[i];
  Phi[i] = make_double2(p.x + (2.0 * r.x - y.x), p.y + (2.0 * r.y - y.y));
}

// Phi = T + R + P- cA (T - R)(sA) + P+ cB (T - R)(sB)   (M^dagger)
__global__ __launch_bounds__(BLK) void k_wkd_post(const Dims d, int nrhs, const double2 *R,
                                                  const double2 *T, double2 *Phi, double2 z1,
                                                  double2 z2) {
  const long v5 = d.v5();
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= v5 * nrhs) return;
  const long rhs = i / v5, site = i % v5;
  const int s = (int)(site % d.ls);
  const long col = site - s;
  const double2 *r = R + rhs * 4 * v5;
  const double2 *tt = T + rhs * 4 * v5;
  double2 *ph = Phi + rhs * 4 * v5;
  for (int a = 0; a < 4; a++) {
    cx<double> v = ldc(tt, a * v5 + site) + ldc(r, a * v5 + site);
    if (a >= 2) {  // P-: from s-1, wall s=1 <- s=Ls with z1
      if (s > 0) v = v + (ldc(tt, a * v5 + site - 1) - ldc(r, a * v5 + site - 1));
      if (s == 0) {
        const long q = a * v5 + col + d.ls - 1;
        v = v + cmul(cx<double>{z1.x, z1.y}, ldc(tt, q) - ldc(r, q));
      }
    } else {  // P+: from s+1, wall s=Ls <- s=1 with z2
      if (s + 1 < d.ls) v = v + (ldc(tt, a * v5 + site + 1) - ldc(r, a * v5 + site + 1));
      if (s == d.ls - 1) {
        const long q = a * v5 + col;
        v = v + cmul(cx<double>{z2.x, z2.y}, ldc(tt, q) - ldc(r, q));
      }
    }
    st(ph, a * v5 + site, v);
  }
}

// gamval(mu,a)/akappa and gamin(mu,a)-1 for mu = 1..3 (gammamatrices.F90:27-75)
__constant__ double kGre[3][4] = {{0, 0, 0, 0}, {-1, 1, 1, -1}, {0, 0, 0, 0}};
__constant__ double kGim[3][4] = {{-1, -1, 1, 1}, {0, 0, 0, 0}, {-1, 1, 1, -1}};
__constant__ int kGin[3][4] = {{3, 2, 1, 0}, {3, 2, 1, 0}, {2, 3, 0, 1}};

// Shamir force, streaming form.  A block holds nl whole s-lines (columns
// (x, y), Ls consecutive threads each, s fastest: every load of a spin plane
// is one contiguous run) and marches them through a chunk of t.  At each step
// a thread forms the three link terms of its 5-D site, whose neighbours are
// the site itself and x+mu: the t neighbour loaded at step t is the centre of
// step t+1, so per step a thread loads R and X2 at (x+1), (y+1) and (t+1) only.
// The Ls terms of each link are summed in LDS in increasing s (a fixed order,
// so results are identical run to run) and added into dSdpi.
//   link term (x, mu) = w1 sum_a Im(R0_a^* X1_a - R1_a^* X0_a)
//                     + w2 sum_a Im(g_mu,a (R0_a^* X1_b + R1_a^* X0_b)),  b = gamin(mu, a)
// with (R0, X0) at x and (R1, X1) at x+mu, w1 = fl32(tzi/2), w2 = +-tzi
// (derivs_module.F90:131-187).
//
// Each spin's products are summed in pairs before they join the sum over the
// spins (in one chain of 16 the error against 64 bits grew by 5%: 2.36e-16 ->
// 2.48e-16 at 16^3 x 48).  gamval(mu, a) / akappa is one of +-1, +-i (kGamE),
// and only the part of the product that it turns into an imaginary one counts.
// FULL forms the whole complex product all the same (the compiler keeps
// products with a literal 0): twice the FP64 operations, but in the single
// Shamir force the compiler then needs 128 registers, four waves per SIMD,
// against 152 and three (16^3 x 48 11.4 and 12.1 us, 24^3 x 32 19.6 and 20.2,
// 32^3 x 64 73.2 and 74.9).  The batches and the Wilson kernel's force run at
// three waves either way and take the short form (25 pairs at 16^3 x 48 212 and
// 215 us with the call, 12 at 24^3 x 32 214 and 218; Wilson force at 15^2 x 21 x
// 20 9.4 and 9.65).
template <int MU, bool FULL>
__device__ inline double derivs_term(const cx<double> R0[4], const cx<double> X0[4],
                                     const cx<double> R1[4], const cx<double> X1[4], double w1,
                                     double w2) {
  double sw = 0.0, sd = 0.0;
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const int b = kGamP[MU][a], e = kGamE[MU][a];
    if constexpr (FULL) {
      const cx<double> g{e == 0 ? 0.5 : e == 1 ? -0.5 : 0.0, e == 2 ? 0.5 : e == 3 ? -0.5 : 0.0};
      sw += cjmul(R0[a], X1[a]).i - cjmul(R1[a], X0[a]).i;
      sd += cmul(g, cjmul(R0[a], X1[b]) + cjmul(R1[a], X0[b])).i;
    } else {
      sw += (R0[a].r * X1[a].i - R0[a].i * X1[a].r) - (R1[a].r * X0[a].i - R1[a].i * X0[a].r);
      double z;
      if (e < 2)  // +-1: Im (R0_a^* X1_b + R1_a^* X0_b)
        z = (R0[a].r * X1[b].i - R0[a].i * X1[b].r) + (R1[a].r * X0[b].i - R1[a].i * X0[b].r);
      else        // +-i: Re
        z = (R0[a].r * X1[b].r + R0[a].i * X1[b].i) + (R1[a].r * X0[b].r + R1[a].i * X0[b].i);
      sd = (e & 1) ? sd - z : sd + z;
    }
  }
  return w1 * sw + (FULL ? w2 : 0.5 * w2) * sd;
}

// sum of v over each segment of w lanes (a power of two), valid in all of its
// lanes: the butterfly of lane exchanges with register moves down to
// 16 lanes (rotations of a row by 8 and 4 reach lane ^ 8 and ^ 4 when the step
// before has made the lanes ^ 8 equal)
__device__ inline double segment_sum(double v, unsigned w) {
  if (w >= 64) v = swap_add<true>(v);
  if (w >= 32) v = swap_add<false>(v);
  if (w >= 16) {
    v += dpp_value<0x128>(v);
    v += dpp_value<0x124>(v);
  } else if (w >= 8) {
    v += __shfl_xor(v, 4, 64);
  }
  if (w >= 4) v += dpp_value<0x4E>(v);
  if (w >= 2) v += dpp_value<0xB1>(v);
  return v;
}

// LDS x exchange of the marching batched derivs: a block's 4 waves are 4
// consecutive x of one y, so the x+1 neighbour of waves 0-2 is the centre of the
// next wave: each wave stores its centre (R and X2, 8 complex numbers per lane,
// 32 KB per block) and reads the next wave's instead of loading it; wave 3
// loads its own.
struct DXBuf {
  double2 (*b)[8][64];
  __device__ inline void put(unsigned w, unsigned ln, const cx<double> R[4],
                             const cx<double> X[4]) const {
#pragma unroll
    for (int a = 0; a < 4; a++) {
      b[w][a][ln] = make_double2(R[a].r, R[a].i);
      b[w][4 + a][ln] = make_double2(X[a].r, X[a].i);
    }
  }
  __device__ inline void get(unsigned w, unsigned ln, cx<double> R[4], cx<double> X[4]) const {
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const double2 r = b[w][a][ln], x = b[w][4 + a][ln];
      R[a] = {r.x, r.y};
      X[a] = {x.x, x.y};
    }
  }
};

// Ls <= 64: each s-line takes a segment of W lanes of one wave (W the
// smallest power of two >= Ls, lanes s >= Ls idle), so the sum over s is a
// butterfly of wave shuffles inside the segment (a fixed order, no LDS and no
// block barrier); segment lane 0 adds the three link terms into dSdpi.  The
// t march and loads are those of k_derivs_march below.
//
// WK 1, 2: the Wilson kernel's force.  Its extra terms (derivs_module.F90:
// 41-97, 198-410) are the same bilinear form between slices of R and of X2,
// masked to two spins, with the s-couplings' factors; summed over s they are
// the form of (R + Q R, X2) for iflag 0 (WK 1) and of (R, X2 + Q X2) for
// iflag 1 (WK 2).  The couplings come by wave shuffles from the loaded
// lines, so the whole force is this one pass: 15^2 x 21 x 20 takes 11 us
// (the s-sum without them 9.6) against 155 with a second kernel that walked
// the 2 Ls slice pairs of each link one after another.
template <int WK>
__global__ __launch_bounds__(BLK, 3) void k_derivs_seg(const Dims d, const double2 *__restrict__ R,
                                                    const double2 *__restrict__ X2, float tzi,
                                                    int iflag, unsigned wseg, unsigned tchunk,
                                                    double *ds, const WallCoef wall) {
  const unsigned lx = d.lx, ly = d.ly, lt = d.lt, ls = d.ls;
  const unsigned v2 = lx * ly, v3 = v2 * ls, v4 = v2 * lt, v5 = v4 * ls;
  const unsigned nl = BLK / wseg;           // lines per block
  const unsigned nb2 = (v2 + nl - 1) / nl;  // blocks per t-chunk
  const unsigned chunk = blockIdx.x / nb2, lb = blockIdx.x - chunk * nb2;
  const unsigned line = threadIdx.x / wseg, s = threadIdx.x - line * wseg;
  const unsigned col = lb * nl + line;  // 2-D site x + lx y
  const unsigned t0 = chunk * tchunk, t1 = min(t0 + tchunk, lt);
  const bool valid = s < ls && col < v2;
  const double w1 = (double)(tzi * 0.5f);  // tzi_real*real(akappa)
  const double w2 = (double)tzi * (iflag == 0 ? 1.0 : -1.0);
  unsigned x = 0, y = 0;
  if (col < v2) {
    x = col % lx;
    y = col / lx;
  }
  const unsigned xf = (x + 1 == lx) ? 0 : x + 1, yf = (y + 1 == ly) ? 0 : y + 1;
  const unsigned j = s + ls * col, jx = s + ls * (xf + lx * y), jy = s + ls * (x + lx * yf);
  const unsigned lane0 = (threadIdx.x & 63) - s;
  cx<double> R0[4], X0[4];
  if (valid) {
    ld_spinor(R, v5, j + v3 * t0, R0);
    ld_spinor(X2, v5, j + v3 * t0, X0);
  }
  if constexpr (WK == 1) add_couplings(R0, s, ls, lane0, wall);
  if constexpr (WK == 2) add_couplings(X0, s, ls, lane0, wall);
  for (unsigned t = t0; t < t1; t++) {
    double v[3] = {0.0, 0.0, 0.0};
    cx<double> Rx[4], Xx[4], Ry[4], Xy[4], Rt[4], Xt[4];
    if (valid) {
      // all six neighbour spinors of the step in flight together
      const unsigned tf = (t + 1 == lt) ? 0 : t + 1;
      ld_spinor(R, v5, jx + v3 * t, Rx);
      ld_spinor(X2, v5, jx + v3 * t, Xx);
      ld_spinor(R, v5, jy + v3 * t, Ry);
      ld_spinor(X2, v5, jy + v3 * t, Xy);
      ld_spinor(R, v5, j + v3 * tf, Rt);
      ld_spinor(X2, v5, j + v3 * tf, Xt);
    }
    if constexpr (WK == 1) {
      add_couplings(Rx, s, ls, lane0, wall);
      add_couplings(Ry, s, ls, lane0, wall);
      add_couplings(Rt, s, ls, lane0, wall);
    }
    if constexpr (WK == 2) {
      add_couplings(Xx, s, ls, lane0, wall);
      add_couplings(Xy, s, ls, lane0, wall);
      add_couplings(Xt, s, ls, lane0, wall);
    }
    if (valid) {
      v[0] = derivs_term<0, WK == 0>(R0, X0, Rx, Xx, w1, w2);
      v[1] = derivs_term<1, WK == 0>(R0, X0, Ry, Xy, w1, w2);
      v[2] = derivs_term<2, WK == 0>(R0, X0, Rt, Xt, w1, w2);
#pragma unroll
      for (int a = 0; a < 4; a++) {
        R0[a] = Rt[a];
        X0[a] = Xt[a];
      }
    }
    // every lane of the wave takes part (idle lanes add 0)
#pragma unroll
    for (int mu = 0; mu < 3; mu++) v[mu] = segment_sum(v[mu], wseg);
    if (s == 0 && col < v2) {
#pragma unroll
      for (int mu = 0; mu < 3; mu++) ds[(long)mu * v4 + col + v2 * t] += v[mu];
    }
  }
}

// pairs of one batched launch, passed by value: no copy to the device, and no
// wait for one
constexpr int DPAIRS = 32;
struct DerivPairs {
  DerivPair p[DPAIRS];
};

// k_derivs_seg over several (R, X2) pairs in one launch, one t step per
// thread: blockIdx.y is the pair, so the GPU sweeps the pairs in order with
// every neighbour line shared in L2 by the blocks of the same pair (a thread
// looping over the pairs instead let neighbouring waves drift onto different
// pairs and ran at 2.3 TB/s).  Each block writes its links' terms of its pair
// to part[pair][mu][t][y][x]; k_derivs_sum_pairs adds the pairs in order into
// dSdpi.  The force sums derivs over the poles of a rational approximation
// (qmrherm_module.F90:143-181); one launch over all of them reads each
// pair's fields once like separate calls but fills the GPU on lattices whose
// single call cannot (25 MB per pair at 16^3 x 48).
// Bound by memory: 629 MB for 25 pairs there, 101 us at the copy rate.  Blocks
// go to the XCDs round robin, so XCD k takes the k-th eighth of a pair's
// (t, y, x): neighbours in y and most in t are lines of its own L2 (in launch
// order every line was fetched by up to four XCDs: 191 us at 16^3 x 48 with 25
// pairs, so 156; k_derivs_march_batch takes 143).
__global__ __launch_bounds__(BLK, 3) void k_derivs_seg_batch(const Dims d, const DerivPairs pairs,
                                                          unsigned wseg, unsigned nb, double *part) {
  const unsigned lx = d.lx, ly = d.ly, lt = d.lt, ls = d.ls;
  const unsigned v2 = lx * ly, v3 = v2 * ls, v4 = v2 * lt, v5 = v4 * ls;
  const unsigned nl = BLK / wseg;           // lines per block
  const unsigned nb2 = (v2 + nl - 1) / nl;  // blocks per t slice
  // gridDim.x is nb rounded up to a multiple of 8
  const unsigned b = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (b >= nb) return;
  const unsigned t = b / nb2, lb = b - t * nb2;
  const unsigned line = threadIdx.x / wseg, s = threadIdx.x - line * wseg;
  const unsigned col = lb * nl + line;  // 2-D site x + lx y
  const bool valid = s < ls && col < v2;
  const DerivPair P = pairs.p[blockIdx.y];
  unsigned x = 0, y = 0;
  if (col < v2) {
    x = col % lx;
    y = col / lx;
  }
  const unsigned xf = (x + 1 == lx) ? 0 : x + 1, yf = (y + 1 == ly) ? 0 : y + 1;
  const unsigned tf = (t + 1 == lt) ? 0 : t + 1;
  const unsigned j = s + ls * col + v3 * t, jx = s + ls * (xf + lx * y) + v3 * t;
  const unsigned jy = s + ls * (x + lx * yf) + v3 * t, jt = s + ls * col + v3 * tf;
  double v[3] = {0.0, 0.0, 0.0};
  cx<double> R0[4], X0[4], Rx[4], Xx[4], Ry[4], Xy[4], Rt[4], Xt[4];
  if (valid) {
    ld_spinor(P.r, v5, j, R0);
    ld_spinor(P.x2, v5, j, X0);
    ld_spinor(P.r, v5, jx, Rx);
    ld_spinor(P.x2, v5, jx, Xx);
    ld_spinor(P.r, v5, jy, Ry);
    ld_spinor(P.x2, v5, jy, Xy);
    ld_spinor(P.r, v5, jt, Rt);
    ld_spinor(P.x2, v5, jt, Xt);
  }
  if (valid) {
    v[0] = derivs_term<0, false>(R0, X0, Rx, Xx, P.w1, P.w2);
    v[1] = derivs_term<1, false>(R0, X0, Ry, Xy, P.w1, P.w2);
    v[2] = derivs_term<2, false>(R0, X0, Rt, Xt, P.w1, P.w2);
  }
  // every lane of the wave takes part (idle lanes add 0)
#pragma unroll
  for (int mu = 0; mu < 3; mu++) v[mu] = segment_sum(v[mu], wseg);
  if (s == 0 && col < v2) {
    double *o = part + (long)blockIdx.y * 3 * v4;
#pragma unroll
    for (int mu = 0; mu < 3; mu++) o[(long)mu * v4 + col + v2 * t] = v[mu];
  }
}

// The same for 64-lane segments (32 < Ls <= 64) with Lx % 4 == 0: a block is 4
// consecutive x of one y, so x+1 of waves 0-2 comes through LDS, and it marches
// tchunk t steps, the t+1 line of a step being the centre of the next: 2.25
// instead of 3.25 lines loaded per line.  XCD k takes pair 8 g + k of each
// group of 8 whole (no line is fetched twice across XCDs), and the k-th eighth
// of each pair left over.  25 pairs, one call: 32^3 x 64 1.89 -> 1.53 ms, 16^3 x
// 48 185 -> 180 us against k_derivs_seg_batch with the LDS exchange, which it
// replaces.  Without the exchange (other Ls) the march did not pay: 24^3 x 32
// 382 and 388 us.
__global__ __launch_bounds__(BLK, 3) void k_derivs_march_batch(const Dims d, const DerivPairs pairs,
                                                            unsigned nb, unsigned npair,
                                                            unsigned tchunk, double *part) {
  const unsigned lx = d.lx, ly = d.ly, lt = d.lt, ls = d.ls;
  const unsigned v2 = lx * ly, v3 = v2 * ls, v4 = v2 * lt, v5 = v4 * ls;
  const unsigned nb2 = v2 / 4;  // blocks per t chunk
  // whole groups of 8 pairs: XCD k takes pair 8 g + k; the others: XCD k takes
  // the k-th eighth of each pair
  const unsigned xcd = blockIdx.x & 7, q = blockIdx.x >> 3, whole = npair & ~7u;
  unsigned b, pair;
  if (q < (whole >> 3) * nb) {
    pair = q / nb;
    b = q - pair * nb;
    pair = pair * 8 + xcd;
  } else {
    const unsigned per = (nb + 7) / 8, q2 = q - (whole >> 3) * nb;
    pair = q2 / per;
    b = xcd * per + (q2 - pair * per);
    pair += whole;
    if (b >= nb) return;
  }
  const unsigned chunk = b / nb2, lb = b - chunk * nb2;
  const unsigned t0 = chunk * tchunk, t1 = min(t0 + tchunk, lt);
  const unsigned w = threadIdx.x >> 6, s = threadIdx.x & 63;
  const unsigned col = lb * 4 + w;  // 2-D site x + lx y
  const bool valid = s < ls;
  const DerivPair P = pairs.p[pair];
  const unsigned x = col % lx, y = col / lx;
  const unsigned xf = (x + 1 == lx) ? 0 : x + 1, yf = (y + 1 == ly) ? 0 : y + 1;
  const unsigned j = s + ls * col, jx = s + ls * (xf + lx * y), jy = s + ls * (x + lx * yf);
  __shared__ double2 xraw[4][8][64];
  const DXBuf xb{xraw};
  cx<double> R0[4], X0[4];
  if (valid) {
    ld_spinor(P.r, v5, j + v3 * t0, R0);
    ld_spinor(P.x2, v5, j + v3 * t0, X0);
  }
  double *o = part + (long)pair * 3 * v4;
  for (unsigned t = t0; t < t1; t++) {
    const unsigned tf = (t + 1 == lt) ? 0 : t + 1;
    double v[3] = {0.0, 0.0, 0.0};
    cx<double> Rx[4], Xx[4], Ry[4], Xy[4], Rt[4], Xt[4];
    if (valid) {
      if (w == 3) {
        ld_spinor(P.r, v5, jx + v3 * t, Rx);
        ld_spinor(P.x2, v5, jx + v3 * t, Xx);
      }
      ld_spinor(P.r, v5, jy + v3 * t, Ry);
      ld_spinor(P.x2, v5, jy + v3 * t, Xy);
      ld_spinor(P.r, v5, j + v3 * tf, Rt);
      ld_spinor(P.x2, v5, j + v3 * tf, Xt);
    }
    if (t > t0) __syncthreads();  // the reads of the step before are done
    if (valid) xb.put(w, s, R0, X0);
    __syncthreads();
    if (valid && w < 3) xb.get(w + 1, s, Rx, Xx);
    if (valid) {
      v[0] = derivs_term<0, false>(R0, X0, Rx, Xx, P.w1, P.w2);
      v[1] = derivs_term<1, false>(R0, X0, Ry, Xy, P.w1, P.w2);
      v[2] = derivs_term<2, false>(R0, X0, Rt, Xt, P.w1, P.w2);
#pragma unroll
      for (int a = 0; a < 4; a++) {
        R0[a] = Rt[a];
        X0[a] = Xt[a];
      }
    }
    // every lane of the wave takes part (idle lanes add 0)
#pragma unroll
    for (int mu = 0; mu < 3; mu++) v[mu] = wave_sum(v[mu]);
    if (s == 0) {
#pragma unroll
      for (int mu = 0; mu < 3; mu++) o[(long)mu * v4 + col + v2 * t] = v[mu];
    }
  }
}

// dSdpi[e] += sum over the pairs, in pair order, of part[pair][e]; 8 loads in
// flight per thread (one after another they took 11 us for 25 pairs at 16^3)
__global__ __launch_bounds__(64) void k_derivs_sum_pairs(long n, int npair,
                                                         const double *__restrict__ part,
                                                         double *ds) {
  const long e = (long)blockIdx.x * 64 + threadIdx.x;
  if (e >= n) return;
  constexpr int U = 8;
  const double d0 = ds[e];
  double v = 0.0;
  for (int k0 = 0; k0 < npair; k0 += U) {
    double a[U];
#pragma unroll
    for (int u = 0; u < U; u++) a[u] = part[(long)min(k0 + u, npair - 1) * n + e];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + u < npair) v += a[u];
  }
  ds[e] = d0 + v;
}

__global__ __launch_bounds__(BLK) void k_derivs_march(const Dims d, const double2 *__restrict__ R,
                                                      const double2 *__restrict__ X2, float tzi,
                                                      int iflag, unsigned nl, unsigned tchunk,
                                                      double *ds) {
  __shared__ double terms[2][3][BLK];
  const unsigned lx = d.lx, ly = d.ly, lt = d.lt, ls = d.ls;
  const unsigned v2 = lx * ly, v3 = v2 * ls, v4 = v2 * lt, v5 = v4 * ls;
  const unsigned nb2 = (v2 + nl - 1) / nl;  // blocks per t-chunk
  const unsigned chunk = blockIdx.x / nb2, lb = blockIdx.x - chunk * nb2;
  const unsigned line = threadIdx.x / ls, s = threadIdx.x - line * ls;
  const unsigned col = lb * nl + line;  // 2-D site x + lx y
  const unsigned t0 = chunk * tchunk, t1 = min(t0 + tchunk, lt);
  const bool valid = line < nl && col < v2;
  const double w1 = (double)(tzi * 0.5f);  // tzi_real*real(akappa)
  const double w2 = (double)tzi * (iflag == 0 ? 1.0 : -1.0);
  unsigned x = 0, y = 0;
  if (valid) {
    x = col % lx;
    y = col / lx;
  }
  const unsigned xf = (x + 1 == lx) ? 0 : x + 1, yf = (y + 1 == ly) ? 0 : y + 1;
  const unsigned j = s + ls * col, jx = s + ls * (xf + lx * y), jy = s + ls * (x + lx * yf);
  cx<double> R0[4], X0[4];
  if (valid) {
    ld_spinor(R, v5, j + v3 * t0, R0);
    ld_spinor(X2, v5, j + v3 * t0, X0);
  }
  for (unsigned t = t0; t < t1; t++) {
    const unsigned pb = (t - t0) & 1;
    if (valid) {
      const unsigned tf = (t + 1 == lt) ? 0 : t + 1;
      cx<double> R1[4], X1[4], Rt[4], Xt[4];
      ld_spinor(R, v5, jx + v3 * t, R1);
      ld_spinor(X2, v5, jx + v3 * t, X1);
      terms[pb][0][threadIdx.x] = derivs_term<0, true>(R0, X0, R1, X1, w1, w2);
      ld_spinor(R, v5, jy + v3 * t, R1);
      ld_spinor(X2, v5, jy + v3 * t, X1);
      terms[pb][1][threadIdx.x] = derivs_term<1, true>(R0, X0, R1, X1, w1, w2);
      ld_spinor(R, v5, j + v3 * tf, Rt);
      ld_spinor(X2, v5, j + v3 * tf, Xt);
      terms[pb][2][threadIdx.x] = derivs_term<2, true>(R0, X0, Rt, Xt, w1, w2);
#pragma unroll
      for (int a = 0; a < 4; a++) {
        R0[a] = Rt[a];
        X0[a] = Xt[a];
      }
    }
    // one barrier per step: buffer pb is written again two steps later, after
    // the next step's barrier, by when its readers below are done
    __syncthreads();
    for (unsigned r = threadIdx.x; r < 3 * nl; r += blockDim.x) {  // 3 nl > blockDim when Ls < 3
      const unsigned mu = r / nl, ln = r - mu * nl, c = lb * nl + ln;
      if (c < v2) {
        double sum = 0.0;
        for (unsigned k = 0; k < ls; k++) sum += terms[pb][mu][ln * ls + k];
        ds[(long)mu * v4 + c + v2 * t] += sum;
      }
    }
  }
}

// any Ls: one thread per link, serial over s and spin (used when an s-line
// does not fit one block)
__global__ __launch_bounds__(BLK) void k_derivs(const Dims d, const double2 *__restrict__ R,
                                                const double2 *__restrict__ X2, float tzi,
                                                int iflag, double *ds) {
  const long v4 = d.v4(), v5 = d.v5();
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= v4 * 3) return;
  const int mu = (int)(i / v4);
  const long s4 = i % v4;
  const int x = (int)(s4 % d.lx), y = (int)((s4 / d.lx) % d.ly), t = (int)(s4 / ((long)d.lx * d.ly));
  int xf = x, yf = y, tf = t;
  if (mu == 0) xf = (x + 1 == d.lx) ? 0 : x + 1;
  if (mu == 1) yf = (y + 1 == d.ly) ? 0 : y + 1;
  if (mu == 2) tf = (t + 1 == d.lt) ? 0 : t + 1;
  const long f4 = xf + (long)d.lx * (yf + (long)d.ly * tf);
  const long c0 = s4 * d.ls, c1 = f4 * d.ls;
  const double w1 = (double)(tzi * 0.5f);  // tzi_real*real(akappa)
  const double w2 = (double)tzi * (iflag == 0 ? 1.0 : -1.0);
  double acc = 0.0;
  for (int a = 0; a < 4; a++) {
    const int b = kGin[mu][a];
    const cx<double> g{0.5 * kGre[mu][a], 0.5 * kGim[mu][a]};
    double sw = 0.0, sd = 0.0;
    for (int s = 0; s < d.ls; s++) {
      const cx<double> r0 = ldc(R, a * v5 + c0 + s), r1 = ldc(R, a * v5 + c1 + s);
      const cx<double> xa0 = ldc(X2, a * v5 + c0 + s), xa1 = ldc(X2, a * v5 + c1 + s);
      const cx<double> xb0 = ldc(X2, b * v5 + c0 + s), xb1 = ldc(X2, b * v5 + c1 + s);
      sw += cjmul(r0, xa1).i - cjmul(r1, xa0).i;
      sd += cmul(g, cjmul(r0, xb1) + cjmul(r1, xb0)).i;
    }
    acc = acc + w1 * sw;
    acc = acc + w2 * sd;
  }
  ds[i] += acc;
}

// Wilson-kernel extra force terms (derivs_module.F90:41-97, 198-410) where an
// s-line does not fit one wave (Ls > 64): the s-couplings of the
// Wilson-kernel operator, each a derivSlice() between a slice of R and a slice
// of X2 with spin masks and a complex multiplier.
struct SlicePair {
  int sl, sr;       // 0-based s of the R slice and the X2 slice
  int l0, l1;       // R spins kept [l0, l1)
  int r0, r1;       // X2 spins kept [r0, r1)
  double cr, ci;    // cmult
};

__global__ __launch_bounds__(BLK) void k_derivs_wilson_extra(const Dims d, const double2 *__restrict__ R,
                                                             const double2 *__restrict__ X2,
                                                             float tzi, int iflag,
                                                             const SlicePair *pairs, int npairs,
                                                             double *ds) {
  const long v4 = d.v4(), v5 = d.v5();
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= v4 * 3) return;
  const int mu = (int)(i / v4);
  const long s4 = i % v4;
  const int x = (int)(s4 % d.lx), y = (int)((s4 / d.lx) % d.ly), t = (int)(s4 / ((long)d.lx * d.ly));
  int xf = x, yf = y, tf = t;
  if (mu == 0) xf = (x + 1 == d.lx) ? 0 : x + 1;
  if (mu == 1) yf = (y + 1 == d.ly) ? 0 : y + 1;
  if (mu == 2) tf = (t + 1 == d.lt) ? 0 : t + 1;
  const long f4 = xf + (long)d.lx * (yf + (long)d.ly * tf);
  const double w1 = (double)(tzi * 0.5f);
  const double w2 = (double)(tzi * (iflag == 1 ? -1.0f : 1.0f));
  double acc = ds[i];
  for (int k = 0; k < npairs; k++) {
    const SlicePair P = pairs[k];
    const cx<double> cm{P.cr, P.ci};
    const long l0 = s4 * d.ls + P.sl, l1 = f4 * d.ls + P.sl;
    const long r0 = s4 * d.ls + P.sr, r1 = f4 * d.ls + P.sr;
    for (int a = 0; a < 4; a++) {
      const bool la = a >= P.l0 && a < P.l1;
      const cx<double> zero{0.0, 0.0};
      const cx<double> L0 = la ? ldc(R, a * v5 + l0) : zero, L1 = la ? ldc(R, a * v5 + l1) : zero;
      const bool ra = a >= P.r0 && a < P.r1;
      const cx<double> Ra0 = ra ? ldc(X2, a * v5 + r0) : zero, Ra1 = ra ? ldc(X2, a * v5 + r1) : zero;
      const double v = cmul(cm, cjmul(L0, Ra1)).i - cmul(cm, cjmul(L1, Ra0)).i;
      acc += w1 * v;
      const int b = kGin[mu][a];
      const bool rb = b >= P.r0 && b < P.r1;
      const cx<double> Rb0 = rb ? ldc(X2, b * v5 + r0) : zero, Rb1 = rb ? ldc(X2, b * v5 + r1) : zero;
      const cx<double> g{0.5 * kGre[mu][a], 0.5 * kGim[mu][a]};
      acc += w2 * cmul(cmul(cm, g), cjmul(L0, Rb1) + cjmul(L1, Rb0)).i;
    }
  }
  ds[i] = acc;
}

}  // namespace

static int launch_derivs_wk(const Dims &d, const double2 *R, const double2 *X2, double anum,
                            int iflag, int wk, const WallCoef &wall, double *dsdpi, hipStream_t s);

int launch_derivs_wilson(const Dims &d, const double2 *R, const double2 *X2, double anum,
                         int iflag, float am, int imass, double *dsdpi, void *pair_buf,
                         hipStream_t s) {
  THR_CHECK(imass == 1 || imass == 3, THR_ERR_ARG, "Wilson kernel supports imass 1 and 3");
  const int L = d.ls;
  const double m = (double)am;
  // derivsWilsonMass (derivs_module.F90:198-249): cmplx(-am,0) | cmplx(0,-am), then
  // cmplx(-am,0) | cmplx(0,am)
  const double c1r = imass == 1 ? -m : 0.0, c1i = imass == 1 ? 0.0 : -m;
  const double c2r = imass == 1 ? -m : 0.0, c2i = imass == 1 ? 0.0 : m;
  if (L <= 64) {
    // an s-line fits one wave: the extra terms join the s-sum.  On R (iflag 0)
    // the walls' factors are conj(c2), conj(c1), which are c1, c2
    const WallCoef w{c1r, c1i, c2r, c2i};
    return launch_derivs_wk(d, R, X2, anum, iflag, iflag == 0 ? 1 : iflag == 1 ? 2 : 0, w, dsdpi, s);
  }
  int rc = launch_derivs(d, R, X2, anum, iflag, dsdpi, s);
  if (rc) return rc;
  std::vector<SlicePair> pr;
  if (iflag == 1) {
    pr.push_back({0, L - 1, 0, 4, 0, 2, c1r, c1i});   // DP: L all, R spins 1:2
    pr.push_back({L - 1, 0, 0, 4, 2, 4, c2r, c2i});   // DM: L all, R spins 3:4
  } else if (iflag == 0) {
    pr.push_back({0, L - 1, 2, 4, 0, 4, c1r, c1i});   // MD: L spins 3:4, R all
    pr.push_back({L - 1, 0, 0, 2, 0, 4, c2r, c2i});   // PD: L spins 1:2, R all
  }
  // s-couplings (derivs_module.F90:73-81)
  for (int il = 0; il < L - 1; il++) {
    if (iflag == 1) {
      pr.push_back({il, il + 1, 0, 4, 2, 4, 1.0, 0.0});  // DM
      pr.push_back({il + 1, il, 0, 4, 0, 2, 1.0, 0.0});  // DP
    } else if (iflag == 0) {
      pr.push_back({il, il + 1, 0, 2, 0, 4, 1.0, 0.0});  // PD
      pr.push_back({il + 1, il, 2, 4, 0, 4, 1.0, 0.0});  // MD
    }
  }
  if (pr.empty()) return THR_OK;
  THR_HIP(hipMemcpyAsync(pair_buf, pr.data(), sizeof(SlicePair) * pr.size(), hipMemcpyHostToDevice, s));
  const float tzi = 2.0f * (float)anum;
  const unsigned nb = (unsigned)((d.v4() * 3 + BLK - 1) / BLK);
  hipLaunchKernelGGL(k_derivs_wilson_extra, dim3(nb), dim3(BLK), 0, s, d, R, X2, tzi, iflag,
                     (const SlicePair *)pair_buf, (int)pr.size(), dsdpi);
  THR_HIP(hipGetLastError());
  // pr must stay alive until the copy is done
  THR_HIP(hipStreamSynchronize(s));
  return THR_OK;
}

long wilson_blocks(const Dims &d) {
  if (d.ls > 64) return (d.v5() + BLK - 1) / BLK;
  const long nl = BLK / segment(d.ls);
  return ((long)d.lx * d.ly + nl - 1) / nl * d.lt;
}

int launch_wilson_epi(DslashLaunch L, hipStream_t s) {
  THR_CHECK(L.imass == 1 || L.imass == 3, THR_ERR_ARG, "Wilson kernel supports imass 1 and 3");
  THR_CHECK(L.d.ls <= 64, THR_ERR_ARG, "fused Wilson kernel: Ls above 64");
  THR_CHECK(4 * L.d.v5() * (long)sizeof(double2) < (1L << 32), THR_ERR_SIZE,
            "spinor too large for the Wilson kernel");
  const double m = (double)L.am[0];
  // -am | -i am at s = 1 (dirac.F90:274-278, 602-606), -am | +i am at s = Ls
  // (287-291, 615-619)
  const WallCoef w = L.imass == 1 ? WallCoef{-m, 0.0, -m, 0.0} : WallCoef{0.0, -m, 0.0, m};
  THR_CHECK(L.mode != EPI_TRES && !L.in_stride, THR_ERR_ARG, "Wilson kernel: no such epilogue");
  THR_CHECK(!L.scal == !L.fsum && (!L.scal || (L.nrhs == 1 && L.sst)), THR_ERR_ARG,
            "Wilson kernel: a fused sum comes with its scalar step");
  THR_CHECK(L.mode != EPI_HPREC || (!L.dagger && L.x), THR_ERR_ARG, "direction epilogue: M with its vector");
  const dim3 grid((unsigned)wilson_blocks(L.d) + (L.scal ? SCAL_LEAD : 0u), (unsigned)L.nrhs);
  const unsigned seg = segment(L.d.ls);
#define THR_GO(D, M) hipLaunchKernelGGL((k_wilson<D, M>), grid, dim3(BLK), 0, s, L, seg, w)
#define THR_DAG(M)         \
  do {                     \
    if (L.dagger)          \
      THR_GO(true, M);     \
    else                   \
      THR_GO(false, M);    \
  } while (0)
  switch (L.mode) {
    case EPI_STORE: THR_DAG(EPI_STORE); break;
    case EPI_NORM: THR_DAG(EPI_NORM); break;
    case EPI_DOTW: THR_DAG(EPI_DOTW); break;
    case EPI_HREC: THR_DAG(EPI_HREC); break;
    case EPI_HPREC: THR_GO(false, EPI_HPREC); break;
    default: THR_DAG(EPI_CG); break;
  }
#undef THR_DAG
#undef THR_GO
  THR_HIP(hipGetLastError());
  return THR_OK;
}

int launch_dslash_wilson(const Dims &d, int nrhs, int dagger, int imass, float am, float am3,
                         const double2 *in, double2 *out, const double2 *links, double2 *tmp,
                         hipStream_t s) {
  THR_CHECK(imass == 1 || imass == 3, THR_ERR_ARG, "Wilson kernel supports imass 1 and 3");
  if (d.ls <= 64) {
    DslashLaunch F{};
    F.d = d;
    F.nrhs = nrhs;
    F.dagger = dagger;
    F.imass = imass;
    F.am3 = am3;
    F.am[0] = am;
    F.in = in;
    F.out = out;
    F.links = links;
    F.mode = EPI_STORE;
    return launch_wilson_epi(F, s);
  }
  THR_CHECK(tmp, THR_ERR_ARG, "Wilson kernel: scratch spinor required");
  const long n = d.v5() * nrhs;
  const unsigned nb = (unsigned)((n + BLK - 1) / BLK);
  DslashLaunch L{};
  L.d = d;
  L.nrhs = nrhs;
  L.prec = P64;
  L.dagger = dagger;
  L.imass = imass;
  L.am3 = am3;
  L.links = links;
  L.mode = EPI_STORE;
  L.wilson4d = 1;
  const double m = (double)am;
  if (!dagger) {
    // c1 = -am | -i am (dirac.F90:274-278), c2 = -am | +i am (287-291)
    const double2 c1 = imass == 1 ? make_double2(-m, 0.0) : make_double2(0.0, -m);
    const double2 c2 = imass == 1 ? make_double2(-m, 0.0) : make_double2(0.0, m);
    hipLaunchKernelGGL(k_wk_pre, dim3(nb), dim3(BLK), 0, s, d, nrhs, in, tmp, c1, c2);
    THR_HIP(hipGetLastError());
    L.in = tmp;
    L.out = out;
    int rc = launch_dslash(L, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_wk_post, dim3((unsigned)((n * 4 + BLK - 1) / BLK)), dim3(BLK), 0, s,
                       n * 4, in, tmp, out);
  } else {
    L.in = in;
    L.out = tmp;
    int rc = launch_dslash(L, s);
    if (rc) return rc;
    // zkappa: -am | -i am (dirac.F90:602-606), -am | +i am (615-619)
    const double2 z1 = imass == 1 ? make_double2(-m, 0.0) : make_double2(0.0, -m);
    const double2 z2 = imass == 1 ? make_double2(-m, 0.0) : make_double2(0.0, m);
    hipLaunchKernelGGL(k_wkd_post, dim3(nb), dim3(BLK), 0, s, d, nrhs, in, tmp, out, z1, z2);
  }
  THR_HIP(hipGetLastError());
  return THR_OK;
}

DerivPair derivs_pair(const double2 *R, const double2 *X2, double anum, int iflag) {
  const float tzi = 2.0f * (float)anum;  // real :: tzi_real = 2*real(anum)
  return DerivPair{R, X2, (double)(tzi * 0.5f), (double)tzi * (iflag == 0 ? 1.0 : -1.0)};
}

// the batched derivs' march with the LDS x exchange applies with 64-lane segments (32 < Ls
// <= 64) when a block's 4 lines are 4 consecutive x of one y (Lx % 4 == 0);
// THR_DERIVS_LDSX=0 switches it off
static bool derivs_lds_x(const Dims &d, unsigned wseg) {
  if (const char *e = std::getenv("THR_DERIVS_LDSX"))
    if (std::atoi(e) == 0) return false;
  return wseg == 64 && d.lx % 4 == 0;
}

int launch_derivs_batch(const Dims &d, int npair, const DerivPair *pairs, double *part,
                        double *dsdpi, hipStream_t s) {
  THR_CHECK(npair >= 1 && npair <= 65535, THR_ERR_ARG, "derivs batch: 1..65535 pairs");
  THR_CHECK(d.v5() * 4 < (1L << 31), THR_ERR_SIZE, "derivs: 4*V5 must be below 2^31");
  THR_CHECK(d.ls <= 64, THR_ERR_ARG, "derivs batch: Ls above 64");
  THR_CHECK(part, THR_ERR_ARG, "derivs batch: NULL buffer");
  const long n = 3 * d.v4();
  const unsigned w = segment(d.ls);
  const unsigned nl = BLK / w;
  const unsigned v2 = (unsigned)(d.lx * d.ly);
  const bool march = derivs_lds_x(d, w);
  for (int k0 = 0; k0 < npair; k0 += DPAIRS) {
    const int np = std::min(DPAIRS, npair - k0);
    DerivPairs P{};
    std::copy(pairs + k0, pairs + k0 + np, P.p);
    double *out = part + (long)k0 * n;
    if (march) {
      // t steps per block: up to 8 as long as the launch keeps 2048 blocks
      const long steps = (long)(v2 / 4) * d.lt * np;
      const unsigned tc = (unsigned)std::max(1L, std::min({8L, (long)d.lt, steps / 2048}));
      const unsigned nb = (v2 / 4) * ((d.lt + tc - 1) / tc);
      const unsigned grid = 8 * ((unsigned)(np / 8) * nb + (unsigned)(np % 8) * ((nb + 7) / 8));
      hipLaunchKernelGGL(k_derivs_march_batch, dim3(grid), dim3(BLK), 0, s, d, P, nb, (unsigned)np,
                         tc, out);
    } else {
      const unsigned nb = ((v2 + nl - 1) / nl) * (unsigned)d.lt;
      hipLaunchKernelGGL(k_derivs_seg_batch, dim3((nb + 7) / 8 * 8, (unsigned)np), dim3(BLK), 0, s,
                         d, P, w, nb, out);
    }
  }
  hipLaunchKernelGGL(k_derivs_sum_pairs, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, n, npair,
                     (const double *)part, dsdpi);
  THR_HIP(hipGetLastError());
  return THR_OK;
}

int launch_derivs(const Dims &d, const double2 *R, const double2 *X2, double anum, int iflag,
                  double *dsdpi, hipStream_t s) {
  return launch_derivs_wk(d, R, X2, anum, iflag, 0, WallCoef{}, dsdpi, s);
}

// wk: the Wilson kernel's couplings on R (1) or X2 (2), Ls <= 64 only
static int launch_derivs_wk(const Dims &d, const double2 *R, const double2 *X2, double anum,
                            int iflag, int wk, const WallCoef &wall, double *dsdpi,
                            hipStream_t s) {
  const float tzi = 2.0f * (float)anum;  // real :: tzi_real = 2*real(anum)
  THR_CHECK(d.v5() * 4 < (1L << 31), THR_ERR_SIZE, "derivs: 4*V5 must be below 2^31");
  // one t step per thread: marching longer t-chunks reuses the t neighbour
  // from registers but leaves fewer threads in flight, and measured slower
  // (32^3 x 64: 76-80 us at one step, 82-90 us at 2-16; 16^3 x 48: 12-13
  // against 14-44 us) (THR_DERIVS_TCHUNK overrides)
  unsigned tchunk = 1;
  if (const char *e = std::getenv("THR_DERIVS_TCHUNK"))
    tchunk = (unsigned)std::max(1, std::min(d.lt, std::atoi(e)));
  // resident blocks per CU capped by LDS padding (THR_DERIVS_OCC = k: k + 1
  // blocks): fewer resident s-lines per XCD keep the x+1 / y+1 neighbours in L2
  size_t pad = 0;
  if (const char *e = std::getenv("THR_DERIVS_OCC")) {
    const int k = std::max(0, std::min(3, std::atoi(e)));
    if (k > 0) pad = (size_t)(160 * 1024 / (k + 1)) & ~(size_t)511;
    if (pad > 65536) pad = 65536;
  }
  const unsigned nchunk = (d.lt + tchunk - 1) / tchunk;
  const unsigned v2 = (unsigned)d.lx * d.ly;
  if (d.ls <= 64) {
    const unsigned w = segment(d.ls);
    const unsigned nl = BLK / w;
    const unsigned nb = ((v2 + nl - 1) / nl) * nchunk;
#define THR_SEG(K) \
  hipLaunchKernelGGL(K, dim3(nb), dim3(BLK), pad, s, d, R, X2, tzi, iflag, w, tchunk, dsdpi, wall)
    if (wk == 1)
      THR_SEG(k_derivs_seg<1>);
    else if (wk == 2)
      THR_SEG(k_derivs_seg<2>);
    else
      THR_SEG(k_derivs_seg<0>);
#undef THR_SEG
    THR_HIP(hipGetLastError());
    return THR_OK;
  }
  if (d.ls <= BLK) {
    // whole s-lines per block, summed in LDS
    const unsigned nl = BLK / d.ls;
    const unsigned nb = ((v2 + nl - 1) / nl) * nchunk;
    hipLaunchKernelGGL(k_derivs_march, dim3(nb), dim3(nl * d.ls), 0, s, d, R, X2, tzi, iflag, nl,
                       tchunk, dsdpi);
    THR_HIP(hipGetLastError());
    return THR_OK;
  }
  const unsigned nb = (unsigned)((d.v4() * 3 + BLK - 1) / BLK);
  hipLaunchKernelGGL(k_derivs, dim3(nb), dim3(BLK), 0, s, d, R, X2, tzi, iflag, dsdpi);
  THR_HIP(hipGetLastError());
  return THR_OK;
}

}  // namespace thr
