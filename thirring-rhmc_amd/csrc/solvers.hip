// Reference-faithful Krylov solvers with device-resident scalars.
//
// The reference runs every dot product through an MPI_AllReduce and a host
// round trip.  Here all scalars (alpha, beta, zeta recurrences, convergence
// window) live in a small device state struct.  One block at a time writes it,
// summing the per-block partials in a fixed order: the first block of the
// operator launch that follows, or a kernel of its own (krylov_scalars.h).  So
// results are deterministic and the host only polls a stop flag every few
// iterations.  Kernels of an iteration that starts after the stop flag was
// raised exit immediately, so the iteration counts and final vectors are
// exactly those of the reference's loop structure.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "krylov_scalars.h"
#include "solvers.h"

namespace thr {

// ---------------------------------------------------------------------------
// workspace: one set of device buffers and one stream per context; a thread
// works in the context it bound (thr_context_bind), else in the default one,
// so independent solves on different threads never share scratch memory
// ---------------------------------------------------------------------------
namespace {
struct Buf {
  void *p = nullptr;
  size_t n = 0;
  // a buffer that a call can do without: freed when another allocation of the
  // context fails, unless a call holds it
  bool spare = false, held = false;
};
}  // namespace

struct Context {
  std::map<int, Buf> ws;
  std::map<int, Buf> hws;  // pinned host buffers for small state transfers
  std::mutex mu;
  hipStream_t stream = nullptr;
  // hipGraph capture of solver blocks; off in created contexts, which run
  // next to other threads' allocations and copies (a stream capture is
  // invalidated by device-synchronising calls from any thread)
  bool graphs = true;
  // reliable updates of the mixed multishift's base residual: taken each time
  // the residual falls by this factor while the Krylov storage is FP32/FP16
  // (0: never); and how many the last solve in this context took
  double reliable = 0.1;
  int last_reliable = 0;
};

namespace {
Context g_default;
thread_local Context *t_ctx = nullptr;
Context &cur() { return t_ctx ? *t_ctx : g_default; }
}  // namespace

Context *context_create() {
  Context *c = new Context();
  c->graphs = false;
  return c;
}

bool context_graphs() { return cur().graphs; }
double context_reliable() { return cur().reliable; }
void context_set_reliable(double delta) { cur().reliable = delta; }
void context_note_reliable(int n) { cur().last_reliable = n; }
int context_last_reliable() { return cur().last_reliable; }

void context_destroy(Context *c) {
  if (!c) return;
  (void)hipDeviceSynchronize();
  for (auto &kv : c->ws)
    if (kv.second.p) (void)hipFree(kv.second.p);
  for (auto &kv : c->hws)
    if (kv.second.p) (void)hipHostFree(kv.second.p);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  if (t_ctx == c) t_ctx = nullptr;
  delete c;
}

void context_bind(Context *c) { t_ctx = c; }

// device memory for b, or null with no error left behind
static bool grow(Buf &b, size_t bytes) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
  b.n = 0;
  if (hipMalloc(&b.p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    b.p = nullptr;
    return false;
  }
  b.n = bytes;
  return true;
}

void *workspace(int slot, size_t bytes) {
  Context &c = cur();
  std::lock_guard<std::mutex> lk(c.mu);
  Buf &b = c.ws[slot];
  if (b.n < bytes && !grow(b, bytes)) {
    bool freed = false;
    for (auto &kv : c.ws) {
      Buf &o = kv.second;
      if (!o.spare || o.held || !o.p) continue;
      (void)hipFree(o.p);
      o.p = nullptr;
      o.n = 0;
      freed = true;
    }
    if (!freed || !grow(b, bytes)) {
      set_error("hipMalloc of workspace failed");
      return nullptr;
    }
  }
  return b.p;
}

void *spare_workspace(int slot, size_t bytes) {
  Context &c = cur();
  std::lock_guard<std::mutex> lk(c.mu);
  Buf &b = c.ws[slot];
  if (b.n < bytes) {
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    if (bytes > (free + b.n) / 4 || !grow(b, bytes)) return nullptr;
  }
  b.spare = b.held = true;
  return b.p;
}

void release_spare(int slot) {
  Context &c = cur();
  std::lock_guard<std::mutex> lk(c.mu);
  c.ws[slot].held = false;
}

void *host_workspace(int slot, size_t bytes) {
  Context &c = cur();
  std::lock_guard<std::mutex> lk(c.mu);
  Buf &b = c.hws[slot];
  if (b.n < bytes) {
    if (b.p) (void)hipHostFree(b.p);
    b.p = nullptr;
    b.n = 0;
    if (hipHostMalloc(&b.p, bytes, hipHostMallocDefault) != hipSuccess) {
      set_error("hipHostMalloc of host workspace failed");
      b.p = nullptr;
      return nullptr;
    }
    b.n = bytes;
  }
  return b.p;
}

size_t workspace_bytes() {
  Context &c = cur();
  std::lock_guard<std::mutex> lk(c.mu);
  size_t t = 0;
  for (auto &kv : c.ws) t += kv.second.n;
  return t;
}

double *partial_buffer(int nblocks) {
  return (double *)workspace(0, sizeof(double) * (size_t)nblocks);
}

hipStream_t default_stream() {
  Context &c = cur();
  // non-blocking: no implicit ordering with the legacy null stream, which
  // would break graph capture while another thread copies on it
  if (!c.stream) (void)hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking);
  return c.stream;
}

void release_workspace() {
  Context &c = cur();
  std::lock_guard<std::mutex> lk(c.mu);
  for (auto &kv : c.ws)
    if (kv.second.p) (void)hipFree(kv.second.p);
  c.ws.clear();
}

// ---------------------------------------------------------------------------
// streaming kernels (one thread per 5-D site, 4 spins; same grid as the Dslash
// so that partial-sum buffers line up)
// ---------------------------------------------------------------------------
namespace {

__device__ inline double fin_sum(const double *partial, int n) { return partial_sum(partial, n); }

template <int P> using TT = typename Store<P>::T;
template <int P> using CC = typename Store<P>::C;

template <int P> __device__ inline cx<CC<P>> L1(const TT<P> *p, long i) { return ldc(p, i); }

// r += a*s ; partial |r|^2
template <int P>
__global__ __launch_bounds__(BLK) void k_axpy_norm(long v5, TT<P> *r, const TT<P> *s,
                                                   const double *a, const int *stop,
                                                   double *partial) {
  if (stop && *stop) return;
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  const CC<P> av = (CC<P>)(*a);
  double red = 0.0;
  if (i < v5) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      cx<CC<P>> rv = L1<P>(r, k * v5 + i) + av * L1<P>(s, k * v5 + i);
      st(r, k * v5 + i, rv);
      red += (double)norm2(rv);
    }
  }
  const double t = block_sum(red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// p = r + b*p
template <int P>
__global__ __launch_bounds__(BLK) void k_xpay(long n, const TT<P> *r, TT<P> *p, const double *b,
                                              const int *stop) {
  if (stop && *stop) return;
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= n) return;
  const CC<P> bv = (CC<P>)(*b);
  st(p, i, L1<P>(r, i) + bv * L1<P>(p, i));
}

// partial |x|^2 (per-element products in the storage precision, summed in FP64)
template <int P>
__global__ __launch_bounds__(BLK) void k_norm(long v5, const TT<P> *x, double *partial) {
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  double red = 0.0;
  if (i < v5) {
#pragma unroll
    for (int k = 0; k < 4; k++) red += (double)norm2(L1<P>(x, k * v5 + i));
  }
  const double t = block_sum(red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// epilogues for operators that cannot fuse them (Wilson kernel, Ls > 64)
__global__ __launch_bounds__(BLK) void k_epi(long v5, int mode, const double2 *o, const double2 *w,
                                             const double2 *r, double2 *ro, double2 *x,
                                             const double2 *p, const double *a, const double *b,
                                             const int *stop, double *partial) {
  if (stop && *stop) return;
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  double red = 0.0;
  if (i < v5) {
    for (int k = 0; k < 4; k++) {
      const long e = k * v5 + i;
      const cx<double> ov = ldc(o, e);
      if (mode == EPI_NORM) {
        red += norm2(ov);
      } else if (mode == EPI_DOTW) {
        const cx<double> wv = ldc(w, e);
        red += wv.r * ov.r + wv.i * ov.i;
      } else if (mode == EPI_HREC || mode == EPI_HPREC) {
        // r: h, in place; EPI_HPREC also x = p + b x (p the operator's input)
        const double bv = b ? *b : 0.0;
        const cx<double> hv = ov + bv * ldc(r, e);
        st(ro, e, hv);
        red += norm2(hv);
        if (mode == EPI_HPREC) st(x, e, b ? ldc(p, e) + bv * ldc(x, e) : ldc(p, e));
      } else if (mode == EPI_CG) {
        const cx<double> rv = ldc(r, e) - (*a) * ov;
        st(ro, e, rv);
        red += norm2(rv);
        if (b) st(x, e, ldc(x, e) + (*b) * ldc(p, e));
      }
    }
  }
  const double t = block_sum(red);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// the scalar steps as kernels of their own (one block), where no operator
// launch carries them (DslashLaunch::scal)
__global__ void k_cg_init(CgState *st, float resid, int niterc) {
  st->alpha = 1.0;
  st->alphan = 0.0;
  st->betacg = 0.0;
  st->lam[0] = st->lam[1] = 1.0;
  st->resid = resid;
  st->niterc = niterc;
  // iteration 1 (r = phi - M^+M x, no scalar of its own) always runs
  st->nx = niterc < 1 ? 0 : 1;
  st->itercg = st->nx;
  st->stop = niterc < 1 ? 1 : 0;
  st->iterations = niterc < 1 ? 1 : 0;
}

__global__ __launch_bounds__(BLK) void k_scalar(int kind, void *st, double *slot,
                                                const double *partial, int nb) {
  if (*scalar_stop(kind, st)) return;
  scalar_step(kind, st, slot, [&] { return partial_sum(partial, nb); });
}

__global__ __launch_bounds__(BLK) void k_ms_init(MsState *st, const double *partial, int nb) {
  const double d = fin_sum(partial, nb);
  if (threadIdx.x == 0) {
    st->delta = d;
    st->dl[0] = d;
    st->omega = 1.0;
    st->alpha = 0.0;
    st->gammag = 0.0;
    for (int i = 0; i < st->n; i++) {
      st->flags[i] = 1;
      st->zeta_i[i] = 1.0;
      st->zeta_ii[i] = 1.0;
      st->gammas[i] = 0.0;
      st->cg_returns[i] = 0;
    }
    st->cg_return = 0;
    st->maxi = st->n;
    st->mini = 1;
    st->umin = 1;
    st->umax = 0;
    for (int i = 0; i < MAXSHIFT; i++) st->cnt[i] = 0;
    st->jcount = 0;
    st->nonfinite = isfinite(d) ? 0 : 1;
    st->stop = (st->maxcg <= 0 || st->n <= 0 || st->nonfinite) ? 1 : 0;
    st->done = st->stop;
    // reference rule: sqrt(delta zeta^2) corr_i < res; plain rule (corr_i = 1):
    // shifted residual below res |b|
    st->resd = st->plain ? (double)st->res * sqrt(d) : (double)st->res;
  }
}

// the per-iteration updates' scalars: done also ends k_ms_update
__global__ __launch_bounds__(BLK) void k_ms_alpha(MsState *st, const double *partial, int nb) {
  if (st->stop) {
    if (threadIdx.x == 0) st->done = 1;
    return;
  }
  ms_alpha_step(st, [&] { return partial_sum(partial, nb); });
}
__global__ __launch_bounds__(BLK) void k_ms_lambda(MsState *st, const double *partial, int nb) {
  if (st->stop) return;
  ms_lambda_step<false>(st, nullptr, [&] { return partial_sum(partial, nb); });
}

// The block's coefficients from its recorded scalars, one thread per shift.
// With p_{j+1} = g_j p_j + z_j R_j and x_{j+1} = x_j - o_j p_j (shift i, j =
// 0 .. c-1), backwards over j: the weight of R_j in the last p is z_j times
// the product of the later g, and in x it is -z_j G_j with
// G_{j-1} = o_j + g_j G_j.  O(c) per shift and block, instead of updating c
// coefficients in every iteration.
// The block's last lambda (its iteration's partial sums) is taken here too.
__global__ __launch_bounds__(BLK) void k_ms_coef(MsState *st, const double *partial, int nb) {
  if (!st->stop) {  // uniform: nothing writes it before every thread has read it
    ms_lambda_step<true>(st, st->dl, [&] { return partial_sum(partial, nb); });
    __syncthreads();
  }
  const int i = threadIdx.x, n = st->n;
  if (i < n) {
    const int c = st->cnt[i];
    double g = 0.0, prod = 1.0;
    // the records of NQ iterations at a time: one wait for 3 NQ loads instead
    // of one per iteration (18 -> 7.2 us at c = 32)
    constexpr int NQ = 8;
    for (int q0 = MSR - NQ; q0 >= 0; q0 -= NQ) {
      double ze[NQ], ga[NQ], om[NQ];
#pragma unroll
      for (int k = 0; k < NQ; k++) {
        ze[k] = st->rec_ze[q0 + k][i];
        ga[k] = st->rec_ga[q0 + k][i];
        om[k] = st->rec_om[q0 + k][i];
      }
#pragma unroll
      for (int k = NQ - 1; k >= 0; k--) {
        const int q = q0 + k;
        double b = 0.0, d = 0.0;
        if (q < c) {
          b = ze[k] * prod;
          d = -(ze[k] * g);
          prod *= ga[k];
          g = om[k] + ga[k] * g;
        }
        st->cb[i][q] = b;
        st->cd[i][q] = d;
      }
    }
    st->ca[i] = prod;
    st->cc[i] = -g;
    st->fcnt[i] = c;
    st->fact[i] = !st->stop && i >= st->mini - 1 && i < st->maxi;
    st->cnt[i] = 0;
  }
  if (i == 0) {
    st->fjc = st->jcount;
    st->jcount = 0;
  }
}

// x_i, p_i of every shift that the block updated, from its residuals R_0 ..
// R_{c-1}: ring slot q of residual j = t0 + q.  Bound by memory: one read of
// each residual and, per shift, p and x read and written (c + 4 k field
// streams per block of c iterations, against 4 k + 3 per iteration when every
// iteration updates its shifts).  The residuals of an element stay in
// registers for all shifts.  Nothing here is read again before 32 iterations
// have passed through the caches, so all of it is non-temporal: 1.0 GB at 16^3
// x 48 with 12 shifts in the window in 190 us (5.2 TB/s).  Median launch of a
// solve of 25 shifts there 208 us; 244 through the caches, 256 also without the
// load of the next shift ahead of this one's work (four shifts ahead: 304).  The
// first block starts from p_i = b, x_i = 0 and writes every shift (x_i = 0
// where nothing was updated).
__global__ __launch_bounds__(BLK) void k_ms_flush(long ns, const MsState *S, const double2 *b,
                                                  const double2 *ring, double2 *X, double2 *P,
                                                  int first) {
  const int jc = S->fjc, n = S->n;
  if (jc == 0 && !first) return;
  __shared__ double sa[MAXSHIFT], sc[MAXSHIFT], sb[MAXSHIFT][MSR], sd[MAXSHIFT][MSR];
  __shared__ int scnt[MAXSHIFT], sact[MAXSHIFT];
  for (int k = threadIdx.x; k < n * MSR; k += BLK) {
    (&sb[0][0])[k] = (&S->cb[0][0])[k];
    (&sd[0][0])[k] = (&S->cd[0][0])[k];
  }
  for (int k = threadIdx.x; k < n; k += BLK) {
    sa[k] = S->ca[k];
    sc[k] = S->cc[k];
    scnt[k] = S->fcnt[k];
    sact[k] = S->fact[k];
  }
  __syncthreads();
  const long e = (long)blockIdx.x * BLK + threadIdx.x;
  if (e >= ns) return;
  cx<double> R[MSR];
#pragma unroll
  for (int q = 0; q < MSR; q++) R[q] = q < jc ? ldc_nt(ring, q * ns + e) : cx<double>{0.0, 0.0};
  const cx<double> bv = first ? ldc(b, e) : cx<double>{0.0, 0.0};
  // the next shift's p and x are loaded before this one's are worked on
  cx<double> pn = bv, xn{0.0, 0.0};
  const auto fetch = [&](int i) {
    if (!first && i < n && scnt[i]) {
      pn = ldc_nt(P, i * ns + e);
      xn = ldc_nt(X, i * ns + e);
    }
  };
  fetch(0);
  for (int i = 0; i < n; i++) {
    const cx<double> base = pn;
    const cx<double> x = xn;
    fetch(i + 1);
    if (!scnt[i]) {
      if (first) st(X, i * ns + e, cx<double>{0.0, 0.0});
      if (first && sact[i]) st(P, i * ns + e, bv);
      continue;
    }
    // the block's own sum first: its roundings are of its size, not of x_i's
    cx<double> dx = sc[i] * base;
    if (sact[i]) {
      cx<double> p = sa[i] * base;
#pragma unroll
      for (int q = 0; q < MSR; q++) {
        if (q < jc) {
          dx = dx + sd[i][q] * R[q];
          p = p + sb[i][q] * R[q];
        }
      }
      st_nt(P, i * ns + e, p);
    } else {
#pragma unroll
      for (int q = 0; q < MSR; q++)
        if (q < jc) dx = dx + sd[i][q] * R[q];
    }
    st_nt(X, i * ns + e, x + dx);
  }
}

// p = r + gammag p ; x_k -= omegas_k p_k ; p_k = gammas_k p_k + zeta_iii_k r
// (multishift_module.F90:145, 155-176), all active shifts in one pass over r
template <int P>
__global__ __launch_bounds__(BLK) void k_ms_update(long n, const TT<P> *r, TT<P> *p, TT<P> *xs,
                                                   TT<P> *ps, const MsState *S) {
  if (S->done) return;
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= n) return;
  using C = CC<P>;
  const cx<C> rv = L1<P>(r, i);
  st(p, i, rv + (C)S->gammag * L1<P>(p, i));
  for (int k = S->umin - 1; k < S->umax; k++) {
    TT<P> *x = xs + (long)k * n;
    TT<P> *q = ps + (long)k * n;
    const cx<C> pk = L1<P>(q, i);
    st(x, i, L1<P>(x, i) - (C)S->omegas[k] * pk);
    st(q, i, (C)S->gammas[k] * pk + (C)S->zeta_iii[k] * rv);
  }
}

template <int P>
__global__ __launch_bounds__(BLK) void k_bcast_copy(long n, int nshift, const TT<P> *src, TT<P> *dst) {
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i >= n) return;
  const auto v = src[i];
  for (int k = 0; k < nshift; k++) dst[(long)k * n + i] = v;
}

// element-wise FP64 -> FP32 complex conversion (link fields)
__global__ __launch_bounds__(BLK) void k_d2f(long n, const double2 *a, float2 *b) {
  const long i = (long)blockIdx.x * BLK + threadIdx.x;
  if (i < n) b[i] = make_float2((float)a[i].x, (float)a[i].y);
}

inline unsigned nblk(long n) { return (unsigned)((n + BLK - 1) / BLK); }

// streaming copy, 16 bytes per lane, non-temporal loads and stores, a
// grid-stride loop over a few blocks per CU: the fastest plain read+write
// stream measured on gfx950 (the HBM ceiling the Dslash is compared with)
typedef __attribute__((ext_vector_type(4))) unsigned U4;
__global__ __launch_bounds__(BLK) void k_stream_copy(const U4 *__restrict__ a, U4 *__restrict__ b,
                                                     long n) {
  const long stride = (long)gridDim.x * BLK;
  for (long i = (long)blockIdx.x * BLK + threadIdx.x; i < n; i += stride)
    __builtin_nontemporal_store(__builtin_nontemporal_load(a + i), b + i);
}

}  // namespace

int stream_copy(const void *src, void *dst, size_t bytes, hipStream_t s) {
  THR_CHECK(bytes % 16 == 0, THR_ERR_ARG, "byte count must be a multiple of 16");
  THR_CHECK(((uintptr_t)src | (uintptr_t)dst) % 16 == 0, THR_ERR_ARG, "pointers must be 16-byte aligned");
  if (bytes == 0) return THR_OK;
  int dev = 0, cus = 256;
  THR_HIP(hipGetDevice(&dev));
  THR_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const long n = (long)(bytes / 16);
  const long want = (long)cus * 4;
  const unsigned grid = (unsigned)std::max(1L, std::min(want, (long)nblk(n)));
  hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(BLK), 0, s, (const U4 *)src, (U4 *)dst, n);
  THR_HIP(hipGetLastError());
  return THR_OK;
}

int convert_d2f(long n, const double2 *a, float2 *b, hipStream_t s) {
  hipLaunchKernelGGL(k_d2f, dim3(nblk(n)), dim3(BLK), 0, s, n, a, b);
  THR_HIP(hipGetLastError());
  return THR_OK;
}

int apply_op(const OpDesc &op, int dagger, const double2 *in, double2 *out, hipStream_t s) {
  if (op.kernel == 1) {
    double2 *tmp = nullptr;
    if (op.d.ls > 64) {
      tmp = (double2 *)workspace(1, sizeof(double2) * op.d.nspinor());
      THR_CHECK(tmp, THR_ERR_HIP, "workspace allocation failed");
    }
    return launch_dslash_wilson(op.d, 1, dagger, op.imass, op.am, op.am3, in, out, op.u64, tmp, s);
  }
  DslashLaunch L{};
  L.d = op.d;
  L.nrhs = 1;
  L.prec = P64;
  L.dagger = dagger;
  L.imass = op.imass;
  L.am3 = op.am3;
  L.am[0] = op.am;
  L.in = in;
  L.out = out;
  L.links = op.u64;
  L.mode = EPI_STORE;
  L.sc_stride = 1;
  L.done_stride = 1;
  return launch_dslash(L, s);
}

// M or M^+ with a fused or (Wilson kernel, Ls > 64) separate epilogue, FP64.  L
// holds the epilogue's fields (mode, in, out, w, r, r_out, x, p, a_ptr,
// b_ptr, partial, done) and dagger; cfg is the solve's launch shape
static int apply_op_epi(const OpDesc &op, DslashLaunch L, const DslashConfig &cfg, hipStream_t s) {
  L.d = op.d;
  L.nrhs = 1;
  L.prec = P64;
  L.imass = op.imass;
  L.am3 = op.am3;
  L.am[0] = op.am;
  L.links = op.u64;
  L.sc_stride = 1;
  L.done_stride = 1;
  if (op.kernel == 1 && op.d.ls <= 64) return launch_wilson_epi(L, s);
  if (op.kernel == 1) {
    // the operator's passes are not gated by the stop flag, the epilogue is
    const bool hrec = L.mode == EPI_HREC || L.mode == EPI_HPREC;  // these read the old out
    const bool direct = L.out && !hrec;
    double2 *o = direct ? (double2 *)L.out : (double2 *)workspace(2, sizeof(double2) * op.d.nspinor());
    double2 *tmp = (double2 *)workspace(1, sizeof(double2) * op.d.nspinor());
    THR_CHECK(o && tmp, THR_ERR_HIP, "workspace allocation failed");
    TRY_RC(launch_dslash_wilson(op.d, 1, L.dagger, op.imass, op.am, op.am3, (const double2 *)L.in, o,
                                op.u64, tmp, s));
    if (L.mode != EPI_STORE) {
      hipLaunchKernelGGL(k_epi, dim3(nblk(op.d.v5())), dim3(BLK), 0, s, op.d.v5(), L.mode, o,
                         (const double2 *)L.w, (const double2 *)(hrec ? L.out : L.r),
                         (double2 *)(hrec ? L.out : L.r_out ? L.r_out : L.r), (double2 *)L.x,
                         (const double2 *)(hrec ? L.in : L.p), L.a_ptr, L.b_ptr, L.done, L.partial);
      THR_HIP(hipGetLastError());
    }
    return THR_OK;
  }
  return launch_dslash_cfg(L, cfg, s);
}

// whether the operator's launches may carry the solver's scalar steps
static bool op_fuses_scalars(const OpDesc &op, const DslashConfig &cfg) {
  return op.kernel == 1 ? op.d.ls <= 64 : dslash_fuses_scalars(cfg);
}

// the partial sums that an operator's epilogue writes, all of them
static int op_partials(const OpDesc &op, const DslashConfig &cfg) {
  return (int)(op.kernel == 1 ? wilson_blocks(op.d) : dslash_grid_blocks(op.d, cfg));
}

// poll a device int every `batch` iterations; batches grow to bound host syncs
template <typename F>
static int run_batched(F &&one_iteration, const int *dev_flag, hipStream_t s, long max_iters) {
  int *h = (int *)host_workspace(21, sizeof(int));
  THR_CHECK(h, THR_ERR_HIP, "host workspace allocation failed");
  *h = 0;
  int batch = 4;
  long done_iters = 0;
  for (;;) {
    for (int k = 0; k < batch; k++) TRY_RC(one_iteration());
    done_iters += batch;
    THR_HIP(hipMemcpyAsync(h, dev_flag, sizeof(int), hipMemcpyDeviceToHost, s));
    THR_HIP(hipStreamSynchronize(s));
    if (*h) return THR_OK;
    THR_CHECK(done_iters <= max_iters + 8, THR_ERR_STATE, "solver did not raise its stop flag");
    if (batch < 64) batch *= 2;
  }
}

size_t cg_state_bytes() { return sizeof(CgState); }

int cg_reference(const OpDesc &op, const double2 *phi, double2 *x, float res, int niterc,
                 int *itercg, int *iterations, hipStream_t s) {
  const Dims &d = op.d;
  const long n = d.nspinor();
  const int np = (int)std::max(dslash_blocks(d), wilson_blocks(d));
  CgBuffers B{};
  B.h = (double2 *)workspace(10, sizeof(double2) * n);
  B.r = (double2 *)workspace(11, sizeof(double2) * n);
  B.p = (double2 *)workspace(12, sizeof(double2) * n);
  B.state = workspace(13, sizeof(CgState));
  B.partial = partial_buffer(2 * np);
  THR_CHECK(B.h && B.r && B.p && B.state && B.partial, THR_ERR_HIP, "workspace allocation failed");
  B.partial2 = B.partial + np;
  return cg_reference_bufs(op, phi, x, res, niterc, itercg, iterations, s, B, false);
}

// The reference's CG with h = M p by recurrence (h_new = M r + beta h; M is
// linear), so the p update rides on the M pass and an iteration is two
// operator passes and two scalar steps.  Where the passes may carry the
// scalar steps (small launches) they do, and those cost no launches; the last
// step of a batch runs by itself, so the poll sees its verdict.  12^3 x 24: 27
// us per iteration with five launches, 15 with two.
int cg_reference_bufs(const OpDesc &op, const double2 *phi, double2 *x, float res, int niterc,
                      int *itercg, int *iterations, hipStream_t s, const CgBuffers &B,
                      bool no_alloc) {
  const Dims &d = op.d;
  const DslashConfig cfg = dslash_config(d, P64);
  const int nb = op_partials(op, cfg);
  double2 *h = B.h, *r = B.r, *p = B.p;
  CgState *st = (CgState *)B.state;
  THR_CHECK(h && r && p && st && B.partial, THR_ERR_ARG, "congrad: missing buffers");
  THR_CHECK(op.kernel == 0 || !no_alloc, THR_ERR_ARG,
            "congrad on caller buffers runs the Shamir kernel only");
  const bool fused = B.partial2 && op_fuses_scalars(op, cfg);
  double *apart = B.partial, *lpart = fused ? B.partial2 : B.partial;  // |h|^2 and |r|^2 sums
  // resid = 4*ksize*ksize*ksizet*kthird*res*res in default real (measure_module.F90:41)
  const long nsite4 = 4L * d.lx * d.ly * d.lt * d.ls;
  const float resid = ((float)nsite4 * res) * res;
  hipLaunchKernelGGL(k_cg_init, dim3(1), dim3(1), 0, s, st, resid, niterc);
  auto scalar = [&](int kind, long k, const double *partial) {
    hipLaunchKernelGGL(k_scalar, dim3(1), dim3(BLK), 0, s, kind, (void *)st, &st->lam[k & 1], partial,
                       nb);
  };
  // iteration k of the Fortran loop; first, last: of a batch
  auto iter = [&](long k, bool first, bool last) -> int {
    DslashLaunch a{};
    a.in = k == 1 ? x : r;
    a.out = h;
    a.partial = apart;
    a.done = &st->stop;
    if (k == 1) {
      a.mode = EPI_STORE;  // alpha = 1, x stays (measure_module.F90:60-66)
    } else {
      a.mode = EPI_HPREC;
      a.x = p;
      a.b_ptr = k == 2 ? nullptr : &st->betacg;  // p = r after the first iteration
      if (fused && !first) {
        a.fsum = lpart;
        a.fsum_n = nb;
        a.fdelta = &st->lam[k & 1];  // |r|^2 of iteration k - 2
        a.scal = SCAL_CG_BETA;
        a.sst = st;
        a.sslot = &st->lam[(k - 1) & 1];
      }
    }
    TRY_RC(apply_op_epi(op, a, cfg, s));
    DslashLaunch c{};
    c.dagger = 1;
    c.in = h;
    c.mode = EPI_CG;
    c.r = k == 1 ? const_cast<double2 *>(phi) : r;
    c.r_out = r;
    c.a_ptr = &st->alpha;
    c.partial = lpart;
    c.done = &st->stop;
    if (k > 1) {
      c.x = x;
      c.p = p;
      c.b_ptr = &st->alpha;
      if (fused) {
        c.fsum = apart;
        c.fsum_n = nb;
        c.fdelta = &st->lam[(k - 1) & 1];
        c.scal = SCAL_CG_ALPHA;
        c.sst = st;
      } else {
        scalar(SCAL_CG_ALPHA, k, apart);
      }
    }
    TRY_RC(apply_op_epi(op, c, cfg, s));
    if (!fused || last) scalar(SCAL_CG_BETA, k, lpart);
    THR_HIP(hipGetLastError());
    return THR_OK;
  };
  // Batches between polls: each poll drains the stream (15 us), each iteration
  // enqueued past the end is two launches that find the stop flag (6 us).  From
  // the third poll on the next batch is most of what the mean rate of decay
  // since the last poll leaves to do.
  CgState local;  // pageable: the read-back of a solve that may not allocate
  CgState *pinned = no_alloc ? nullptr : (CgState *)host_workspace(22, sizeof(CgState));
  CgState &hs = pinned ? *pinned : local;
  int batch = 4;
  double was = 0.0;
  for (long k = 0;;) {
    for (int b = 0; b < batch; b++) TRY_RC(iter(k + b + 1, b == 0, b + 1 == batch));
    k += batch;
    THR_HIP(hipMemcpyAsync(&hs, st, sizeof(CgState), hipMemcpyDeviceToHost, s));
    THR_HIP(hipStreamSynchronize(s));
    if (hs.stop) break;
    THR_CHECK(k <= (long)niterc + 8, THR_ERR_STATE, "solver did not raise its stop flag");
    const double now = std::log(hs.lam[k & 1] / (double)resid);
    const double left = was > now ? now / (was - now) * batch : 128.0;
    batch = was == 0.0 ? 8 : (int)std::max(4.0, std::min(std::min(64.0, 2.0 * batch), 0.8 * left));
    was = now;
  }
  *itercg = hs.itercg;
  if (iterations) *iterations = hs.iterations;
  THR_CHECK(hs.stop != 3, THR_ERR_NONFINITE,
            "congrad: non-finite dot product (NaN or Inf in the source, guess or links)");
  return THR_OK;
}

static int ms_setup(MsState *st, int n, const double *aden, const double *anum, float res,
                    int maxcg, hipStream_t s, int plain = 0) {
  THR_CHECK(n >= 1 && n <= MAXSHIFT, THR_ERR_ARG, "number of shifts out of range");
  MsState *hp = (MsState *)host_workspace(20, sizeof(MsState));
  THR_CHECK(hp, THR_ERR_HIP, "host workspace allocation failed");
  MsState &h = *hp;
  const size_t head = offsetof(MsState, rec_om);  // the rest is written before it is read
  std::memset(&h, 0, head);
  h.n = n;
  h.res = res;
  h.maxcg = maxcg;
  // correction = |anum/aden| / geometric mean (multishift_module.F90:87-88)
  double lsum = 0.0;
  for (int i = 0; i < n; i++) {
    h.corr[i] = std::fabs(anum[i] / aden[i]);
    lsum += std::log(h.corr[i]);
  }
  const double gm = std::exp(lsum / n);
  for (int i = 0; i < n; i++) {
    h.corr[i] = plain ? 1.0 : h.corr[i] / gm;
    h.aden[i] = aden[i];
  }
  h.plain = plain;
  THR_HIP(hipMemcpyAsync(st, &h, head, hipMemcpyHostToDevice, s));
  THR_HIP(hipStreamSynchronize(s));  // the pinned copy is written again by the read-back
  return THR_OK;
}

// the solve's counts and its error, read back from the device state
static int ms_result(const MsState *st, int n, int *cg_return, int *cg_returns, hipStream_t s) {
  MsState *h = (MsState *)host_workspace(20, sizeof(MsState));
  THR_CHECK(h, THR_ERR_HIP, "host workspace allocation failed");
  const size_t head = offsetof(MsState, rec_om);  // the counts and flags lie before the records
  THR_HIP(hipMemcpyAsync(h, st, head, hipMemcpyDeviceToHost, s));
  THR_HIP(hipStreamSynchronize(s));
  *cg_return = h->cg_return;
  if (cg_returns)
    for (int i = 0; i < n; i++) cg_returns[i] = h->cg_returns[i];
  THR_CHECK(!h->nonfinite, THR_ERR_NONFINITE,
            "multishift: non-finite dot product (NaN or Inf in the source or links)");
  return THR_OK;
}

// The same solve with the shift vectors updated once per block of MSR
// iterations (k_ms_coef, k_ms_flush) and neither p nor M^+M p stored: alpha =
// |M p|^2 comes from the M pass, h = M p obeys h_new = M r_new + gamma h (M is
// linear), and the M^+ pass updates r in its epilogue, into the next slot of
// the residual ring.  16^3 x 48, 25 poles: 195 us per iteration with the shift
// updates in every iteration (four streams per active shift: 120 us), of which
// this leaves the two operator passes and (MSR + 4 k) / MSR streams.  On small
// launches and with the Wilson kernel the passes also carry the scalar steps.
static int multishift_blocked(const OpDesc &op, int n, const double2 *input, double2 *out,
                              MsState *st, double2 *h, double2 *ring, double2 *P, double *apart,
                              double *lpart, int maxcg, const DslashConfig &cfg, hipStream_t s) {
  const Dims &d = op.d;
  const long ns = d.nspinor();
  const int nbl = op_partials(op, cfg);
  // the passes carry the scalar steps: each takes the sum that the other left
  const bool fused = op_fuses_scalars(op, cfg);
  int *stop = (int *)host_workspace(21, sizeof(int));
  THR_CHECK(stop, THR_ERR_HIP, "host workspace allocation failed");
  for (long t0 = 0;; t0 += MSR) {
    for (long t = t0; t < t0 + MSR; t++) {
      const double2 *rin = t == 0 ? input : ring + ((t - 1) % MSR) * ns;
      DslashLaunch a{};
      a.in = rin;
      a.out = h;
      a.mode = t == 0 ? EPI_NORM : EPI_HREC;
      a.b_ptr = t == 0 ? nullptr : &st->gammag;
      a.partial = apart;
      a.done = &st->stop;
      if (fused && t > t0) {
        a.fsum = lpart;
        a.fsum_n = nbl;
        a.fdelta = &st->dl[(t - 1) & 1];
        a.scal = SCAL_MS_LAMBDA;
        a.sst = st;
        a.sslot = &st->dl[t & 1];
      }
      TRY_RC(apply_op_epi(op, a, cfg, s));
      DslashLaunch b{};
      b.dagger = 1;
      b.in = h;
      b.mode = EPI_CG;
      b.r = const_cast<double2 *>(rin);
      b.r_out = ring + (t % MSR) * ns;
      b.a_ptr = &st->minus_omega;
      b.partial = lpart;
      b.done = &st->stop;
      if (fused) {
        b.fsum = apart;
        b.fsum_n = nbl;
        b.fdelta = &st->dl[t & 1];
        b.scal = SCAL_MS_ALPHA;
        b.sst = st;
      } else {
        hipLaunchKernelGGL(k_scalar, dim3(1), dim3(BLK), 0, s, (int)SCAL_MS_ALPHA, (void *)st,
                           (double *)nullptr, apart, nbl);
      }
      TRY_RC(apply_op_epi(op, b, cfg, s));
      if (!fused && t + 1 < t0 + MSR)
        hipLaunchKernelGGL(k_scalar, dim3(1), dim3(BLK), 0, s, (int)SCAL_MS_LAMBDA, (void *)st, st->dl,
                           lpart, nbl);
    }
    hipLaunchKernelGGL(k_ms_coef, dim3(1), dim3(BLK), 0, s, st, lpart, nbl);
    hipLaunchKernelGGL(k_ms_flush, dim3(nblk(ns)), dim3(BLK), 0, s, ns, st, input, ring, out, P,
                       t0 == 0 ? 1 : 0);
    THR_HIP(hipGetLastError());
    THR_HIP(hipMemcpyAsync(stop, &st->stop, sizeof(int), hipMemcpyDeviceToHost, s));
    THR_HIP(hipStreamSynchronize(s));
    if (*stop) return THR_OK;
    THR_CHECK(t0 <= (long)maxcg + 2 * MSR, THR_ERR_STATE, "solver did not raise its stop flag");
  }
}

int multishift_reference(const OpDesc &op, int n, const double *aden, const double *anum,
                         const double2 *input, double2 *out, float res, int maxcg,
                         int *cg_return, int *cg_returns, hipStream_t s, int plain) {
  const Dims &d = op.d;
  const long ns = d.nspinor();
  const int nb = (int)dslash_blocks(d);
  double2 *h = (double2 *)workspace(21, sizeof(double2) * ns);
  double2 *ps = (double2 *)workspace(24, sizeof(double2) * ns * n);
  MsState *st = (MsState *)workspace(25, sizeof(MsState));
  const int np = (int)std::max<long>(nb, wilson_blocks(d));
  double *partial = partial_buffer(2 * np);
  THR_CHECK(h && ps && st && partial, THR_ERR_HIP, "workspace allocation failed");
  // Blocked updates keep MSR residuals (16 GiB at most here: 512 MiB fields;
  // 32^3 x 64 takes 4.3).  Larger fields, and a card on which the ring is more
  // than a quarter of the free memory, update every shift in every iteration:
  // 16^3 x 48, 25 shifts 8.0 ms with the ring, 49.4 ms without.
  // THR_MULTISHIFT_RING=0: never.  The context keeps the ring, and gives it
  // back when one of its own allocations would fail.
  const char *ring_env = std::getenv("THR_MULTISHIFT_RING");
  const size_t ring_bytes = sizeof(double2) * ns * MSR;
  struct Ring {
    double2 *p = nullptr;
    ~Ring() {
      if (p) release_spare(26);
    }
  } held;
  if (!(ring_env && std::atoi(ring_env) == 0) && ring_bytes <= (size_t(16) << 30))
    held.p = (double2 *)spare_workspace(26, ring_bytes);
  double2 *ring = held.p;
  int rc = ms_setup(st, n, aden, anum, res, maxcg, s, plain);
  if (rc) return rc;
  const DslashConfig cfg = dslash_config(d, P64);
  hipLaunchKernelGGL(k_norm<P64>, dim3(nb), dim3(BLK), 0, s, d.v5(), input, partial);
  hipLaunchKernelGGL(k_ms_init, dim3(1), dim3(BLK), 0, s, st, partial, nb);
  THR_HIP(hipGetLastError());
  if (ring) {
    TRY_RC(multishift_blocked(op, n, input, out, st, h, ring, ps, partial, partial + np, maxcg, cfg, s));
    return ms_result(st, n, cg_return, cg_returns, s);
  }
  double2 *r = (double2 *)workspace(20, sizeof(double2) * ns);
  double2 *sv = (double2 *)workspace(22, sizeof(double2) * ns);
  double2 *p = (double2 *)workspace(23, sizeof(double2) * ns);
  THR_CHECK(r && sv && p, THR_ERR_HIP, "workspace allocation failed");
  THR_HIP(hipMemcpyAsync(r, input, sizeof(double2) * ns, hipMemcpyDeviceToDevice, s));
  THR_HIP(hipMemcpyAsync(p, input, sizeof(double2) * ns, hipMemcpyDeviceToDevice, s));
  THR_HIP(hipMemsetAsync(out, 0, sizeof(double2) * ns * n, s));
  hipLaunchKernelGGL(k_bcast_copy<P64>, dim3(nblk(ns)), dim3(BLK), 0, s, ns, n, input, ps);
  THR_HIP(hipGetLastError());
  const int *stop = &st->stop;
  const int nbl = op_partials(op, cfg);
  auto iter = [&]() -> int {
    DslashLaunch a{};
    a.in = p;
    a.out = h;
    a.mode = EPI_STORE;
    a.done = stop;
    TRY_RC(apply_op_epi(op, a, cfg, s));
    DslashLaunch b{};
    b.dagger = 1;
    b.in = h;
    b.out = sv;
    b.mode = EPI_DOTW;
    b.w = p;
    b.partial = partial;
    b.done = stop;
    TRY_RC(apply_op_epi(op, b, cfg, s));
    hipLaunchKernelGGL(k_ms_alpha, dim3(1), dim3(BLK), 0, s, st, partial, nbl);
    hipLaunchKernelGGL(k_axpy_norm<P64>, dim3(nb), dim3(BLK), 0, s, d.v5(), r, sv, &st->omega,
                       stop, partial);
    hipLaunchKernelGGL(k_ms_lambda, dim3(1), dim3(BLK), 0, s, st, partial, nb);
    hipLaunchKernelGGL(k_ms_update<P64>, dim3(nblk(ns)), dim3(BLK), 0, s, ns, r, p, out, ps, st);
    THR_HIP(hipGetLastError());
    return THR_OK;
  };
  rc = run_batched(iter, stop, s, maxcg);
  if (rc) return rc;
  return ms_result(st, n, cg_return, cg_returns, s);
}

int multishift_reference_sp(const OpDesc &op, int n, const double *aden, const double *anum,
                            const double2 *input, double2 *out, float res, int maxcg,
                            int *cg_return, int *cg_returns, hipStream_t s) {
  THR_CHECK(op.kernel == 0, THR_ERR_ARG, "the FP32 multishift is Shamir-only (qmrherm_module.F90:54-63)");
  const Dims &d = op.d;
  const long ns = d.nspinor();
  const int nb = (int)dslash_blocks(d);
  float2 *r = (float2 *)workspace(30, sizeof(float2) * ns);
  float2 *h = (float2 *)workspace(31, sizeof(float2) * ns);
  float2 *sv = (float2 *)workspace(32, sizeof(float2) * ns);
  float2 *p = (float2 *)workspace(33, sizeof(float2) * ns);
  float2 *ps = (float2 *)workspace(34, sizeof(float2) * ns * n);
  float2 *xs = (float2 *)workspace(35, sizeof(float2) * ns * n);
  float2 *u32 = (float2 *)workspace(36, sizeof(float2) * d.v4() * 3);
  MsState *st = (MsState *)workspace(37, sizeof(MsState));
  double *partial = partial_buffer(nb);
  THR_CHECK(r && h && sv && p && ps && xs && u32 && st && partial, THR_ERR_HIP,
            "workspace allocation failed");
  int rc = ms_setup(st, n, aden, anum, res, maxcg, s);
  if (rc) return rc;
  // u = cmplx(udp), input = cmplx(inputdp) (multishift_module.F90:351-352)
  hipLaunchKernelGGL(k_d2f, dim3(nblk(d.v4() * 3)), dim3(BLK), 0, s, d.v4() * 3, op.u64, u32);
  // FP32 spinors keep a site's spins together: the conversion reorders too
  TRY_RC(convert_spinors(d, 1, input, nullptr, P64, r, nullptr, P32, s));
  THR_HIP(hipMemcpyAsync(p, r, sizeof(float2) * ns, hipMemcpyDeviceToDevice, s));
  THR_HIP(hipMemsetAsync(xs, 0, sizeof(float2) * ns * n, s));
  hipLaunchKernelGGL(k_bcast_copy<P32>, dim3(nblk(ns)), dim3(BLK), 0, s, ns, n, r, ps);
  hipLaunchKernelGGL(k_norm<P32>, dim3(nb), dim3(BLK), 0, s, d.v5(), r, partial);
  hipLaunchKernelGGL(k_ms_init, dim3(1), dim3(BLK), 0, s, st, partial, nb);
  THR_HIP(hipGetLastError());
  const int *stop = &st->stop;
  DslashLaunch L{};
  L.d = d;
  L.nrhs = 1;
  L.prec = P32;
  L.imass = op.imass;
  L.am3 = op.am3;
  L.am[0] = op.am;
  L.links = u32;
  L.sc_stride = 1;
  L.done = stop;
  L.done_stride = 1;
  L.partial = partial;
  auto iter = [&]() -> int {
    DslashLaunch a = L;
    a.dagger = 0;
    a.in = p;
    a.out = h;
    a.mode = EPI_STORE;
    int rc2 = launch_dslash(a, s);
    if (rc2) return rc2;
    DslashLaunch b = L;
    b.dagger = 1;
    b.in = h;
    b.out = sv;
    b.mode = EPI_DOTW;
    b.w = p;
    rc2 = launch_dslash(b, s);
    if (rc2) return rc2;
    hipLaunchKernelGGL(k_ms_alpha, dim3(1), dim3(BLK), 0, s, st, partial, nb);
    hipLaunchKernelGGL(k_axpy_norm<P32>, dim3(nb), dim3(BLK), 0, s, d.v5(), r, sv, &st->omega,
                       stop, partial);
    hipLaunchKernelGGL(k_ms_lambda, dim3(1), dim3(BLK), 0, s, st, partial, nb);
    hipLaunchKernelGGL(k_ms_update<P32>, dim3(nblk(ns)), dim3(BLK), 0, s, ns, r, p, xs, ps, st);
    THR_HIP(hipGetLastError());
    return THR_OK;
  };
  rc = run_batched(iter, stop, s, maxcg);
  if (rc) return rc;
  TRY_RC(convert_spinors(d, n, xs, nullptr, P32, out, nullptr, P64, s));
  return ms_result(st, n, cg_return, cg_returns, s);
}

}  // namespace thr
