// Shared device/host definitions for the gfx950 domain-wall library.
//
// Device layout (halo-free, everything resident in HBM):
//   spinor   [rhs][spin 0..3][t][y][x][s]   complex, s fastest
//   links    [mu 0..2][t][y][x]             complex
//   fp16 spinors store half2 per complex plus one float scale per 5-D site
//   [rhs][t][y][x][s] shared by the 4 spins.
// This is the reference's column-major Phi(1:Ls,1:Lx,1:Ly,1:Lt,1:4) with the
// halos stripped: periodic and antiperiodic boundaries are index arithmetic
// on the device (the antiperiodic t sign lives in the links, as in coef).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdio>
#include <string>

namespace thr {

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------
void set_error(const std::string &msg);
const char *last_error();

#define THR_HIP(call)                                                                   \
  do {                                                                                  \
    hipError_t _e = (call);                                                             \
    if (_e != hipSuccess) {                                                             \
      ::thr::set_error(std::string(#call) + ": " + hipGetErrorString(_e));             \
      return THR_ERR_HIP;                                                               \
    }                                                                                   \
  } while (0)

#define TRY_RC(x)            \
  do {                       \
    int _rc = (x);           \
    if (_rc) return _rc;     \
  } while (0)

#define THR_CHECK(cond, code, msg) \
  do {                             \
    if (!(cond)) {                 \
      ::thr::set_error(msg);       \
      return (code);               \
    }                              \
  } while (0)

// ---------------------------------------------------------------------------
// precision tags
// ---------------------------------------------------------------------------
enum Prec { P64 = 0, P32 = 1, P16 = 2 };

struct Dims {
  int lx, ly, lt, ls;
  __host__ __device__ long v4() const { return (long)lx * ly * lt; }
  __host__ __device__ long v5() const { return v4() * ls; }
  __host__ __device__ long nspinor() const { return v5() * 4; }  // complex elements per spinor
};

// ---------------------------------------------------------------------------
// complex helpers (compute type C = double or float)
// ---------------------------------------------------------------------------
template <typename C> struct cx { C r, i; };

template <typename C> __host__ __device__ inline cx<C> mk(C r, C i) { return cx<C>{r, i}; }
template <typename C> __device__ inline cx<C> operator+(cx<C> a, cx<C> b) { return {a.r + b.r, a.i + b.i}; }
template <typename C> __device__ inline cx<C> operator-(cx<C> a, cx<C> b) { return {a.r - b.r, a.i - b.i}; }
template <typename C> __device__ inline cx<C> operator*(C s, cx<C> a) { return {s * a.r, s * a.i}; }
template <typename C> __device__ inline cx<C> cmul(cx<C> a, cx<C> b) {
  return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r};
}
// conj(a) * b
template <typename C> __device__ inline cx<C> cjmul(cx<C> a, cx<C> b) {
  return {a.r * b.r + a.i * b.i, a.r * b.i - a.i * b.r};
}
template <typename C> __device__ inline cx<C> conj(cx<C> a) { return {a.r, -a.i}; }
// i * a
template <typename C> __device__ inline cx<C> muli(cx<C> a) { return {-a.i, a.r}; }
template <typename C> __device__ inline C norm2(cx<C> a) { return a.r * a.r + a.i * a.i; }

// ---------------------------------------------------------------------------
// storage access: load/store a complex of compute type C from storage of Prec
// ---------------------------------------------------------------------------
template <int PREC> struct Store;

template <> struct Store<P64> {
  using C = double;
  using T = double2;
  static constexpr int bytes = 16;
};
template <> struct Store<P32> {
  using C = float;
  using T = float2;
  static constexpr int bytes = 8;
};
template <> struct Store<P16> {
  using C = float;
  using T = __half2;
  static constexpr int bytes = 4;
};

__device__ inline cx<double> ldc(const double2 *p, long i) {  // cached (stencil) load
  double2 v = p[i];
  return {v.x, v.y};
}
__device__ inline cx<float> ldc(const float2 *p, long i) {
  float2 v = p[i];
  return {v.x, v.y};
}
__device__ inline void st(double2 *p, long i, cx<double> v) { p[i] = make_double2(v.r, v.i); }
__device__ inline void st(float2 *p, long i, cx<float> v) { p[i] = make_float2(v.r, v.i); }
// non-temporal: data that is not read again before the caches have turned over
typedef __attribute__((ext_vector_type(2))) double V2d;
typedef __attribute__((ext_vector_type(2))) float V2f;
__device__ inline cx<double> ldc_nt(const double2 *p, long i) {
  const V2d v = __builtin_nontemporal_load((const V2d *)p + i);
  return {v.x, v.y};
}
__device__ inline cx<float> ldc_nt(const float2 *p, long i) {
  const V2f v = __builtin_nontemporal_load((const V2f *)p + i);
  return {v.x, v.y};
}
__device__ inline void st_nt(double2 *p, long i, cx<double> c) {
  const V2d v = {c.r, c.i};
  __builtin_nontemporal_store(v, (V2d *)p + i);
}

__device__ inline cx<float> ldh(const __half2 *p, long i, float scale) {
  float2 f = __half22float2(p[i]);
  return {f.x * scale, f.y * scale};
}

constexpr int BLK = 256;  // threads per block for every streaming kernel

// v of another lane of its 16-lane row, by DPP control CTRL
template <int CTRL> __device__ inline double dpp_value(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// v of lane i plus v of lane i ^ 32 (HALF) or i ^ 16: a row swap of two copies
// leaves the one in the first and the other in the second
template <bool HALF> __device__ inline double swap_add(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)(b & 0xffffffffLL), hi = (unsigned)(b >> 32);
  const auto l = HALF ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                      : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = HALF ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                      : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  const unsigned l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1];
  return __longlong_as_double(((long long)h0 << 32) | l0) +
         __longlong_as_double(((long long)h1 << 32) | l1);
}
// sum over the wave, valid in every lane: the butterfly over lanes ^ 32, 16, 8,
// 4, 2, 1.  Register moves; wave shuffles go through LDS, and six of them one
// after another cost 0.3 us, as much as the loads of a small Dslash.
__device__ inline double wave_sum(double v) {
  v = swap_add<true>(v);
  v = swap_add<false>(v);
  v += dpp_value<0x128>(v);  // lane ^ 8: rotation of the row by 8
  v += dpp_value<0x124>(v);  // by 4: lane ^ 4 or ^ 12, equal by now
  v += dpp_value<0x4E>(v);   // lane ^ 2
  v += dpp_value<0xB1>(v);   // lane ^ 1
  return v;
}

// deterministic block reduction over NTH threads: wave sums, then a
// fixed-order LDS sum; the result is valid in every thread.  One barrier; the
// LDS buffer is TAG's, so sums of different tags may follow each other freely
// and sums of one tag need a barrier in between (block_sum_n has it).
template <int NTH, int TAG>
__device__ inline double block_sum_once(double v) {
  __shared__ double sm[NTH / 64];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < NTH / 64; k++) t += sm[k];
  return t;
}
template <int NTH>
__device__ inline double block_sum_n(double v) {
  const double t = block_sum_once<NTH, 0>(v);
  __syncthreads();
  return t;
}
__device__ inline double block_sum(double v) { return block_sum_n<BLK>(v); }

// thread k (< BLK) of a sum of n per-block partial sums: p[k] + p[k + BLK] +
// ... in that order.  The loads are issued 8 at a time before they are added,
// so a long row costs a few memory latencies instead of one per element.
__device__ inline double partial_thread(const double *p, int n) {
  constexpr int U = 8;
  double v = 0.0;
  for (int k0 = threadIdx.x; k0 < n; k0 += U * BLK) {
    double a[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + u * BLK;
      a[u] = k < n ? p[k] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + u * BLK < n) v += a[u];
  }
  return v;
}

// sum of n per-block partial sums by BLK threads (partial_thread, then
// block_sum): the result depends only on the values and n
__device__ inline double partial_sum(const double *p, int n) {
  return block_sum(partial_thread(p, n));
}

}  // namespace thr

// status codes shared with the C ABI
#define THR_OK 0
#define THR_ERR_ARG 1
#define THR_ERR_HIP 2
#define THR_ERR_NOCONV 3
#define THR_ERR_SIZE 4
#define THR_ERR_STATE 5
#define THR_ERR_NONFINITE 6
