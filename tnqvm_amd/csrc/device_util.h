// device_util.h -- device helpers shared by the libhipmps kernel files (internal).
#pragma once
#include <hip/hip_runtime.h>

namespace hipmps {

// ------------------------------------------------------------------ complex helpers
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
// c + a*b
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
  c.x = fma(a.x, b.x, c.x);
  c.x = fma(-a.y, b.y, c.x);
  c.y = fma(a.x, b.y, c.y);
  c.y = fma(a.y, b.x, c.y);
  return c;
}
// c + conj(a)*b
__device__ __forceinline__ double2 cfmac(double2 a, double2 b, double2 c) {
  c.x = fma(a.x, b.x, c.x);
  c.x = fma(a.y, b.y, c.x);
  c.y = fma(a.x, b.y, c.y);
  c.y = fma(-a.y, b.x, c.y);
  return c;
}
__device__ __forceinline__ double cabs2(double2 a) { return a.x * a.x + a.y * a.y; }

// Loads and stores through a pointer that came out of a task descriptor.  The compiler cannot tell
// which memory such a pointer names and emits flat accesses, which count as LDS accesses too and
// complete in no known order, so that every wait on an LDS read also waits for every load in flight.
// These go through the global address space.
typedef double gvec_d2 __attribute__((ext_vector_type(2)));
typedef float gvec_f2 __attribute__((ext_vector_type(2)));
#define HIPMPS_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ double2 gld(const double2* p) {
  const gvec_d2 v = *(const HIPMPS_GLOBAL gvec_d2*)p;
  return make_double2(v.x, v.y);
}
__device__ __forceinline__ float2 gld(const float2* p) {
  const gvec_f2 v = *(const HIPMPS_GLOBAL gvec_f2*)p;
  return make_float2(v.x, v.y);
}
__device__ __forceinline__ void gst(double2* p, double2 v) {
  gvec_d2 x;
  x.x = v.x;
  x.y = v.y;
  *(HIPMPS_GLOBAL gvec_d2*)p = x;
}
__device__ __forceinline__ void gst(float2* p, float2 v) {
  gvec_f2 x;
  x.x = v.x;
  x.y = v.y;
  *(HIPMPS_GLOBAL gvec_f2*)p = x;
}

// base uniform over the wave, idx < 2^28 (the byte offset wraps at 2^32): one scalar base and a 32-bit offset
// instead of a 64-bit address per load
__device__ __forceinline__ double2 gld_at(const double2* base, unsigned idx) {
  const gvec_d2 v = *(const HIPMPS_GLOBAL gvec_d2*)((const HIPMPS_GLOBAL char*)base + (size_t)(idx * 16u));
  return make_double2(v.x, v.y);
}
__device__ __forceinline__ void gst_at(double2* base, unsigned idx, double2 v) {
  gvec_d2 x;
  x.x = v.x;
  x.y = v.y;
  *(HIPMPS_GLOBAL gvec_d2*)((HIPMPS_GLOBAL char*)base + (size_t)(idx * 16u)) = x;
}

template <typename T>
__device__ __forceinline__ double2 ld(const T* p, size_t i);
template <>
__device__ __forceinline__ double2 ld<double2>(const double2* p, size_t i) { return gld(p + i); }
template <>
__device__ __forceinline__ double2 ld<float2>(const float2* p, size_t i) {
  const float2 v = gld(p + i);
  return make_double2((double)v.x, (double)v.y);
}
template <typename T>
__device__ __forceinline__ void st(T* p, size_t i, double2 v);
template <>
__device__ __forceinline__ void st<double2>(double2* p, size_t i, double2 v) { gst(p + i, v); }
template <>
__device__ __forceinline__ void st<float2>(float2* p, size_t i, double2 v) {
  gst(p + i, make_float2((float)v.x, (float)v.y));
}

// Largest t with begin(t) <= b, for task arrays sorted by their first block.
template <typename Task, typename F>
__device__ __forceinline__ int find_task(const Task* tasks, int ntasks, int b, F begin) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (begin(tasks[mid]) <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}


// FP64 MFMA v_mfma_f64_16x16x4f64 operand layout on gfx950 (measured):
//   A[i][k] in lane i + 16k, B[k][j] in lane j + 16k, D[i][j] in lane j + 16*(i%4),
//   accumulator register i/4.
typedef double mfma_d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ mfma_d4 mfma64(double a, double b, mfma_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Sum over the wave, the same value in every lane: four DPP steps within the rows of 16 lanes, then
// the four row sums through scalar registers.  A shuffle-based tree goes through the LDS crossbar at
// every level (about 7 times the latency, and these sums are most of a reflector's serial chain).
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, 0xf, 0xf, true);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_value(double v, int lane) {  // lane: wave-uniform
  const long long x = __double_as_longlong(v);
  const unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)x, lane);
  const unsigned int hi = (unsigned int)__builtin_amdgcn_readlane((int)(x >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | lo);
}
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0xb1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4e>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x124>(v);  // row_ror:4
  v = dpp_add<0x128>(v);  // row_ror:8
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}
__device__ __forceinline__ double2 wave_sum2(double2 v) { return make_double2(wave_sum(v.x), wave_sum(v.y)); }

// Round-robin ("circle") ordering of nb slots: slot 0 holds 0, slot s > 0 holds 1 + (s - 1 + round) mod
// (nb - 1); slots i and nb - 1 - i meet.
__device__ __forceinline__ int circle_slot(int s, int round, int nb) {
  return s == 0 ? 0 : 1 + (s - 1 + round) % (nb - 1);
}

// 1/sqrt(a) and 1/d: the hardware approximations (5e-8) refined by one Newton step, which leaves up to 19 and 10
// eps (0.8 and 0.5 on average; 4 M arguments over all mantissas and 1000 binades).
__device__ __forceinline__ double nr_rsq(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double hy = 0.5 * a * y;
  return fma(y, fma(-hy, y, 0.5), y);
}
__device__ __forceinline__ double nr_rcp(double d) {
  const double x = __builtin_amdgcn_rcp(d);
  return fma(x, fma(-d, x, 1.0), x);
}
// The same to the last bit, 0.62 and 0.50 eps at worst (1 / sqrt(a) of the library: 0.75), by the third-order term
// and by a second step: for reflectors, whose vector has to have length 1 to working precision.
__device__ __forceinline__ double full_rsq(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double e = fma(-a * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double full_rcp(double d) {
  const double x = nr_rcp(d);
  return fma(x, fma(-d, x, 1.0), x);
}

// Rotation that annihilates gamma in the Hermitian 2x2 [[alpha, gamma], [conj(gamma), beta]]
// (Golub & Van Loan Alg. 8.4.1 with a phase): h = beta - alpha,
// tau = 2 sign(h) gamma / (|h| + sqrt(h^2 + 4|gamma|^2))  (|tau| = t, the smaller root),
// c = 1/sqrt(1 + |tau|^2);  J = c [[1, tau], [-conj(tau), 1]].
// The rotated diagonal is alpha - f |gamma|^2, beta + f |gamma|^2 with tau = f gamma; it replaces
// alpha and beta.  The identity when |gamma| <= tol sqrt(alpha beta) or a diagonal entry is 0.
__device__ __forceinline__ void jacobi_rotation(double& alpha, double& beta, double2 gamma, double tol, double floor2,
                                                double& c, double2& tau) {
  const double g2 = cabs2(gamma);
  if (!(alpha > floor2) || !(beta > floor2) || !(g2 > tol * tol * alpha * beta)) {
    c = 1.0;
    tau = make_double2(0.0, 0.0);
    return;
  }
  const double h = beta - alpha;
  const double a = fma(h, h, 4.0 * g2);
  const double d = fabs(h) + a * nr_rsq(a);
  const double f = (h >= 0.0 ? 2.0 : -2.0) * nr_rcp(d);
  tau = make_double2(f * gamma.x, f * gamma.y);
  c = nr_rsq(1.0 + cabs2(tau));
  alpha = fma(-f, g2, alpha);
  beta = fma(f, g2, beta);
}

}  // namespace hipmps
