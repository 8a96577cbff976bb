// small.hip -- a whole 2-qubit gate of small bonds in one workgroup.
//
// theta' = G (Ai Aj), its SVD, the truncation and the two new sites (ExaTnMpsVisitor.cpp:1387-1730,
// :2366-2536) for theta' of at most 64 rows or columns whose other side fits the LDS beside it.  The
// general path takes about 15 launches and, per Jacobi sweep, two copies, a memset, a launch per round
// and a synchronisation; at these sizes each launch works for a few us on a few kilobytes, and a wave
// took 0.3 to 0.9 ms.  Here theta', its rows and every intermediate stay in LDS, convergence is tested
// on the device, and a wave is one launch.
//
// The SVD is the one-sided Jacobi of the general path on single rows: the rows of X = theta' (or
// theta'^H) in circle order, r / 2 disjoint pairs a step.  A pair belongs to 16 lanes (one DPP row): they
// form both squared norms and the inner product from the rows, rotate and write them back, so every angle
// comes from the rows themselves and no Gram matrix is carried.  A step is bound by its chain (LDS read,
// products, four DPP sums, the rotation, LDS write, barrier), and at 64 rows by FP64 issue of the one CU.
// Measured, a wave: 13 us at bonds up to 4, 60 to 80 us up to 16, 320 to 465 us up to 32.
#include <cfloat>
#include <cstddef>

#include "kernels.h"
#include "device_util.h"

namespace hipmps {

// Sum over the 16 lanes of a DPP row, bit for bit the same in each of them: every step adds two lanes'
// values in both (rotations by 4 and 8 would add the four quads in two different orders, and lanes that
// disagree on an angle of nearly equal rows rotate their columns differently).
__device__ __forceinline__ double row16_sum(double v) {
  v = dpp_add<0xb1>(v);          // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4e>(v);          // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);         // row_half_mirror
  return dpp_add<0x140>(v);      // row_mirror
}

// One-sided Jacobi on the rows of Y (nr even, stride elements apart, 16 NJ columns): sweeps until no pair's
// relative inner product exceeds tol.  Returns the sweeps used; *flag (LDS) is 0 when converged.
template <int NT, int NJ>
__device__ __forceinline__ int jacobi_rows(double2* Y, int stride, int nr, double tol, double floor2, int max_sweeps,
                                           int* flag) {
  const int tid = threadIdx.x, group = tid >> 4, l16 = tid & 15;
  const double itol = 0.25 * tol, tol2 = tol * tol;
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    if (tid == 0) *flag = 0;
    __syncthreads();
    for (int step = 0; step < nr - 1; ++step) {
      for (int p = group; p < nr / 2; p += NT / 16) {
        double2* yp = Y + circle_slot(p, step, nr) * stride + l16;
        double2* yq = Y + circle_slot(nr - 1 - p, step, nr) * stride + l16;
        double2 a[NJ], b[NJ];
        double alpha = 0.0, beta = 0.0;
        double2 g = make_double2(0, 0);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          a[j] = yp[16 * j];
          b[j] = yq[16 * j];
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          alpha = fma(a[j].x, a[j].x, fma(a[j].y, a[j].y, alpha));
          beta = fma(b[j].x, b[j].x, fma(b[j].y, b[j].y, beta));
          g = cfmac(a[j], b[j], g);
        }
        alpha = row16_sum(alpha);
        beta = row16_sum(beta);
        g = make_double2(row16_sum(g.x), row16_sum(g.y));
        if (alpha > floor2 && beta > floor2 && cabs2(g) > tol2 * (alpha * beta) && l16 == 0) *flag = 1;
        double c;
        double2 tau;
        jacobi_rotation(alpha, beta, g, itol, floor2, c, tau);
        if (tau.x != 0.0 || tau.y != 0.0) {  // rows' = W^T rows, W = c [[1, tau], [-conj(tau), 1]]
          const double2 nt = make_double2(-tau.x, tau.y);
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            yp[16 * j] = cscale(cfma(nt, b[j], a[j]), c);
            yq[16 * j] = cscale(cfma(tau, a[j], b[j]), c);
          }
        }
      }
      __syncthreads();
    }
    const int again = *flag;
    __syncthreads();
    if (!again) return sweep + 1;
  }
  return sweep;
}

template <int NT>
__device__ __forceinline__ int jacobi_rows_n(double2* Y, int stride, int nr, double tol, double floor2, int max_sweeps,
                                             int* flag) {
  switch (stride >> 4) {
    case 1: return jacobi_rows<NT, 1>(Y, stride, nr, tol, floor2, max_sweeps, flag);
    case 2: return jacobi_rows<NT, 2>(Y, stride, nr, tol, floor2, max_sweeps, flag);
    case 4: return jacobi_rows<NT, 4>(Y, stride, nr, tol, floor2, max_sweeps, flag);
    default: return jacobi_rows<NT, 8>(Y, stride, nr, tol, floor2, max_sweeps, flag);
  }
}

// Norms of the rows of Y, sorted descending, ties by row: sig[rank], perm[rank].  NaN / Inf sorted as 0 and
// flagged.  tmp, sig, perm: LDS, SMALL_MAX_ROWS entries.
template <int NT>
__device__ __forceinline__ void sort_rows(const double2* Y, int stride, int r, int c, double* tmp, double* sig,
                                          int* perm, int* bad) {
  const int tid = threadIdx.x, group = tid >> 4, l16 = tid & 15;
  for (int i = group; i < r; i += NT / 16) {
    double a = 0.0;
    for (int j = l16; j < c; j += 16) a += cabs2(Y[i * stride + j]);
    a = sqrt(row16_sum(a));
    if (l16 == 0) {
      if (!(a >= 0.0 && a <= DBL_MAX)) {
        a = 0.0;
        *bad = 1;
      }
      tmp[i] = a;
    }
  }
  __syncthreads();
  if (tid < r) {
    const double a = tmp[tid];
    int rank = 0;
    for (int j = 0; j < r; ++j) {
      const double b = tmp[j];
      rank += b > a || (b == a && j < tid);
    }
    sig[rank] = a;
    perm[rank] = tid;
  }
  __syncthreads();
}

// One vector of X's other side per 16 lanes: u[i] = <y, X row i> * scale for the rows i = l16 + 16 q < r;
// returns the sum of |u|^2 over all rows.  The lanes start at different columns: rows are a multiple of 256
// bytes apart, the same column of 16 rows is one LDS bank (measured 27 of 320 us at 64 rows).
__device__ __forceinline__ double other_side(const double2* X, const double2* y, int stride, int r, int c,
                                             double scale, double2 (&u)[SMALL_MAX_ROWS / 16]) {
  const int l16 = threadIdx.x & 15;
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < SMALL_MAX_ROWS / 16; ++q) {
    u[q] = make_double2(0, 0);
    const int i = l16 + 16 * q;
    if (i < r) {
      const double2* x = X + i * stride;
      double2 d = make_double2(0, 0);
      int j = l16 % c;
      for (int e = 0; e < c; ++e) {
        d = cfmac(y[j], x[j], d);
        j = j + 1 == c ? 0 : j + 1;
      }
      u[q] = cscale(d, scale);
      t += cabs2(u[q]);
    }
  }
  return row16_sum(t);
}

template <typename S, int NT, int CAP>
__global__ __launch_bounds__(NT) void k_gate_small(const GateTask* tasks) {
  __shared__ GateTask T;
  __shared__ double2 sX[CAP], sY[CAP];
  __shared__ double s_sig[SMALL_MAX_ROWS], s_scy[SMALL_MAX_ROWS], s_scw[SMALL_MAX_ROWS], s_inv[SMALL_MAX_ROWS];
  __shared__ int s_perm[SMALL_MAX_ROWS];
  __shared__ double s_red[NT / 64];
  __shared__ int s_flag, s_K, s_bad;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, group = tid >> 4, l16 = tid & 15;
  for (int e = tid; e < (int)(sizeof(GateTask) / 4); e += NT) ((int*)&T)[e] = ((const int*)(tasks + blockIdx.x))[e];
  if (tid == 0) {
    s_flag = 0;
    s_bad = 0;
  }
  __syncthreads();
  const int m = T.m, n = T.n, r = T.r, cr = T.cr, cm = T.cm, ki = T.ki, tr = T.transposed;
  const int nr = small_rows(r);
  const int stride = small_stride(T.c);
  for (int e = tid; e < nr * stride; e += NT) sX[e] = sY[e] = make_double2(0, 0);
  __syncthreads();
  // ---- theta' (rows (l, kap, a), columns (b, r)), one thread per (l, kap, r) ----
  double f2 = 0.0;
  {
    const S* Ai = (const S*)T.Ai;
    const S* Aj = (const S*)T.Aj;
    const int cl = T.chi_l * ki;
    for (int e = tid; e < cl * cr; e += NT) {
      const int lk = e / cr, rr = e - lk * cr, l = lk / ki, k = lk - l * ki;
      const size_t a0 = ((size_t)(2 * l) * ki + k) * cm, a1 = ((size_t)(2 * l + 1) * ki + k) * cm;
      double2 x[4] = {make_double2(0, 0), make_double2(0, 0), make_double2(0, 0), make_double2(0, 0)};
#pragma unroll 4
      for (int q = 0; q < cm; ++q) {
        const double2 u0 = ld(Ai, a0 + q), u1 = ld(Ai, a1 + q);
        const double2 v0 = ld(Aj, (size_t)(2 * q) * cr + rr), v1 = ld(Aj, (size_t)(2 * q + 1) * cr + rr);
        x[0] = cfma(u0, v0, x[0]);
        x[1] = cfma(u0, v1, x[1]);
        x[2] = cfma(u1, v0, x[2]);
        x[3] = cfma(u1, v1, x[3]);
      }
#pragma unroll
      for (int ab = 0; ab < 4; ++ab) {
        double2 o = make_double2(0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) o = cfma(T.G[ab * 4 + q], x[q], o);
        // stabilizeTensorBody: |x| < 1e-100 -> 0 (ExaTnMpsVisitor.cpp:141-161)
        if (cabs2(o) < 1e-200) o = make_double2(0, 0);
        f2 += cabs2(o);
        const int i = 2 * lk + (ab >> 1), j = (ab & 1) * cr + rr;
        const int at = tr ? j * stride + i : i * stride + j;
        if (tr) o = cconj(o);
        sX[at] = o;
        sY[at] = o;
      }
    }
  }
  f2 = wave_sum(f2);
  if (lane == 0) s_red[wave] = f2;
  __syncthreads();
  f2 = 0.0;
  for (int w = 0; w < NT / 64; ++w) f2 += s_red[w];
  __syncthreads();
  const int sweeps = jacobi_rows_n<NT>(sY, stride, nr, T.tol, JAC_FLOOR2 * f2, T.max_sweeps, &s_flag);
  __syncthreads();
  sort_rows<NT>(sY, stride, r, T.c, s_inv, s_sig, s_perm, &s_bad);
  // ---- truncation rule and factor scales, as k_select ----
  if (wave == 0) {
    const double sg = lane < r ? s_sig[lane] : 0.0;
    const double pn = T.pn_l2 ? sqrt(sg) : sg;
    const unsigned long long below = __ballot(lane < r && pn < T.cutoff);
    int K = below ? (int)__ffsll(below) : r;  // first sub-threshold index i: keep i + 1
    K = max(1, min(K, T.max_bond));
    const double kept = wave_sum(lane < K ? sg * sg : 0.0), disc = wave_sum(lane >= K ? sg * sg : 0.0);
    const double ssum = wave_sum(sg);
    const double f = T.renorm && kept > 0.0 ? sqrt((kept + disc) / kept) : 1.0;
    if (lane < r) {
      double gy = 0.0, gw = 0.0, is = 0.0;
      if (lane < K && sg > 1e-150) {
        // exponents of f sigma: left aL, right 1 - aL; Y's side is the right one unless transposed
        const double sf = sg * f, h = sqrt(sf);
        const double left = T.absorb == 0 ? h : 1.0, right = T.absorb == 0 ? h : sf;
        gy = (tr ? left : right) / sg;
        gw = tr ? right : left;
        is = 1.0 / sg;
      }
      s_scy[lane] = gy;
      s_scw[lane] = gw;
      s_inv[lane] = is;
    }
    if (lane == 0) {
      s_K = K;
      GateResult R;
      R.K = K;
      R.sweeps = sweeps;
      R.converged = s_flag == 0;
      R.pad = 0;
      R.w[0] = disc;
      R.w[1] = kept;
      R.w[2] = kept + disc;
      R.w[3] = f;
      R.w[4] = ssum;
      R.w[5] = s_bad ? 1.0 : 0.0;
      *T.res = R;
    }
  }
  __syncthreads();
  const int K = s_K;
  S* Oi = (S*)T.Oi;
  S* Oj = (S*)T.Oj;
  // left site element of theta' row i = (l, kap, a) and bond index k
  auto left = [&](int i, int k) {
    const int lk = i >> 1, l = lk / ki;
    return ((size_t)(2 * l + (i & 1)) * ki + (lk - l * ki)) * K + k;
  };
  // ---- factor on Y's side ----
  for (int e = tid; e < K * T.c; e += NT) {
    if (!tr) {
      const int k = e / n, j = e - k * n;
      st(Oj, (size_t)e, cscale(sY[s_perm[k] * stride + j], s_scy[k]));
    } else {
      const int i = e / K, k = e - i * K;
      st(Oi, left(i, k), cscale(cconj(sY[s_perm[k] * stride + i]), s_scy[k]));
    }
  }
  // ---- the other factor: X's rows on the kept rows of Y, each vector scaled to its length ----
  for (int k = group; k < K; k += NT / 16) {
    double2 u[SMALL_MAX_ROWS / 16];
    const double t = other_side(sX, sY + s_perm[k] * stride, stride, r, T.c, s_inv[k], u);
    const double f = t > 0.0 ? s_scw[k] / sqrt(t) : 0.0;
#pragma unroll
    for (int q = 0; q < SMALL_MAX_ROWS / 16; ++q) {
      const int i = l16 + 16 * q;
      if (i >= r) continue;
      if (!tr) st(Oi, left(i, k), cscale(u[q], f));
      else st(Oj, (size_t)k * n + i, cscale(cconj(u[q]), f));
    }
  }
}

hipError_t launch_gate_small(const GateTask* d_tasks, int ntasks, int fp32, bool lo, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  if (fp32) {
    if (lo) hipLaunchKernelGGL((k_gate_small<float2, 256, SMALL_CAP_LO>), dim3(ntasks), dim3(256), 0, s, d_tasks);
    else hipLaunchKernelGGL((k_gate_small<float2, 512, SMALL_CAP>), dim3(ntasks), dim3(512), 0, s, d_tasks);
  } else {
    if (lo) hipLaunchKernelGGL((k_gate_small<double2, 256, SMALL_CAP_LO>), dim3(ntasks), dim3(256), 0, s, d_tasks);
    else hipLaunchKernelGGL((k_gate_small<double2, 512, SMALL_CAP>), dim3(ntasks), dim3(512), 0, s, d_tasks);
  }
  return hipGetLastError();
}

// ------------------------------------------------------------------ noise channels of small sites
// A whole channel in one workgroup: the rows of X (one per old Kraus index and operator, columns (l, p, r))
// or of X^H when X has more rows than columns, their Jacobi sweeps, the kept rows, and the new site in its
// final layout, K of its Kraus index known here, in T.out.  The general path (kraus.hip) takes a copy, an
// expansion, a launch per Jacobi round, a synchronisation per sweep and a gather per channel; at these sizes
// each of them is a launch for a few us of work.  From X^H: W X^H = Y with orthogonal rows of length sigma_j
// makes Sigma W a square root of X^H X like X itself, and its row j is (Y_j X) / sigma_j, scaled to length
// sigma_j; no identity is carried through the rotations.
template <typename S, int NT, int CAP>
__global__ __launch_bounds__(NT) void k_kraus_small(const KrausTask* tasks) {
  __shared__ KrausTask T;
  __shared__ double2 sX[CAP], sY[CAP];
  __shared__ double s_sig[SMALL_MAX_ROWS], s_tmp[SMALL_MAX_ROWS];
  __shared__ int s_perm[SMALL_MAX_ROWS];
  __shared__ int s_flag, s_K, s_bad;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, group = tid >> 4, l16 = tid & 15;
  {
    const KrausTask* t = tasks + blockIdx.x;
    const int words = (int)(offsetof(KrausTask, K) / 4) + 16 * t->n_ops;
    for (int e = tid; e < words; e += NT) ((int*)&T)[e] = ((const int*)t)[e];
  }
  if (tid == 0) {
    s_flag = 0;
    s_bad = 0;
  }
  __syncthreads();
  const int cr = T.cr, kap = T.kap, n_ops = T.n_ops, adj = T.adj, r = T.r, c = T.c;
  const int nr = small_rows(r), stride = small_stride(c);
  for (int e = tid; e < nr * stride; e += NT) sX[e] = sY[e] = make_double2(0, 0);
  __syncthreads();
  {  // one thread per (l, k, r): its 2 n_ops elements of X
    const S* A = (const S*)T.site;
    for (int e = tid; e < T.cl * kap * cr; e += NT) {
      const int rr = e % cr, lk = e / cr, l = lk / kap, k = lk - l * kap;
      const double2 a0 = ld(A, ((size_t)(2 * l) * kap + k) * cr + rr);
      const double2 a1 = ld(A, ((size_t)(2 * l + 1) * kap + k) * cr + rr);
      for (int op = 0; op < 2 * n_ops; ++op) {  // (operator, new physical index)
        const int row = k * n_ops + (op >> 1), col = (2 * l + (op & 1)) * cr + rr;
        const double2 v = cadd(cmul(T.K[2 * op], a0), cmul(T.K[2 * op + 1], a1));
        const int at = adj ? col * stride + row : row * stride + col;
        sX[at] = sY[at] = adj ? cconj(v) : v;
      }
    }
  }
  __syncthreads();
  const int sweeps = jacobi_rows_n<NT>(sY, stride, nr, T.tol, 0.0, T.max_sweeps, &s_flag);
  __syncthreads();
  sort_rows<NT>(sY, stride, r, c, s_tmp, s_sig, s_perm, &s_bad);
  if (wave == 0) {  // kept rows, as k_select's keep_rule
    const double sg = lane < r ? s_sig[lane] : 0.0;
    const double pn = T.pn_l2 ? sg : sg * sg;
    const unsigned long long below = __ballot(lane < r && pn < T.cutoff);
    const int K = max(1, min(below ? (int)__ffsll(below) - 1 : r, T.max_bond));
    const double kept = wave_sum(lane < K ? sg * sg : 0.0), disc = wave_sum(lane >= K ? sg * sg : 0.0);
    if (lane == 0) {
      s_K = K;
      GateResult R;
      R.K = K;
      R.sweeps = sweeps;
      R.converged = s_flag == 0;
      R.pad = 0;
      R.w[0] = disc;
      R.w[1] = kept;
      R.w[2] = kept + disc;
      R.w[3] = 1.0;
      R.w[4] = 0.0;
      R.w[5] = s_bad ? 1.0 : 0.0;
      *T.res = R;
    }
  }
  __syncthreads();
  const int K = s_K;
  S* out = (S*)T.out;
  if (!adj) {
    for (int e = tid; e < K * c; e += NT) {  // e = (lp, j, r)
      const int rr = e % cr, lpj = e / cr, lp = lpj / K, j = lpj - lp * K;
      st(out, (size_t)e, sY[s_perm[j] * stride + lp * cr + rr]);
    }
    return;
  }
  for (int j = group; j < K; j += NT / 16) {
    const double sg = s_sig[j];
    double2 u[SMALL_MAX_ROWS / 16];
    const double t = other_side(sX, sY + s_perm[j] * stride, stride, r, c, sg > 1e-150 ? 1.0 / sg : 0.0, u);
    const double f = t > 0.0 ? sg / sqrt(t) : 0.0;
#pragma unroll
    for (int q = 0; q < SMALL_MAX_ROWS / 16; ++q) {
      const int i = l16 + 16 * q;
      if (i < r) st(out, ((size_t)(i / cr) * K + j) * cr + i % cr, cscale(cconj(u[q]), f));
    }
  }
}

hipError_t launch_kraus_small(const KrausTask* d_tasks, int ntasks, int fp32, bool lo, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  if (fp32) {
    if (lo) hipLaunchKernelGGL((k_kraus_small<float2, 256, SMALL_CAP_LO>), dim3(ntasks), dim3(256), 0, s, d_tasks);
    else hipLaunchKernelGGL((k_kraus_small<float2, 512, SMALL_CAP>), dim3(ntasks), dim3(512), 0, s, d_tasks);
  } else {
    if (lo) hipLaunchKernelGGL((k_kraus_small<double2, 256, SMALL_CAP_LO>), dim3(ntasks), dim3(256), 0, s, d_tasks);
    else hipLaunchKernelGGL((k_kraus_small<double2, 512, SMALL_CAP>), dim3(ntasks), dim3(512), 0, s, d_tasks);
  }
  return hipGetLastError();
}

// The new sites of a wave of channels from scratch to their buffers, one workgroup each (units of 8 bytes).
__global__ __launch_bounds__(256) void k_copy_sites(const CopyTask* tasks) {
  const CopyTask T = tasks[blockIdx.x];
  const HIPMPS_GLOBAL double* src = (const HIPMPS_GLOBAL double*)T.src;
  HIPMPS_GLOBAL double* dst = (HIPMPS_GLOBAL double*)T.dst;
#pragma unroll 8
  for (size_t e = threadIdx.x; e < T.units; e += 256) dst[e] = src[e];
}

hipError_t launch_copy_sites(const CopyTask* d_tasks, int ntasks, hipStream_t s) {
  if (ntasks > 0) hipLaunchKernelGGL(k_copy_sites, dim3(ntasks), dim3(256), 0, s, d_tasks);
  return hipGetLastError();
}

// |0..0>: one launch for all sites instead of an upload and a synchronisation each.
template <typename S>
__global__ __launch_bounds__(256) void k_zero_state(void* const* sites, int n) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  S* A = (S*)sites[k];
  st(A, 0, make_double2(1, 0));
  st(A, 1, make_double2(0, 0));
}

hipError_t launch_zero_state(void* const* sites, int n, int fp32, hipStream_t s) {
  const dim3 grid((n + 255) / 256);
  if (fp32) hipLaunchKernelGGL(k_zero_state<float2>, grid, dim3(256), 0, s, sites, n);
  else hipLaunchKernelGGL(k_zero_state<double2>, grid, dim3(256), 0, s, sites, n);
  return hipGetLastError();
}

// ------------------------------------------------------------------ environment chain of small bonds
// E <- sum_s d_s A_s^H (E A_s) over the sites, s = (p, kap), E and A_s in LDS.  A chain of products launched
// one by one costs two launches a site, 8 to 20 us, for a few us of work on few workgroups; here a site is
// a few steps of three barriers, and every diagonal of a measurement -- one per <Z_i>, per pair, per outcome
// string -- is a workgroup of the same launch.  A step takes as many s side by side as fit the workgroup's
// threads (chain_slots); the next A_s are read while these are used.
template <typename S>
__global__ __launch_bounds__(256) void k_env_chain(const ChainSite* sites, int n, const double* diags, double* out) {
  constexpr int B = CHAIN_MAX_BOND, Q = B * B / 256;
  __shared__ double2 sE[B * (B + 1)], sA[B * (B + 1)], sX[B * (B + 1)];
  const int tid = threadIdx.x;
  const double* diag = diags + (size_t)blockIdx.x * 2 * n;
  if (tid == 0) sE[0] = make_double2(1.0, 0.0);
  for (int k = 0; k < n; ++k) {
    const ChainSite site = sites[k];
    const int cl = site.cl, cr = site.cr, kap = site.kap, na = cl * cr, ne = cr * cr;
    const S* A = (const S*)site.A;
    const double dg[2] = {diag[2 * k], diag[2 * k + 1]};
    const int slots = chain_slots(cl, cr), w = max(na, ne);
    const int slot = slots > 1 ? tid / w : 0;
    const int i0 = tid - slot * w;  // first element of this thread
    const bool on = slot < slots;
    const double2* eA = sA + slot * na;
    double2* eX = sX + slot * na;
    int al[Q], ar[Q];  // this thread's elements (l, r) of A_s and X, and (i, j) of the result
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      al[q] = (i0 + 256 * q) / cr;
      ar[q] = (i0 + 256 * q) - al[q] * cr;
    }
    auto has = [&](int q, int count) { return on && (q == 0 || slots == 1) && i0 + 256 * q < count; };
    double2 acc[Q], next[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = make_double2(0, 0);
    // the s with a nonzero diagonal: [s0, s1)
    const int s0 = dg[0] != 0.0 ? 0 : kap, s1 = dg[1] != 0.0 ? 2 * kap : kap;
    auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        next[q] = make_double2(0, 0);
        if (has(q, na) && s < s1) next[q] = ld(A, ((size_t)al[q] * 2 * kap + s) * cr + ar[q]);
      }
    };
    if (s0 < s1) fetch(s0 + slot);
    for (int sb = s0; sb < s1; sb += slots) {
      const int s = sb + slot;
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (has(q, na)) sA[slot * na + i0 + 256 * q] = next[q];
      __syncthreads();
      if (sb + slots < s1) fetch(s + slots);
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (has(q, na)) {
          double2 x = make_double2(0, 0);
          for (int l = 0; l < cl; ++l) x = cfma(sE[al[q] * cl + l], eA[l * cr + ar[q]], x);
          eX[i0 + 256 * q] = x;
        }
      __syncthreads();
      const double d = s < kap ? dg[0] : dg[1];
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (has(q, ne)) {
          double2 x = make_double2(0, 0);
          for (int l = 0; l < cl; ++l) x = cfmac(eA[l * cr + al[q]], eX[l * cr + ar[q]], x);
          acc[q] = make_double2(fma(d, x.x, acc[q].x), fma(d, x.y, acc[q].y));
        }
      __syncthreads();
    }
    __syncthreads();
    if (slots > 1) {  // the slots' sums, in order
      if (has(0, ne)) sX[slot * ne + i0] = acc[0];
      __syncthreads();
      if (tid < ne) {
        double2 t = make_double2(0, 0);
        for (int q = 0; q < slots; ++q) t = cadd(t, sX[q * ne + tid]);
        sE[tid] = t;
      }
    } else {
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (has(q, ne)) sE[i0 + 256 * q] = acc[q];
    }
    __syncthreads();
  }
  if (tid == 0) out[blockIdx.x] = sE[0].x;
}

hipError_t launch_env_chain(const ChainSite* d_sites, int n, const double* d_diags, double* d_out, int nchains,
                            int fp32, hipStream_t s) {
  if (nchains <= 0) return hipSuccess;
  if (fp32) hipLaunchKernelGGL(k_env_chain<float2>, dim3(nchains), dim3(256), 0, s, d_sites, n, d_diags, d_out);
  else hipLaunchKernelGGL(k_env_chain<double2>, dim3(nchains), dim3(256), 0, s, d_sites, n, d_diags, d_out);
  return hipGetLastError();
}

}  // namespace hipmps
