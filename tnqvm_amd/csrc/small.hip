// small.hip -- a whole 2-qubit gate of small bonds in one workgroup.
//
// theta' = G (Ai Aj), its SVD, the truncation and the two new sites (ExaTnMpsVisitor.cpp:1387-1730,
// :2366-2536) for theta' of at most 64 rows or columns whose other side fits the LDS beside it.  The
// general path takes about 15 launches and, per Jacobi sweep, two copies, a memset, a launch per round
// and a synchronisation; at these sizes each launch works for a few us on a few kilobytes, and a wave
// took 0.3 to 0.9 ms.  Here theta', its rows and every intermediate stay in LDS, convergence is tested
// on the device, and a wave is one launch.
//
// The SVD is an LQ and the one-sided Jacobi of the general path on single rows: the rows of L^H in circle
// order, r / 2 disjoint pairs a step.  A pair belongs to 16 lanes (one DPP row): they form the inner product
// from the rows, rotate and write them back, so every angle comes from the rows themselves and no Gram matrix
// is carried.  A step is bound by its chain (LDS read, products, two DPP sums, the rotation, LDS write,
// barrier: 1050 clocks up to 16 rows, 1200 at 32), and at 64 rows by LDS bandwidth and FP64 issue of the one
// CU one after the other (2290).  Measured, random theta' (8 to 9 sweeps): 18 us at 4 x 4, 31 at 8 x 8, 68 at
// 16 x 16, 160 at 32 x 32, 620 at 64 x 64; a line of 12 qubits whose waves are at most 64 x 64 took 9.6 ms
// with the sweeps on the rows of theta' and norms formed at every step, 7.7 ms with these.
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

// X = L Q by Householder reflections from the right, X (r x c, r <= c, in Y) replaced by L^H: its first r
// columns upper triangular, columns r .. 16 NJ - 1 (of the sweeps that follow) zero.  At a step every 16 lanes
// form the reflector of row k from the row themselves and apply it to their rows below: one barrier a step,
// the diagonal kept aside in d (LDS, r entries) because the others still read row k.
template <int NT, int NC>
__device__ __forceinline__ void lq_rows(double2* Y, int stride, int r, int c, int zero_to, double2* d) {
  const int tid = threadIdx.x, group = tid >> 4, l16 = tid & 15;
  for (int k = 0; k < r; ++k) {
    const double2* yk = Y + k * stride;
    const double2 head = yk[k];
    double2 w[NC];
    double tail = 0.0;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      w[q] = yk[l16 + 16 * q];
      if (l16 + 16 * q <= k) w[q] = make_double2(0, 0);
      tail = fma(w[q].x, w[q].x, fma(w[q].y, w[q].y, tail));
    }
    tail = row16_sum(tail);
    if (tail > 1e-290) {  // below: nothing to reflect that a double would show
      // w = x + e norm e_k with e = head / |head|; x becomes -e norm, other rows y - (y w^H) w / (norm (norm + |head|))
      const double a2 = cabs2(head), n2 = a2 + tail, norm = n2 * full_rsq(n2);
      const double ra = a2 > 1e-290 ? full_rsq(a2) : 0.0, a = a2 * ra;
      const double2 e = ra > 0.0 ? cscale(head, ra) : make_double2(1, 0);
      const double scale = full_rcp(norm * (norm + a));
      const double2 wk = cscale(e, a + norm);
#pragma unroll
      for (int q = 0; q < NC; ++q)
        if (l16 + 16 * q == k) w[q] = wk;
      for (int i = k + 1 + group; i < r; i += NT / 16) {
        double2* y = Y + i * stride + l16;
        double2 v[NC], t = make_double2(0, 0);
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          v[q] = y[16 * q];
          t = cfmac(w[q], v[q], t);
        }
        t = cscale(make_double2(row16_sum(t.x), row16_sum(t.y)), -scale);
#pragma unroll
        for (int q = 0; q < NC; ++q) y[16 * q] = cfma(t, w[q], v[q]);
      }
      if (tid == 0) d[k] = cscale(e, -norm);
    } else if (tid == 0) {
      d[k] = head;
    }
    __syncthreads();
  }
  for (int e = tid; e < r * zero_to; e += NT) {
    const int i = e / zero_to, j = e - i * zero_to;
    double2* at = Y + i * stride + j;
    if (j < i) {
      Y[j * stride + i] = cconj(*at);
      *at = make_double2(0, 0);
    } else if (j == i) {
      *at = cconj(d[i]);
    } else if (j >= r) {
      *at = make_double2(0, 0);
    }
  }
  __syncthreads();
}

// One-sided Jacobi on the rows of Y (nr even, stride elements apart, 16 NJ columns): sweeps until no pair's
// relative inner product exceeds tol.  A pair a group: nr / 2 <= NT / 16.  The squared norms travel with the
// rotations in n2 (LDS) and are formed from the rows again at every sweep, so the sweep that finds nothing to
// rotate has tested the rows' own.  Blocks of two rows a group, four rotations a step with half the LDS
// traffic, are on four waves instead of eight and no faster (64 rows: 2310 clocks a rotation's step for 2290).
// Returns the sweeps used; *flag (LDS) is 0 when converged.
template <int NT, int NJ>
__device__ __forceinline__ int jacobi_rows(double2* Y, int stride, int nr, double tol, double floor2, int max_sweeps,
                                           int* flag, double* n2) {
  const int tid = threadIdx.x, group = tid >> 4, l16 = tid & 15;
  const double itol = 0.25 * tol, tol2 = tol * tol;
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
    if (tid == 0) *flag = 0;
    for (int i = group; i < nr; i += NT / 16) {
      double a = 0.0;
#pragma unroll
      for (int j = 0; j < NJ; ++j) a += cabs2(Y[i * stride + l16 + 16 * j]);
      a = row16_sum(a);
      if (l16 == 0) n2[i] = a;
    }
    __syncthreads();
    bool above = false;
    // the rows of this group's pair: slots group and nr - 1 - group of the circle ordering
    int ip = group, iq = nr - 1 - group;
    for (int step = 0; step < nr - 1; ++step) {
      if (group < nr / 2) {
        double2* yp = Y + ip * stride + l16;
        double2* yq = Y + iq * stride + l16;
        double alpha = n2[ip], beta = n2[iq];
        double2 a[NJ], b[NJ];
        double2 g = make_double2(0, 0), g1 = make_double2(0, 0);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          a[j] = yp[16 * j];
          b[j] = yq[16 * j];
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          if (j & 1) g1 = cfmac(a[j], b[j], g1);
          else g = cfmac(a[j], b[j], g);
        }
        if (NJ > 1) g = cadd(g, g1);
        g = make_double2(row16_sum(g.x), row16_sum(g.y));
        above |= (alpha > floor2) & (beta > floor2) & (cabs2(g) > tol2 * (alpha * beta));
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
          if (l16 == 0) {
            n2[ip] = alpha;
            n2[iq] = beta;
          }
        }
      }
      ip = ip == 0 ? 0 : (ip + 1 == nr ? 1 : ip + 1);
      iq = iq + 1 == nr ? 1 : iq + 1;
      __syncthreads();
    }
    if (above) *flag = 1;
    __syncthreads();
    const int again = *flag;
    __syncthreads();
    if (!again) return sweep + 1;
  }
  return sweep;
}

template <int NT>
__device__ __forceinline__ int jacobi_rows_n(double2* Y, int stride, int nr, int cols, double tol, double floor2,
                                             int max_sweeps, int* flag, double* n2) {
  switch (cols >> 4) {
    case 1: return jacobi_rows<NT, 1>(Y, stride, nr, tol, floor2, max_sweeps, flag, n2);
    case 2: return jacobi_rows<NT, 2>(Y, stride, nr, tol, floor2, max_sweeps, flag, n2);
    case 4: return jacobi_rows<NT, 4>(Y, stride, nr, tol, floor2, max_sweeps, flag, n2);
    default: return jacobi_rows<NT, 8>(Y, stride, nr, tol, floor2, max_sweeps, flag, n2);
  }
}

// L of X = L Q (r x c in Y) and Jacobi sweeps on the rows of L^H: rows sigma_j u_j^H, r columns, u_j the left
// singular vectors of X.  On theta' of decaying spectra the sweeps on the rows of X itself were 11 to 13 at 32
// and 64 rows (24 over ten decades), on L^H 8 to 9, on rows of r columns instead of c; the LQ costs the
// barriers of half a sweep.
template <int NT>
__device__ __forceinline__ int svd_rows(double2* Y, int stride, int r, int c, double tol, double floor2,
                                        int max_sweeps, int* flag, double* n2, double2* d) {
  const int zero_to = small_stride(r) - 1;
  switch (stride >> 4) {
    case 1: lq_rows<NT, 1>(Y, stride, r, c, zero_to, d); break;
    case 2: lq_rows<NT, 2>(Y, stride, r, c, zero_to, d); break;
    case 4: lq_rows<NT, 4>(Y, stride, r, c, zero_to, d); break;
    default: lq_rows<NT, 8>(Y, stride, r, c, zero_to, d); break;
  }
  return jacobi_rows_n<NT>(Y, stride, small_rows(r), zero_to, tol, floor2, max_sweeps, flag, n2);
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

// X's other side: u[j] = sum_i y_i X_ij for the columns j = l16 + 16 q < c, two vectors y per 16 lanes.
__device__ __forceinline__ void other_side(const double2* X, const double2* y0, const double2* y1, int stride, int r,
                                           int c, double2 (&u0)[SMALL_MAX_COLS / 16],
                                           double2 (&u1)[SMALL_MAX_COLS / 16]) {
  const int l16 = threadIdx.x & 15;
#pragma unroll
  for (int q = 0; q < SMALL_MAX_COLS / 16; ++q) u0[q] = u1[q] = make_double2(0, 0);
  for (int i = 0; i < r; ++i) {
    const double2 v0 = y0[i], v1 = y1[i];
#pragma unroll
    for (int q = 0; q < SMALL_MAX_COLS / 16; ++q)
      if (16 * q < c) {
        const double2 x = X[i * stride + l16 + 16 * q];  // X is zero from c to the stride
        u0[q] = cfma(v0, x, u0[q]);
        u1[q] = cfma(v1, x, u1[q]);
      }
  }
}
// u <- u times `scale`, then to the length `len`
__device__ __forceinline__ void to_length(double2 (&u)[SMALL_MAX_COLS / 16], double scale, double len) {
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < SMALL_MAX_COLS / 16; ++q) {
    u[q] = cscale(u[q], scale);
    t += cabs2(u[q]);
  }
  t = row16_sum(t);
  const double f = t > 0.0 ? len / sqrt(t) : 0.0;
#pragma unroll
  for (int q = 0; q < SMALL_MAX_COLS / 16; ++q) u[q] = cscale(u[q], f);
}

template <typename S, int NT, int CAP>
__global__ __launch_bounds__(NT) void k_gate_small(const GateTask* tasks) {
  __shared__ GateTask T;
  __shared__ double2 sX[CAP], sY[CAP];
  __shared__ double s_sig[SMALL_MAX_ROWS], s_scy[SMALL_MAX_ROWS], s_scw[SMALL_MAX_ROWS], s_inv[SMALL_MAX_ROWS];
  __shared__ double2 s_d[SMALL_MAX_ROWS];
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
  // NaN / Inf anywhere in theta': the LQ drops what is right of a row's diagonal when its tail is a NaN, so the
  // norms of the rows it leaves need not show it
  if (tid == 0 && !(f2 <= DBL_MAX)) s_bad = 1;
  __syncthreads();
  const int sweeps = svd_rows<NT>(sY, stride, r, T.c, T.tol, JAC_FLOOR2 * f2, T.max_sweeps, &s_flag, s_inv, s_d);
  __syncthreads();
  sort_rows<NT>(sY, stride, r, r, s_inv, s_sig, s_perm, &s_bad);
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
      // Of the index kept below the cutoff, a row under the floor of the sweeps is rounding residue: its vectors, of
      // length sqrt(sigma) in the sites, would come back in the next theta' as a singular value far above both.
      const bool residue = pn < T.cutoff && !(sg * sg > JAC_FLOOR2 * f2);
      if (lane < K && sg > 1e-150 && !residue) {
        // exponents of f sigma: left aL, right 1 - aL; Y's side is the left one unless transposed
        const double sf = sg * f, h = sqrt(sf);
        const double left = T.absorb == 0 ? h : 1.0, right = T.absorb == 0 ? h : sf;
        gy = (tr ? right : left) / sg;
        gw = tr ? left : right;
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
  for (int e = tid; e < K * r; e += NT) {
    if (!tr) {
      const int i = e / K, k = e - i * K;
      st(Oi, left(i, k), cscale(cconj(sY[s_perm[k] * stride + i]), s_scy[k]));
    } else {
      const int k = e / r, i = e - k * r;
      st(Oj, (size_t)e, cscale(sY[s_perm[k] * stride + i], s_scy[k]));
    }
  }
  // ---- the other factor: the kept rows of Y on X, each vector scaled to its length ----
  for (int k0 = 2 * group; k0 < K; k0 += NT / 8) {
    const int k1 = min(k0 + 1, K - 1);
    double2 u[2][SMALL_MAX_COLS / 16];
    other_side(sX, sY + s_perm[k0] * stride, sY + s_perm[k1] * stride, stride, r, T.c, u[0], u[1]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = h ? k1 : k0;
      to_length(u[h], s_inv[k], s_scw[k]);
#pragma unroll
      for (int q = 0; q < SMALL_MAX_COLS / 16; ++q) {
        const int j = l16 + 16 * q;
        if (j >= T.c) continue;
        if (!tr) st(Oj, (size_t)k * n + j, u[h][q]);
        else st(Oi, left(j, k), cconj(u[h][q]));
      }
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

// One vector per 16 lanes: u[i] = <y, X row i> * scale for the rows i = l16 + 16 q < r; returns the sum of |u|^2
// over all rows.  The lanes start at different columns, for rows that start in the same LDS bank.
__device__ __forceinline__ double other_rows(const double2* X, const double2* y, int stride, int r, int c,
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
  const int sweeps = jacobi_rows_n<NT>(sY, stride, nr, stride - 1, T.tol, 0.0, T.max_sweeps, &s_flag, s_tmp);
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
    const double t = other_rows(sX, sY + s_perm[j] * stride, stride, r, c, sg > 1e-150 ? 1.0 / sg : 0.0, u);
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
__global__ __launch_bounds__(CHAIN_THREADS) void k_env_chain(const ChainSite* sites, int n, const double* diags,
                                                             double* out) {
  constexpr int B = CHAIN_MAX_BOND, NT = CHAIN_THREADS, Q = B * B / NT;
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
      al[q] = (i0 + NT * q) / cr;
      ar[q] = (i0 + NT * q) - al[q] * cr;
    }
    auto has = [&](int q, int count) { return on && (q == 0 || slots == 1) && i0 + NT * q < count; };
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
        if (has(q, na)) sA[slot * na + i0 + NT * q] = next[q];
      __syncthreads();
      if (sb + slots < s1) fetch(s + slots);
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (has(q, na)) {
          double2 x = make_double2(0, 0);
          for (int l = 0; l < cl; ++l) x = cfma(sE[al[q] * cl + l], eA[l * cr + ar[q]], x);
          eX[i0 + NT * q] = x;
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
        if (has(q, ne)) sE[i0 + NT * q] = acc[q];
    }
    __syncthreads();
  }
  if (tid == 0) out[blockIdx.x] = sE[0].x;
}

hipError_t launch_env_chain(const ChainSite* d_sites, int n, const double* d_diags, double* d_out, int nchains,
                            int fp32, hipStream_t s) {
  if (nchains <= 0) return hipSuccess;
  if (fp32) hipLaunchKernelGGL(k_env_chain<float2>, dim3(nchains), dim3(CHAIN_THREADS), 0, s, d_sites, n, d_diags, d_out);
  else hipLaunchKernelGGL(k_env_chain<double2>, dim3(nchains), dim3(CHAIN_THREADS), 0, s, d_sites, n, d_diags, d_out);
  return hipGetLastError();
}

}  // namespace hipmps
