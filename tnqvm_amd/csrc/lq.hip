// lq.hip -- blocked Householder LQ (row-oriented) used to precondition the one-sided Jacobi SVD.
//
// For X (r x c, r <= c):  X = L Q~  (L lower triangular, Q~ orthonormal rows), then
// L^H = L_Z Q_Z and the Jacobi runs on the rows of R2 = L_Z^H.  X = Q_Z^H R2 Q~, so X and R2
// share their singular values and the right singular vectors of X are those of R2 mapped
// through Q~; the Jacobi's final rows Y_J (sigma_k v_k^H) become [Y_J | 0] Q~.  The two QR
// steps make R2 close to diagonal with a graded diagonal, and the Jacobi needs about a third
// fewer sweeps at 512 x 512 (Drmac & Veselic, SIAM J. Matrix Anal. Appl. 29 (2008) 1322,
// there with column pivoting; unpivoted here, which measured the same on MPS matrices).
//
// Reflectors act on rows from the right: y -> y - 2 <y, w> w with <y, w> = sum_l y_l conj(w_l)
// and w a unit row vector.  A panel of 16 reflectors w_k0 .. w_k0+15 composes to
// H_k0 ... H_k0+15 = I - W^H T W (W the 16 reflector rows, T upper triangular, T_jj = 2,
// T_{0:j,j} = -2 T_{0:j,0:j} G_{0:j,j}, G_ij = <w_i, w_j>); its inverse is I - W^H T^H W.
// Panels of 16 rows: 32-row panels halve the passes over the trailing matrix but put twice as
// long a serial factorization on every launch's critical path, and measured slower.
#include "kernels.h"
#include "device_util.h"

namespace hipmps {

constexpr int LQB = 16;  // rows per panel (reflectors per block reflector)
constexpr int LQR = 16;  // rows per MFMA tile in the block-reflector application
constexpr long long LQ_ONE_STREAM_ROWS = 4096;  // launch_lq_lookahead: rows of all tasks on one stream up to this

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

// Element w_k[col] of reflector k of M (support col >= k; head in W0, tail in M's row k).
__device__ __forceinline__ double2 refl(const double2* M, size_t ld, const double2* W0, int k, int col) {
  if (col < k) return make_double2(0, 0);
  return gld(col == k ? W0 + k : M + (size_t)k * ld + col);
}

// Factor rows [k0, k0 + 16) of T.M over columns [k0, cols) and form the panel's T factor.
// Whole workgroup (256 threads); rows stay in memory (L2), each wave updates every fourth row.
__device__ __forceinline__ void lq_factor_panel(const LqTask& T, int k0, double2 (*sG)[LQB + 1], double2 (*sT)[LQB + 1]) {
  double2* M = T.M;
  const size_t ld = T.ld;
  const int C = T.cols;
  const int k1 = min(k0 + LQB, T.rows);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int k = k0; k < k1; ++k) {
    const double2* rk = M + (size_t)k * ld;
    double s = 0.0;
    for (int l = k + 1 + lane; l < C; l += 64) s += cabs2(gld(rk + l));
    s = wave_sum(s);
    const double2 a = gld(rk + k);
    const double nrm = sqrt(cabs2(a) + s);
    double2 beta = make_double2(0, 0), w0 = make_double2(0, 0);
    double scale = 0.0;
    if (nrm > 0.0) {
      const double aa = sqrt(cabs2(a));
      const double2 ph = aa > 0.0 ? cscale(a, 1.0 / aa) : make_double2(1.0, 0.0);
      beta = cscale(ph, -nrm);  // -e^{i arg a} |x|: no cancellation in a - beta
      const double2 v0 = make_double2(a.x - beta.x, a.y - beta.y);
      scale = 1.0 / sqrt(cabs2(v0) + s);
      w0 = cscale(v0, scale);
    }
    // remaining rows of the panel: y -= 2 <y, w> w
    for (int i = k + 1; i < k1; ++i) {
      if (((i - k0) & 3) != wave) continue;
      double2* yi = M + (size_t)i * ld;
      double2 d = lane == 0 ? cfmac(w0, gld(yi + k), make_double2(0, 0)) : make_double2(0, 0);
      for (int l = k + 1 + lane; l < C; l += 64) d = cfmac(cscale(gld(rk + l), scale), gld(yi + l), d);
      d = wave_sum2(d);  // <y, w> = sum y_l conj(w_l)  (cfmac(a, b) adds conj(a) b)
      const double2 m2d = cscale(d, -2.0);
      if (lane == 0) gst(yi + k, cfma(m2d, w0, gld(yi + k)));
      for (int l = k + 1 + lane; l < C; l += 64) gst(yi + l, cfma(m2d, cscale(gld(rk + l), scale), gld(yi + l)));
    }
    __syncthreads();  // every read of row k done
    for (int l = k + 1 + tid; l < C; l += 256) gst(M + (size_t)k * ld + l, cscale(gld(rk + l), scale));
    if (tid == 0) {
      gst(M + (size_t)k * ld + k, beta);
      gst(T.W0 + k, w0);
    }
    __syncthreads();
  }
  // G_ij = <w_i, w_j> for i < j (common support starts at column k0 + j)
  for (int i = 0; i < LQB; ++i) {
    if ((i & 3) != wave) continue;
    for (int j = i + 1; j < LQB; ++j) {
      double2 d = make_double2(0, 0);
      if (k0 + j < k1)
        for (int l = k0 + j + lane; l < C; l += 64)
          d = cfmac(refl(M, ld, T.W0, k0 + j, l), refl(M, ld, T.W0, k0 + i, l), d);
      d = wave_sum2(d);
      if (lane == 0) sG[i][j] = d;
    }
  }
  __syncthreads();
  // T (upper triangular), column by column: T_jj = 2 (0 past the last row of the panel),
  // T_ij = -2 sum_{i <= m < j} T_im G_mj for i < j
  for (int j = 0; j < LQB; ++j) {
    if (tid < LQB) {
      double2 v = make_double2(0, 0);
      if (tid < j) {
        for (int m = tid; m < j; ++m) v = cfma(sT[tid][m], sG[m][j], v);
        v = cscale(v, -2.0);
      } else if (tid == j) {
        v = make_double2(k0 + j < k1 ? 2.0 : 0.0, 0.0);
      }
      sT[tid][j] = v;
    }
    __syncthreads();
  }
  double2* Tp = T.T + (size_t)(k0 / LQB) * LQB * LQB;
  for (int e = tid; e < LQB * LQB; e += 256) gst(Tp + e, sT[e / LQB][e % LQB]);
  __syncthreads();
}

// Rows [r0, r0 + 16) (clipped to r1) of Y (ld ly): Y <- Y (I - W^H T' W) over columns [k0, C),
// T' = T (conjT = 0) or T^H (conjT = 1), W the LQB reflector rows of the panel at k0.
// P = Y W^H (16 x LQB) by MFMA with the column range split over the 4 waves and the next
// 4-column unit prefetched, Q = P T' with T' staged in LDS, then Y -= Q W by MFMA, each wave
// owning whole 16-column tiles.  Run by teams of four waves (a workgroup of 256 threads is one
// team, one of 512 threads two, each with rows and LDS of its own).
__device__ __forceinline__ void lq_apply_panel(const LqTask& T, int k0, double2* Y, size_t ly, int r0, int r1, int conjT,
                               double2 (*sP)[LQB + 1], double2 (*sQ)[LQB + 1], double2 (*sT)[LQB + 1]) {
  const double2* M = T.M;
  const size_t ld = T.ld;
  const int C = T.cols;
  const int tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, k4 = lane >> 4;
  const int k1 = min(k0 + LQB, T.rows);
  const bool rowok = r0 + l16 < r1;
  const double2* yrow = Y + (size_t)(r0 + l16) * ly;
  constexpr int NG = LQB / LQR;  // 16-column groups of P
  auto wload = [&](int j, int col) -> double2 {
    return (j < k1 && col < C) ? refl(M, ld, T.W0, j, col) : make_double2(0, 0);
  };
  // ---- P[i][j] = sum_c Y[r0+i][c] conj(w_j[c]); B operand of group g: reflector k0 + 16g + l16 ----
  mfma_d4 pr[NG], pim[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    pr[g] = mfma_d4{0, 0, 0, 0};
    pim[g] = mfma_d4{0, 0, 0, 0};
  }
  const int nu = (C - k0 + 3) >> 2;
  int u = wave;
  int col = k0 + 4 * u + k4;
  double2 a = (u < nu && rowok && col < C) ? gld(yrow + col) : make_double2(0, 0);
  double2 wv[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) wv[g] = u < nu ? wload(k0 + LQR * g + l16, col) : make_double2(0, 0);
  for (; u < nu; u += 4) {
    const double2 x = a;
    double2 y[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) y[g] = wv[g];
    const int ncol = col + 16;
    const bool nok = u + 4 < nu;
    a = (nok && rowok && ncol < C) ? gld(yrow + ncol) : make_double2(0, 0);
#pragma unroll
    for (int g = 0; g < NG; ++g) wv[g] = nok ? wload(k0 + LQR * g + l16, ncol) : make_double2(0, 0);
    col = ncol;
    // x conj(y): re = x.x y.x + x.y y.y, im = x.y y.x - x.x y.y
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      pr[g] = mfma64(x.x, y[g].x, pr[g]);
      pr[g] = mfma64(x.y, y[g].y, pr[g]);
      pim[g] = mfma64(x.y, y[g].x, pim[g]);
      pim[g] = mfma64(-x.x, y[g].y, pim[g]);
    }
  }
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          double2 e = make_double2(pr[g][v], pim[g][v]);
          if (w) e = cadd(e, sP[4 * v + k4][LQR * g + l16]);
          sP[4 * v + k4][LQR * g + l16] = e;
        }
    }
    __syncthreads();
  }
  // ---- Q = P T' (16 x LQB), T' staged 16 rows at a time in sT ----
  {
    const double2* Tp = T.T + (size_t)(k0 / LQB) * LQB * LQB;
    double2 q[NG];
    const int i = tid >> 4, j0 = tid & 15;
#pragma unroll
    for (int h = 0; h < NG; ++h) {  // rows 16h .. 16h + 15 of T'
      for (int e = tid; e < LQR * LQB; e += 256) {
        const int m = e / LQB, j = e % LQB, mm = LQR * h + m;
        sT[m][j] = conjT ? cconj(gld(Tp + j * LQB + mm)) : gld(Tp + mm * LQB + j);
      }
      __syncthreads();
#pragma unroll
      for (int x = 0; x < NG; ++x) {
        const int j = j0 + LQR * x;
        double2 acc = h ? q[x] : make_double2(0, 0);
#pragma unroll 4
        for (int m = 0; m < LQR; ++m) acc = cfma(sP[i][LQR * h + m], sT[m][j], acc);
        q[x] = acc;
      }
      __syncthreads();
    }
#pragma unroll
    for (int x = 0; x < NG; ++x) sQ[i][LQR * x + j0] = q[x];
  }
  __syncthreads();
  // ---- Y -= Q W over 16-column tiles ----
  double qr[LQB / 4], qi[LQB / 4];
#pragma unroll
  for (int kk = 0; kk < LQB / 4; ++kk) {
    const double2 q = sQ[l16][kk * 4 + k4];  // A[i][k] = Q[i][j], j = 4kk + k
    qr[kk] = q.x;
    qi[kk] = q.y;
  }
  const int nt = (C - k0 + 15) >> 4;
  for (int t = wave; t < nt; t += 4) {
    const int c0 = k0 + 16 * t + l16;
    mfma_d4 dr = {0, 0, 0, 0}, di = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < LQB / 4; ++kk) {
      const double2 w = wload(k0 + kk * 4 + k4, c0);  // B[k][c] = w_j[c]
      dr = mfma64(qr[kk], w.x, dr);
      dr = mfma64(-qi[kk], w.y, dr);
      di = mfma64(qr[kk], w.y, di);
      di = mfma64(qi[kk], w.x, di);
    }
    if (c0 < C) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + 4 * v + k4;
        if (row < r1) {
          double2* yp = Y + (size_t)row * ly + c0;
          const double2 y = gld(yp);
          gst(yp, make_double2(y.x - dr[v], y.y - di[v]));
        }
      }
    }
  }
  __syncthreads();  // sP / sQ are reused by the caller
}

__global__ __launch_bounds__(256) void k_lq_panel0(const LqTask* tasks) {
  __shared__ double2 sG[LQB][LQB + 1];
  __shared__ double2 sT[LQB][LQB + 1];
  const LqTask& T = tasks[blockIdx.x];
  if (T.rows <= 0) return;
  lq_factor_panel(T, 0, sG, sT);
}

// Trailing update with panel p (k1 = end of panel p): workgroup (0, task) owns the rows of
// panel p + 1, [k1, k1 + LQB), updates them and then factors them; workgroup (x > 0, task)
// owns rows [k1 + LQB + 16 (x - 1), + 16).
__global__ __launch_bounds__(256) void k_lq_update(const LqTask* tasks, int p) {
  __shared__ double2 sP[LQB][LQB + 1];
  __shared__ double2 sQ[LQB][LQB + 1];
  __shared__ double2 sT[LQR][LQB + 1];
  const LqTask& T = tasks[blockIdx.y];
  const int k0 = p * LQB;
  if (k0 >= T.rows) return;
  const int k1 = min(k0 + LQB, T.rows);
  if (blockIdx.x == 0) {
    if (k1 >= T.rows) return;
    const int e1 = min(k1 + LQB, T.rows);
    for (int r0 = k1; r0 < e1; r0 += LQR) lq_apply_panel(T, k0, T.M, T.ld, r0, e1, 0, sP, sQ, sT);
    lq_factor_panel(T, k1, sP, sQ);
    return;
  }
  const int r0 = k1 + LQB + LQR * ((int)blockIdx.x - 1);
  if (r0 >= T.rows) return;
  lq_apply_panel(T, k0, T.M, T.ld, r0, min(r0 + LQR, T.rows), 0, sP, sQ, sT);
}

// Tgt <- Tgt (I - W_p^H T_p^H W_p) for every panel p from the last to the first, on rows [16x, 16x +
// 16) of Tgt: the rows are independent of each other, so one launch applies all panels, each
// workgroup to its rows (one launch a panel left gaps of several us between launches of 7 to 20 us).
__global__ __launch_bounds__(256) void k_lq_apply_q(const LqTask* tasks) {
  __shared__ double2 sP[LQB][LQB + 1];
  __shared__ double2 sQ[LQB][LQB + 1];
  __shared__ double2 sT[LQR][LQB + 1];
  const LqTask& T = tasks[blockIdx.x];
  const int r0 = LQR * (int)blockIdx.y;
  if (r0 >= T.rows_t) return;
  for (int p = (T.rows - 1) / LQB; p >= 0; --p)
    lq_apply_panel(T, p * LQB, T.Tgt, T.ld_t, r0, min(r0 + LQR, T.rows_t), 1, sP, sQ, sT);
}

// dst[i][j] = conj(src[j][i]) for j >= i and i < n, 0 otherwise (the conjugate transpose of
// src's lower triangle, an upper-triangular n x n matrix); rows n .. rows_dst - 1 are zero.
__global__ __launch_bounds__(256) void k_lower_to_upper_h(const TriTask* tasks) {
  __shared__ double2 tile[32][33];
  const TriTask& T = tasks[blockIdx.z];
  const int n = T.n;
  const int i0 = blockIdx.y * 32, j0 = blockIdx.x * 32;
  if (i0 >= T.rows_dst || j0 >= n) return;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int y = ty; y < 32; y += 8) {  // src rows j0 + y, columns i0 + tx
    const int r = j0 + y, c = i0 + tx;
    tile[y][tx] = (r < n && c < n && r >= c) ? T.src[(size_t)r * T.ld_src + c] : make_double2(0, 0);
  }
  __syncthreads();
  for (int y = ty; y < 32; y += 8) {
    const int i = i0 + y, j = j0 + tx;
    if (i < T.rows_dst && j < n) T.dst[(size_t)i * T.ld_dst + j] = cconj(tile[tx][y]);
  }
}

__global__ __launch_bounds__(256) void k_widen(const TriTask* tasks) {
  const TriTask& T = tasks[blockIdx.y];
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t total = (size_t)T.rows_dst * T.ld_dst;
  if (e >= total) return;
  const int i = (int)(e / T.ld_dst), j = (int)(e % T.ld_dst);
  T.dst[e] = j < T.n ? T.src[(size_t)i * T.ld_src + j] : make_double2(0, 0);
}

// ---- factorisation with the panel in registers ------------------------------------------------
struct LqStepShared {
  double2 P[2][LQB][LQB + 1], Q[2][LQB][LQB + 1], T[2][LQR][LQB + 1];  // lq_apply_panel, per team
  double2 w0[LQB];
};

// Factor rows [k0, k1) of T.M (panel p) over columns [k0, cols), at most 64 NC of them, with the
// panel in registers: wave w of eight holds the rows w and w + 8, lane l the columns l + 64 j.  The
// reflectors are those of lq_factor_panel.  Per reflector, its row w_r goes to LDS (zero before column
// r), every wave forms the inner products of its rows with it -- <y_i, w_r> updates a row i > r, and
// is G_ir of the T factor for a row i < r -- and the wave with row r + 1 goes on to the next reflector
// as soon as that row is updated; T's column r - 1 is formed by another wave meanwhile.  One barrier
// per reflector.  Bound by that serial chain; with the rows in LDS and shuffle reductions a panel of
// 128 .. 512 columns took 48 .. 59 us, this form @US@.
template <int NC>
__device__ __forceinline__ void lq_factor_regs(const LqTask& T, int p, LqStepShared& S, double2* srow) {
  const int k0 = p * LQB;
  const int k1 = min(k0 + LQB, T.rows), nr = k1 - k0;
  const int W = T.cols - k0;  // local column c = column - k0
  double2* M = T.M + (size_t)k0 * T.ld + k0;
  const size_t ld = T.ld;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  double2 (*sG)[LQB + 1] = S.P[0];
  double2 (*sT)[LQB + 1] = S.T[0];
  double2 y[2][NC];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int i = wave + 8 * h, c = lane + 64 * j;
      y[h][j] = (i < nr && c < W) ? gld(M + (size_t)i * ld + c) : make_double2(0, 0);
    }
  if (tid < LQB * LQB) sG[tid / LQB][tid % LQB] = sT[tid / LQB][tid % LQB] = make_double2(0, 0);
  // reflector of row r, held by this wave in y[h]: w into srow[r & 1], beta and the scaled tail in place
  auto reflector = [&](double2 (&v)[NC], int r) __attribute__((always_inline)) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (j > 0 || lane > r) s += cabs2(v[j]);
    s = wave_sum(s);
    const double2 a = make_double2(lane_value(v[0].x, r), lane_value(v[0].y, r));
    const double nrm = sqrt(cabs2(a) + s);
    double2 beta = make_double2(0, 0), w0 = make_double2(0, 0);
    double scale = 0.0;
    if (nrm > 0.0) {
      const double aa = sqrt(cabs2(a));
      const double2 ph = aa > 0.0 ? cscale(a, 1.0 / aa) : make_double2(1.0, 0.0);
      beta = cscale(ph, -nrm);  // -e^{i arg a} |x|: no cancellation in a - beta
      const double2 v0 = make_double2(a.x - beta.x, a.y - beta.y);
      scale = 1.0 / sqrt(cabs2(v0) + s);
      w0 = cscale(v0, scale);
    }
    double2* row = srow + (r & 1) * NC * 64;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const double2 t = cscale(v[j], scale);
      if (j > 0) {
        v[j] = t;
        row[lane + 64 * j] = t;
      } else {
        row[lane] = make_double2(lane > r ? t.x : (lane == r ? w0.x : 0.0), lane > r ? t.y : (lane == r ? w0.y : 0.0));
        v[0] = make_double2(lane > r ? t.x : (lane == r ? beta.x : v[0].x),
                            lane > r ? t.y : (lane == r ? beta.y : v[0].y));
      }
    }
    if (lane == 0) S.w0[r] = w0;
  };
  // column j of T (T_jj = 2, T_ij = -2 sum_{i <= m < j} T_im G_mj): four lanes a row
  auto t_column = [&](int j) __attribute__((always_inline)) {
    const int i = lane >> 2, q = lane & 3;
    double2 t = make_double2(0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = q + 4 * e;
      if (m >= i && m < j) t = cfma(sT[i][m], sG[m][j], t);
    }
    t.x = dpp_add<0x4e>(dpp_add<0xb1>(t.x));
    t.y = dpp_add<0x4e>(dpp_add<0xb1>(t.y));
    if (q == 0 && i <= j) sT[i][j] = i == j ? make_double2(2.0, 0.0) : cscale(t, -2.0);
  };
  double2 w[NC];
  auto inner = [&](const double2 (&v)[NC]) __attribute__((always_inline)) {  // <v, w> = sum v conj(w)
    double2 d = make_double2(0, 0);
#pragma unroll
    for (int j = 0; j < NC; ++j) d = cfmac(w[j], v[j], d);
    return wave_sum2(d);
  };
  auto update = [&](double2 (&v)[NC]) __attribute__((always_inline)) {
    const double2 m2d = cscale(inner(v), -2.0);
#pragma unroll
    for (int j = 0; j < NC; ++j) v[j] = cfma(m2d, w[j], v[j]);
  };
  auto gram = [&](const double2 (&v)[NC], int i, int r) __attribute__((always_inline)) {
    const double2 d = inner(v);
    if (lane == 0) sG[i][r] = d;
  };
  auto load_w = [&](int r) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NC; ++j) w[j] = srow[(r & 1) * NC * 64 + lane + 64 * j];
  };
  if (wave == 0 && nr > 0) reflector(y[0], 0);
  __syncthreads();
  // pivots 0 .. 6: the next pivot is among the rows 0 .. 7, the rows 8 .. 15 all update
#pragma unroll 1
  for (int r = 0; r < min(nr, 7); ++r) {
    load_w(r);
    if (wave > r) {
      update(y[0]);
      if (wave == r + 1 && wave < nr) reflector(y[0], r + 1);
    } else if (wave < r) {
      gram(y[0], wave, r);
    }
    update(y[1]);
    if (r > 0 && wave == ((r + 4) & 7)) t_column(r - 1);
    __syncthreads();
  }
  // pivots 7 .. 15: the next pivot is among the rows 8 .. 15, the rows 0 .. 7 are done
#pragma unroll 1
  for (int r = 7; r < nr; ++r) {
    load_w(r);
    if (wave + 8 > r) {
      update(y[1]);
      if (wave + 8 == r + 1 && r + 1 < nr) reflector(y[1], r + 1);
    } else if (wave + 8 < r) {
      gram(y[1], wave + 8, r);
    }
    if (wave < r) gram(y[0], wave, r);
    if (wave == ((r + 4) & 7)) t_column(r - 1);
    __syncthreads();
  }
  if (nr > 0 && wave == 0) t_column(nr - 1);
  __syncthreads();
  double2* Tp = T.T + (size_t)p * LQB * LQB;
  if (tid < LQB * LQB) gst(Tp + tid, sT[tid / LQB][tid % LQB]);
  if (tid < nr) gst(T.W0 + k0 + tid, S.w0[tid]);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int i = wave + 8 * h, c = lane + 64 * j;
      if (i < nr && c < W) gst(M + (size_t)i * ld + c, y[h][j]);
    }
}

// One panel's step, p = -1 .. panels - 2: workgroup (task, 0) applies the block reflector of panel p
// to the rows of panel p + 1 and factors them; workgroup (task, x > 0) applies it to the 32 rows
// from k0 + 2 LQB + 32 (x - 1) (two teams of four waves).  The factoring workgroups come first.
template <int NC>
__global__ __launch_bounds__(512) void k_lq_step(const LqTask* tasks, int p) {
  __shared__ LqStepShared S;
  __shared__ double2 srow[2 * NC * 64];
  const LqTask& T = tasks[blockIdx.x];
  const int team = threadIdx.x >> 8;
  const int k0 = p * LQB, k1 = k0 + LQB;
  if (k1 >= T.rows) return;
  if (blockIdx.y == 0) {
    const int e1 = min(k1 + LQB, T.rows);
    if (p >= 0) lq_apply_panel(T, k0, T.M, T.ld, k1, team ? k1 : e1, 0, S.P[team], S.Q[team], S.T[team]);
    lq_factor_regs<NC>(T, p + 1, S, srow);
    return;
  }
  const int r0 = k1 + LQB + 2 * LQR * ((int)blockIdx.y - 1);
  if (r0 >= T.rows) return;
  const int rt = min(r0 + LQR * team, T.rows);
  lq_apply_panel(T, k0, T.M, T.ld, rt, min(rt + LQR, T.rows), 0, S.P[team], S.Q[team], S.T[team]);
}

// Rows beyond panel p + 1 with the block reflector of panel p, 16 rows per workgroup
__global__ __launch_bounds__(256) void k_lq_rest(const LqTask* tasks, int p) {
  __shared__ double2 sP[LQB][LQB + 1];
  __shared__ double2 sQ[LQB][LQB + 1];
  __shared__ double2 sT[LQR][LQB + 1];
  const LqTask& T = tasks[blockIdx.x];
  const int k0 = p * LQB;
  const int r0 = k0 + 2 * LQB + LQR * (int)blockIdx.y;
  if (r0 >= T.rows) return;
  lq_apply_panel(T, k0, T.M, T.ld, r0, min(r0 + LQR, T.rows), 0, sP, sQ, sT);
}

hipError_t launch_lq_lookahead(const LqTask* d_tasks, int ntasks, int max_rows, int max_cols, hipStream_t sa,
                               hipStream_t sb, hipEvent_t ea, hipEvent_t eb) {
  if (ntasks <= 0 || max_rows <= 0) return hipSuccess;
  if (max_cols > LQ_REG_MAX_COLS) return hipErrorNotSupported;
  const int panels = (max_rows + LQB - 1) / LQB;
  // columns per lane of the panel's registers; the results are the same for every NC that holds them
  auto step = [&](int p, int blocks) {
    const int w = max_cols - (p + 1) * LQB;
    const dim3 g(ntasks, blocks), b(512);
    if (w <= 128) hipLaunchKernelGGL(k_lq_step<2>, g, b, 0, sa, d_tasks, p);
    else if (w <= 256) hipLaunchKernelGGL(k_lq_step<4>, g, b, 0, sa, d_tasks, p);
    else if (w <= 512) hipLaunchKernelGGL(k_lq_step<8>, g, b, 0, sa, d_tasks, p);
    else hipLaunchKernelGGL(k_lq_step<16>, g, b, 0, sa, d_tasks, p);
  };
  // Few trailing rows: one launch per panel for both, on one stream.  Many: the trailing update in
  // workgroups of its own (a third of the registers) on the second stream, beside the next panel.
  if ((long long)ntasks * max_rows <= LQ_ONE_STREAM_ROWS || sb == nullptr) {
    for (int p = -1; p + 1 < panels; ++p) {
      const int trailing = p < 0 ? 0 : max_rows - (p + 2) * LQB;
      step(p, 1 + (trailing > 0 ? (trailing + 2 * LQR - 1) / (2 * LQR) : 0));
    }
    return hipGetLastError();
  }
  hipError_t e = hipSuccess;
  // sb starts after what sa has queued so far (the matrices are ready there)
  if ((e = hipEventRecord(ea, sa)) != hipSuccess) return e;
  if ((e = hipStreamWaitEvent(sb, ea, 0)) != hipSuccess) return e;
  step(-1, 1);
  if ((e = hipEventRecord(ea, sa)) != hipSuccess) return e;
  for (int p = 0; p + 1 < panels; ++p) {
    // sa: rows of panel p + 1 need the rest-update of panel p - 1 (recorded in eb), sb: the rest
    // update of panel p needs panel p's reflectors (recorded in ea); both waits are enqueued before
    // the events are recorded again below
    if (p > 0 && (e = hipStreamWaitEvent(sa, eb, 0)) != hipSuccess) return e;
    if ((e = hipStreamWaitEvent(sb, ea, 0)) != hipSuccess) return e;
    step(p, 1);
    if ((e = hipEventRecord(ea, sa)) != hipSuccess) return e;
    const int trailing = max_rows - (p + 2) * LQB;
    if (trailing > 0)
      hipLaunchKernelGGL(k_lq_rest, dim3(ntasks, (trailing + LQR - 1) / LQR), dim3(256), 0, sb, d_tasks, p);
    if ((e = hipEventRecord(eb, sb)) != hipSuccess) return e;
  }
  // everything after this on sa sees both streams' work
  if ((e = hipEventRecord(eb, sb)) != hipSuccess) return e;
  if ((e = hipStreamWaitEvent(sa, eb, 0)) != hipSuccess) return e;
  return hipGetLastError();
}

hipError_t launch_widen(const TriTask* d_tasks, int ntasks, int max_cols, int max_rows_dst, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  const size_t total = (size_t)max_cols * max_rows_dst;
  hipLaunchKernelGGL(k_widen, dim3((unsigned)((total + 255) / 256), ntasks), dim3(256), 0, s, d_tasks);
  return hipGetLastError();
}

hipError_t launch_lq(const LqTask* d_tasks, int ntasks, int max_rows, hipStream_t s) {
  if (ntasks <= 0 || max_rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_lq_panel0, dim3(ntasks), dim3(256), 0, s, d_tasks);
  const int panels = (max_rows + LQB - 1) / LQB;
  for (int p = 0; p + 1 < panels; ++p) {
    const int trailing = max_rows - (p + 1) * LQB;  // > 0
    const int blocks = 1 + (trailing > LQB ? (trailing - LQB + LQR - 1) / LQR : 0);
    hipLaunchKernelGGL(k_lq_update, dim3(blocks, ntasks), dim3(256), 0, s, d_tasks, p);
  }
  return hipGetLastError();
}

hipError_t launch_lq_apply_q(const LqTask* d_tasks, int ntasks, int max_rows, int max_rows_t, hipStream_t s) {
  if (ntasks <= 0 || max_rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_lq_apply_q, dim3(ntasks, (max_rows_t + LQR - 1) / LQR), dim3(256), 0, s, d_tasks);
  return hipGetLastError();
}

hipError_t launch_lower_to_upper_h(const TriTask* d_tasks, int ntasks, int max_n, int max_rows_dst, hipStream_t s) {
  if (ntasks <= 0 || max_n <= 0) return hipSuccess;
  dim3 grid((max_n + 31) / 32, (max_rows_dst + 31) / 32, ntasks);
  hipLaunchKernelGGL(k_lower_to_upper_h, grid, dim3(256), 0, s, d_tasks);
  return hipGetLastError();
}

// Rank cut of the preconditioned factor J (n x n, ld_dst; TriTask.dst, .n): rows whose squared
// norm is below 1e-28 ||J||_F^2 are set to zero before the sweeps.  Zeroing them perturbs J by
// at most 1e-14 sqrt(n) ||J||_F, which bounds the change of every singular value (Weyl); the cut
// is made only where that bound is below 1e-3 of sigma_cut[t], the singular value under which
// the truncation drops an index, so neither a kept value nor the bond dimension moves.  Rows of
// rounding noise (a rank-deficient theta', as on purified sites) then no longer keep the
// relative convergence test rotating; a full-rank J is only read.
__global__ __launch_bounds__(256) void k_rank_cut(const TriTask* tasks, const double* sigma_cut) {
  __shared__ double rn[4096];
  __shared__ double red[4];
  __shared__ double s_thr;
  const TriTask& T = tasks[blockIdx.x];
  const double cut = sigma_cut[blockIdx.x];
  if (!(cut > 0.0)) return;
  const int n = T.n;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  double part = 0.0;
  for (int i = wave; i < n; i += 4) {
    const double2* row = T.dst + (size_t)i * T.ld_dst;
    double a = 0.0;
    for (int j = lane; j < n; j += 64) a += cabs2(row[j]);
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
    if (lane == 0) rn[i] = a;
    part += a;
  }
  if (lane == 0) red[wave] = part;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double fro2 = red[0] + red[1] + red[2] + red[3];
    s_thr = (1e-14 * sqrt((double)n * fro2) <= 1e-3 * cut) ? 1e-28 * fro2 : -1.0;
  }
  __syncthreads();
  const double thr = s_thr;
  if (thr < 0.0) return;
  for (int i = wave; i < n; i += 4) {
    if (rn[i] >= thr) continue;
    double2* row = T.dst + (size_t)i * T.ld_dst;
    for (int j = lane; j < n; j += 64) row[j] = make_double2(0.0, 0.0);
  }
}

hipError_t launch_rank_cut(const TriTask* d_tasks, const double* d_sigma_cut, int ntasks, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rank_cut, dim3(ntasks), dim3(256), 0, s, d_tasks, d_sigma_cut);
  return hipGetLastError();
}

}  // namespace hipmps
