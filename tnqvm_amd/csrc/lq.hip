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
constexpr int LQ_TWO_ROWS_COLS = 64 * 16;  // widest panel of which a lane's registers hold two rows
// launch_lq_lookahead: rows of all tasks on one stream up to this.  The line is that of an earlier form of the panel
// kernels, whose workgroups beside the factoring one held its registers.  With these, one stream against two, both
// LQs of a wave alone: 8 of 512 x 512 2.44 for 3.37 ms, 64 of them (32768 rows) 4.29 for 5.51, 32 of 1024 x 1024
// 17.3 for 20.7; the 8-circuit chi 256 load 2375 for 2355 applies/s (two wave groups).  One is the faster at every
// size measured, so the line costs a few percent above it.
constexpr long long LQ_ONE_STREAM_ROWS = 4096;

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
// T' = T (conjT = 0) or T^H (conjT = 1), W the reflector rows [k0, k1) of the panel at k0 (at most
// LQB).  P = Y W^H (16 x LQB) by MFMA with the column range split over the 4 waves, Q = P T' with T'
// staged in LDS, then Y -= Q W by MFMA, each wave owning whole 16-column tiles.  PD units of P and a
// whole tile of the update are in flight.  No load is under a condition (behind a load that may not have
// been issued, the wait for an older one is a wait for all): past the end they repeat the last group, and
// the panel's own columns, where its reflectors start, and columns past the end are put right at use.  Run
// by teams of four waves (a workgroup of 256 threads is one team, one of 512 threads two, each with rows and
// LDS of its own).
template <int PD>
__device__ __forceinline__ void lq_apply_panel(const LqTask& T, int k0, int k1, double2* Y, size_t ly, int r0, int r1,
                                               int conjT, double2 (*sP)[LQR][LQB + 1], double2 (*sQ)[LQB + 1],
                                               double2 (*sT)[LQB + 1]) {
  const double2* M = T.M;
  const double2* W0 = T.W0;
  const size_t ld = T.ld;
  const int C = T.cols;
  const int tid = threadIdx.x & 255, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, k4 = lane >> 4;
  {  // T', wanted after P
    const double2* Tp = T.T + (size_t)(k0 / LQB) * LQB * LQB;
    const int i = tid >> 4, j = tid & 15;
    sT[i][j] = conjT ? cconj(gld(Tp + j * LQB + i)) : gld(Tp + i * LQB + j);
  }
  // 32-bit offsets (gld_at) from the panel's first row and from the first of Y's rows: 16 rows of fewer than
  // LQ_MAX_COLS columns each
  const int y0 = __builtin_amdgcn_readfirstlane(min(r0, r1 - 1));
  const double2* Mk = M + (size_t)k0 * ld;
  Y += (size_t)y0 * ly;
  // a reflector past k1 repeats the last one: its rows and columns of T are zero
  const int jl = min(k0 + l16, k1 - 1);
  const unsigned wrow = (unsigned)(jl - k0) * (unsigned)ld;
  const double2 head = gld_at(W0, jl);  // of reflector k0 + l16
  // element w_j[col] of reflector j (support col >= j; head in W0, tail in M's row j), M's element being v
  auto own = [&](double2 v, double2 h, int j, int col) __attribute__((always_inline)) {
    const bool is_head = col == j, zero = col < j || col >= C;
    return make_double2(zero ? 0.0 : (is_head ? h.x : v.x), zero ? 0.0 : (is_head ? h.y : v.y));
  };
  auto special = [&](int g) { return g == 0 || k0 + 16 * g + 16 > C; };
  // ---- P[i][j] = sum_c Y[r0+i][c] conj(w_j[c]); B operand: reflector k0 + l16 ----
  const unsigned yrow = (unsigned)min(l16, r1 - 1 - y0) * (unsigned)ly;  // a row past the end: a repeat, not stored
  mfma_d4 pr = {0, 0, 0, 0}, pim = {0, 0, 0, 0};
  const int nt = (C - k0 + 15) >> 4;  // 16-column groups; this wave's unit of a group: 4 columns
  const int uo = k0 + 4 * wave + k4;
  double2 a[PD], w[PD];
  auto load = [&](int g, double2& y, double2& m) __attribute__((always_inline)) {
    const unsigned col = min(uo + 16 * g, C - 1);
    y = gld_at(Y, yrow + col);
    m = gld_at(Mk, wrow + col);
  };
#pragma unroll
  for (int d = 0; d < PD; ++d) load(d, a[d], w[d]);
#pragma unroll 1
  for (int d0 = 0; d0 < nt; d0 += PD) {
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      const int g = d0 + d;
      const double2 x = a[d];
      double2 y = w[d];
      load(g + PD, a[d], w[d]);
      if (g >= nt) continue;
      if (special(g)) y = own(y, head, jl, uo + 16 * g);
      // x conj(y): re = x.x y.x + x.y y.y, im = x.y y.x - x.x y.y
      pr = mfma64(x.x, y.x, pr);
      pim = mfma64(x.y, y.x, pim);
      pr = mfma64(x.y, y.y, pr);
      pim = mfma64(-x.x, y.y, pim);
    }
  }
  // first tile of the update, while P is summed
  double2 tw[LQB / 4], ty[4];
  unsigned ry[4], rw[LQB / 4];
#pragma unroll
  for (int v = 0; v < 4; ++v) ry[v] = (unsigned)min(4 * v + k4, r1 - 1 - y0) * (unsigned)ly;
#pragma unroll
  for (int kk = 0; kk < LQB / 4; ++kk) rw[kk] = (unsigned)min(kk * 4 + k4, k1 - 1 - k0) * (unsigned)ld;
  auto tile = [&](int t) __attribute__((always_inline)) {
    const unsigned c = min(k0 + 16 * t + l16, C - 1);
#pragma unroll
    for (int kk = 0; kk < LQB / 4; ++kk) tw[kk] = gld_at(Mk, rw[kk] + c);  // B[k][c] = w_j[c]
#pragma unroll
    for (int v = 0; v < 4; ++v) ty[v] = gld_at(Y, ry[v] + c);
  };
  tile(wave);
#pragma unroll
  for (int v = 0; v < 4; ++v) sP[wave][4 * v + k4][l16] = make_double2(pr[v], pim[v]);
  __syncthreads();
  // ---- Q = P T' (16 x LQB) ----
  {
    const int i = tid >> 4, j = tid & 15;
    double2 p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = sP[q][i][j];
    const double2 sum = cadd(cadd(p[0], p[1]), cadd(p[2], p[3]));
    __syncthreads();
    sP[0][i][j] = sum;
    __syncthreads();
    double2 acc = make_double2(0, 0);
#pragma unroll 4
    for (int m = 0; m < LQB; ++m) acc = cfma(sP[0][i][m], sT[m][j], acc);
    sQ[i][j] = acc;
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
#pragma unroll 1
  for (int t = wave; t < nt; t += 4) {
    const int c = k0 + 16 * t + l16;
    double2 cwv[LQB / 4], cy[4];
#pragma unroll
    for (int kk = 0; kk < LQB / 4; ++kk) cwv[kk] = tw[kk];
#pragma unroll
    for (int v = 0; v < 4; ++v) cy[v] = ty[v];
    tile(t + 4);
    if (special(t)) {
#pragma unroll
      for (int kk = 0; kk < LQB / 4; ++kk) {
        const double2 h = make_double2(__shfl(head.x, kk * 4 + k4), __shfl(head.y, kk * 4 + k4));
        cwv[kk] = own(cwv[kk], h, min(k0 + kk * 4 + k4, k1 - 1), c);
      }
    }
    mfma_d4 dr = {0, 0, 0, 0}, di = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < LQB / 4; ++kk) {
      dr = mfma64(qr[kk], cwv[kk].x, dr);
      di = mfma64(qr[kk], cwv[kk].y, di);
      dr = mfma64(-qi[kk], cwv[kk].y, dr);
      di = mfma64(qi[kk], cwv[kk].x, di);
    }
    if (c < C) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + 4 * v + k4;
        if (row < r1) gst_at(Y, ry[v] + c, make_double2(cy[v].x - dr[v], cy[v].y - di[v]));
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
  __shared__ double2 sP[4][LQR][LQB + 1];
  __shared__ double2 sQ[LQB][LQB + 1];
  __shared__ double2 sT[LQR][LQB + 1];
  const LqTask& T = tasks[blockIdx.y];
  const int k0 = p * LQB;
  if (k0 >= T.rows) return;
  const int k1 = min(k0 + LQB, T.rows);
  if (blockIdx.x == 0) {
    if (k1 >= T.rows) return;
    const int e1 = min(k1 + LQB, T.rows);
    lq_apply_panel<4>(T, k0, k1, T.M, T.ld, k1, e1, 0, sP, sQ, sT);
    lq_factor_panel(T, k1, sP[0], sQ);
    return;
  }
  const int r0 = k1 + LQB + LQR * ((int)blockIdx.x - 1);
  if (r0 >= T.rows) return;
  lq_apply_panel<4>(T, k0, k1, T.M, T.ld, r0, min(r0 + LQR, T.rows), 0, sP, sQ, sT);
}

// Tgt <- Tgt (I - W_p^H T_p^H W_p) for every panel p from the last to the first, on rows [16x, 16x +
// 16) of Tgt: the rows are independent of each other, so one launch applies all panels, each
// workgroup to its rows (one launch a panel left gaps of several us between launches of 7 to 20 us).
__global__ __launch_bounds__(256, 4) void k_lq_apply_q(const LqTask* tasks) {
  __shared__ double2 sP[4][LQR][LQB + 1];
  __shared__ double2 sQ[LQB][LQB + 1];
  __shared__ double2 sT[LQR][LQB + 1];
  const LqTask& T = tasks[blockIdx.x];
  const int r0 = LQR * (int)blockIdx.y;
  if (r0 >= T.rows_t) return;
  for (int p = (T.rows - 1) / LQB; p >= 0; --p)
    lq_apply_panel<2>(T, p * LQB, min(p * LQB + LQB, T.rows), T.Tgt, T.ld_t, r0, min(r0 + LQR, T.rows_t), 1, sP, sQ, sT);
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
  double2 P[2][4][LQR][LQB + 1], Q[2][LQB][LQB + 1], T[2][LQR][LQB + 1];  // lq_apply_panel, per team
  double2 G[LQB][LQB + 1], Tf[LQB][LQB + 1];                           // lq_factor_regs
  double2 w0[LQB];
};

// Factor rows [k0, k1) of T.M (panel p) over columns [k0, cols), at most 64 NC of them, with the
// panel in registers: lane l holds the columns l + 64 j, wave w of eight the rows w and w + 8 (RW = 2),
// or, where two rows of a lane do not fit its registers, first row w and then, after the first eight
// reflectors, row w + 8 (RW = 1).  The reflectors are those of lq_factor_panel.  Per reflector, its
// row w_r goes to LDS (zero before column r), every wave forms the inner products of its rows with it
// -- <y_i, w_r> updates a row i > r, and is G_ir of the T factor for a row i < r -- and the wave with
// row r + 1 goes on to the next reflector as soon as that row is updated; T's column r - 1 is formed by
// another wave meanwhile.  One barrier per reflector.  Bound by that serial chain.  Measured, with the
// update of the panel's rows by the panel before: 24, 31 and 44 us at up to 128, 256 and 512 columns
// (rows in LDS, shuffle reductions: 55, 73 and 100 us), 77 us at 1024 and 193 us at 1536 (rows in L2:
// 350 to 700 us).
template <int NC, int RW>
__device__ __forceinline__ void lq_factor_regs(const LqTask& T, int p, LqStepShared& S, double2* srow) {
  const int k0 = p * LQB;
  const int k1 = min(k0 + LQB, T.rows), nr = k1 - k0;
  const int W = T.cols - k0;  // local column c = column - k0
  double2* M = T.M + (size_t)k0 * T.ld + k0;
  const size_t ld = T.ld;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  double2 (*sG)[LQB + 1] = S.G;
  double2 (*sT)[LQB + 1] = S.Tf;
  constexpr bool WREG = NC <= 16;  // the pivot row in registers too
  double2 y[RW][NC], w[WREG ? NC : 1];
  auto load = [&](double2 (&v)[NC], int i) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = lane + 64 * j;
      v[j] = (i < nr && c < W) ? gld(M + (size_t)i * ld + c) : make_double2(0, 0);
    }
  };
  auto store = [&](const double2 (&v)[NC], int i) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = lane + 64 * j;
      if (i < nr && c < W) gst(M + (size_t)i * ld + c, v[j]);
    }
  };
  // reflector of row r, held by this wave in v: w into srow[r & 1], beta and the scaled tail in place
  auto reflector = [&](double2 (&v)[NC], int r) __attribute__((always_inline)) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (j > 0 || lane > r) s += cabs2(v[j]);
    s = wave_sum(s);
    const double2 a = make_double2(lane_value(v[0].x, r), lane_value(v[0].y, r));
    // reciprocal roots (full_rsq): the library's square roots and divisions one after the other are most of a
    // reflector's scalar chain
    const double a2 = cabs2(a), n2 = a2 + s;
    double2 beta = make_double2(0, 0), w0 = make_double2(0, 0);
    double scale = 0.0;
    if (n2 > 0.0) {
      const double2 ph = a2 > 0.0 ? cscale(a, full_rsq(a2)) : make_double2(1.0, 0.0);
      beta = cscale(ph, -(n2 * full_rsq(n2)));  // -e^{i arg a} |x|: no cancellation in a - beta
      const double2 v0 = make_double2(a.x - beta.x, a.y - beta.y);
      scale = full_rsq(cabs2(v0) + s);
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
  auto pivot = [&](int j, int r) __attribute__((always_inline)) {  // w_r at this lane's column j
    return WREG ? w[WREG ? j : 0] : srow[(r & 1) * NC * 64 + lane + 64 * j];
  };
  auto load_w = [&](int r) __attribute__((always_inline)) {
    if (WREG) {
#pragma unroll
      for (int j = 0; j < NC; ++j) w[WREG ? j : 0] = srow[(r & 1) * NC * 64 + lane + 64 * j];
    }
  };
  auto inner = [&](const double2 (&v)[NC], int r) __attribute__((always_inline)) {  // <v, w> = sum v conj(w)
    double2 d = make_double2(0, 0);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      d = cfmac(pivot(j, r), v[j], d);
      if (!WREG && j % 8 == 7) __builtin_amdgcn_sched_barrier(0);  // 8 LDS reads ahead, not all of them
    }
    return wave_sum2(d);
  };
  auto update = [&](double2 (&v)[NC], int r) __attribute__((always_inline)) {
    const double2 m2d = cscale(inner(v, r), -2.0);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      v[j] = cfma(m2d, pivot(j, r), v[j]);
      if (!WREG && j % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto gram = [&](const double2 (&v)[NC], int i, int r) __attribute__((always_inline)) {
    const double2 d = inner(v, r);
    if (lane == 0) sG[i][r] = d;
  };
  auto store_t = [&]() __attribute__((always_inline)) {
    double2* Tp = T.T + (size_t)p * LQB * LQB;
    if (tid < LQB * LQB) gst(Tp + tid, sT[tid / LQB][tid % LQB]);
    if (tid < nr) gst(T.W0 + k0 + tid, S.w0[tid]);
  };

  if (tid < LQB) S.w0[tid] = make_double2(0, 0);
  if (tid < LQB * LQB) sG[tid / LQB][tid % LQB] = sT[tid / LQB][tid % LQB] = make_double2(0, 0);
  if constexpr (RW == 2) {
    load(y[0], wave);
    load(y[1], wave + 8);
    __syncthreads();
    if (wave == 0 && nr > 0) reflector(y[0], 0);
    __syncthreads();
    // pivots 0 .. 6: the next pivot is among the rows 0 .. 7, the rows 8 .. 15 all update
#pragma unroll 1
    for (int r = 0; r < min(nr, 7); ++r) {
      load_w(r);
      if (wave > r) {
        update(y[0], r);
        if (wave == r + 1 && wave < nr) reflector(y[0], r + 1);
      } else if (wave < r) {
        gram(y[0], wave, r);
      }
      update(y[1], r);
      if (r > 0 && wave == ((r + 4) & 7)) t_column(r - 1);
      __syncthreads();
    }
    // pivots 7 .. 15: the next pivot is among the rows 8 .. 15, the rows 0 .. 7 are done
#pragma unroll 1
    for (int r = 7; r < nr; ++r) {
      load_w(r);
      if (wave + 8 > r) {
        update(y[1], r);
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
    store_t();
    store(y[0], wave);
    store(y[1], wave + 8);
  } else {
#pragma unroll 1
    for (int base = 0; base < nr; base += 8) {
      if (base > 0) {  // rows 8 .. 15 through the first eight reflectors
        const int r0 = k0 + 8;
        const int team = tid >> 8;
        lq_apply_panel<4>(T, k0, r0, T.M, ld, r0, team ? r0 : k1, 0, S.P[team], S.Q[team], S.T[team]);
      }
      load(y[0], wave + base);
      __syncthreads();
      if (wave == 0) reflector(y[0], base);
      __syncthreads();
      const int end = min(nr, base + 8);
#pragma unroll 1
      for (int r = base; r < end; ++r) {
        if (wave + base > r) {
          update(y[0], r);
          if (wave + base == r + 1 && r + 1 < end) reflector(y[0], r + 1);
        } else if (wave + base < r) {
          gram(y[0], wave + base, r);
        }
        if (base > 0) {  // G with the finished row `wave`, from memory
          double2 d = make_double2(0, 0);
#pragma unroll 8
          for (int j = 0; j < NC; ++j) {
            const int c = lane + 64 * j;
            d = cfmac(srow[(r & 1) * NC * 64 + c], gld(M + (size_t)wave * ld + min(c, W - 1)), d);  // w_r is 0 past W
          }
          d = wave_sum2(d);
          if (lane == 0) sG[wave][r] = d;
        }
        if (r > 0 && wave == ((r + 4) & 7)) t_column(r - 1);
        __syncthreads();
      }
      if (wave == 0) t_column(end - 1);
      __syncthreads();
      store_t();
      store(y[0], wave + base);
      __syncthreads();
    }
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
    if (p >= 0) lq_apply_panel<4>(T, k0, k1, T.M, T.ld, k1, team ? k1 : e1, 0, S.P[team], S.Q[team], S.T[team]);
    // one row of a lane or two is the task's own: the two round differently, and a matrix beside wider ones gives
    // what it gives alone
    if (NC <= 16 || T.cols - k1 <= LQ_TWO_ROWS_COLS) lq_factor_regs<(NC <= 16 ? NC : 16), 2>(T, p + 1, S, srow);
    else lq_factor_regs<NC, 1>(T, p + 1, S, srow);
    return;
  }
  const int r0 = k1 + LQB + 2 * LQR * ((int)blockIdx.y - 1);
  if (r0 >= T.rows) return;
  const int rt = min(r0 + LQR * team, T.rows);
  lq_apply_panel<4>(T, k0, k1, T.M, T.ld, rt, min(rt + LQR, T.rows), 0, S.P[team], S.Q[team], S.T[team]);
}

// Rows beyond panel p + 1 with the block reflector of panel p, 16 rows per workgroup
__global__ __launch_bounds__(256, 4) void k_lq_rest(const LqTask* tasks, int p) {
  __shared__ double2 sP[4][LQR][LQB + 1];
  __shared__ double2 sQ[LQB][LQB + 1];
  __shared__ double2 sT[LQR][LQB + 1];
  const LqTask& T = tasks[blockIdx.x];
  const int k0 = p * LQB;
  const int r0 = k0 + 2 * LQB + LQR * (int)blockIdx.y;
  if (r0 >= T.rows) return;
  lq_apply_panel<2>(T, k0, k0 + LQB, T.M, T.ld, r0, min(r0 + LQR, T.rows), 0, sP, sQ, sT);
}

hipError_t launch_lq_lookahead(const LqTask* d_tasks, int ntasks, int max_rows, int max_cols, hipStream_t sa,
                               hipStream_t sb, hipEvent_t ea, hipEvent_t eb) {
  if (ntasks <= 0 || max_rows <= 0) return hipSuccess;
  if (max_cols > LQ_REG_MAX_COLS) return hipErrorNotSupported;
  const int panels = (max_rows + LQB - 1) / LQB;
  // columns per lane of the panel's registers, by the widest task; a task's results are the same for every NC
  // that holds it
  auto step = [&](int p, int blocks) {
    const int w = max_cols - (p + 1) * LQB;
    const dim3 g(ntasks, blocks), b(512);
    if (w <= 128) hipLaunchKernelGGL(k_lq_step<2>, g, b, 0, sa, d_tasks, p);
    else if (w <= 256) hipLaunchKernelGGL(k_lq_step<4>, g, b, 0, sa, d_tasks, p);
    else if (w <= 512) hipLaunchKernelGGL(k_lq_step<8>, g, b, 0, sa, d_tasks, p);
    else if (w <= LQ_TWO_ROWS_COLS) hipLaunchKernelGGL(k_lq_step<16>, g, b, 0, sa, d_tasks, p);
    else if (w <= 1536) hipLaunchKernelGGL(k_lq_step<24>, g, b, 0, sa, d_tasks, p);
    else hipLaunchKernelGGL(k_lq_step<32>, g, b, 0, sa, d_tasks, p);
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
