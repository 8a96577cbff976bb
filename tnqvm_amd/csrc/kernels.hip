// kernels.hip -- gfx950 kernels of libhipmps.
//
// Kernel map (reference function each one replaces, tnqvm/visitors/exatn-mps/):
//   k_apply_1q ......... 1-qubit gate into a site      ExaTnMpsVisitor.cpp:1231-1273
//   k_theta_mfma ....... merge + 2-qubit gate          ExaTnMpsVisitor.cpp:1401-1541
//                        (+ stabilizeTensorBody, :141-161)
//   k_jacobi_prep,
//   k_jacobi_round ..... full SVD (one-sided block Jacobi, FP64)  :1555-1627
//   k_rownorm, k_select  partial norms, cutoff, max-bond clamp    :2366-2536
//   k_gather, k_gemm ... sqrt(S) split into the two new sites     :1623
//   k_gemm, k_chain,
//   k_trace_prod ....... environments / amplitudes / slices       :593-643, :2588-2675
#include "kernels.h"
#include "device_util.h"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>

namespace hipmps {

// ------------------------------------------------------------------ 1-qubit gate
// new[l][b][r] = sum_i M[b][i] A[l][i][r]  (pattern Result(a,b,c)=Q(a,i,c)*G(i,b),
// ExaTnMpsVisitor.cpp:1246, with G(i,b) = M[b][i] from the row-major flattening)
template <typename T>
__global__ __launch_bounds__(256) void k_apply_1q(T* A, int cl, int cr, double2 m0, double2 m1,
                                                  double2 m2, double2 m3) {
  size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  size_t total = (size_t)cl * cr;
  if (idx >= total) return;
  size_t l = idx / cr, r = idx % cr;
  size_t i0 = (l * 2 + 0) * cr + r, i1 = (l * 2 + 1) * cr + r;
  double2 a0 = ld(A, i0), a1 = ld(A, i1);
  st(A, i0, cfma(m1, a1, cmul(m0, a0)));
  st(A, i1, cfma(m3, a1, cmul(m2, a0)));
}

hipError_t launch_apply_1q(void* site, int fp32, int cl, int cr, const double2 m[4], hipStream_t s) {
  size_t total = (size_t)cl * cr;
  dim3 grid((unsigned)((total + 255) / 256));
  if (fp32)
    hipLaunchKernelGGL(k_apply_1q<float2>, grid, dim3(256), 0, s, (float2*)site, cl, cr, m[0], m[1], m[2], m[3]);
  else
    hipLaunchKernelGGL(k_apply_1q<double2>, grid, dim3(256), 0, s, (double2*)site, cl, cr, m[0], m[1], m[2], m[3]);
  return hipGetLastError();
}

// ------------------------------------------------------------------ theta = G (Ai Aj)
// Workgroup tile: 16 values of l (32 rows (l,a)) x 32 values of r (64 columns (b,r)).
constexpr int TH_L = 16, TH_R = 32;

// ------------------------------------------------------------------ theta on MFMA
// theta'[(l,a)][(b,r)] = sum_{a'b'} G[(a,b),(a',b')] sum_m Ai[l][a'][m] Aj[m][b'][r] as a complex
// GEMM on the matrix cores: complex64 sites use v_mfma_f32_16x16x4f32 (FP32 products and FP32
// accumulation), complex128 sites v_mfma_f64_16x16x4f64; each complex product is four real
// MFMAs.  Workgroup tile: 16 l x 32 r; wave w: 8 l x 16 r, i.e. one 16-row MFMA
// tile (rows = 8 l x 2 a) against two 16-column tiles (b = 0, 1).  The MFMA rows are ordered
// so that the a = 0 and a = 1 rows of one l land in the same lane, as do b = 0 and b = 1, so
// the 4x4 gate mixes the (a, b) block of each (l, r) in registers:
//   f32 D[i][j]: lane j + 16 (i / 4), register i % 4  -> row i = 4g + v: l = 2g + (v & 1), a = v >> 1
//   f64 D[i][j]: lane j + 16 (i % 4), register i / 4  -> row i = 4v + g: l = 2g + (v & 1), a = v >> 1
template <typename T>
struct MfmaTraits;
template <>
struct MfmaTraits<float2> {
  typedef float scalar;
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mma(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // (l offset, a) of MFMA row i
  static __device__ __forceinline__ int row_l(int i) { return 2 * (i >> 2) + (i & 1); }
  static __device__ __forceinline__ int row_a(int i) { return (i >> 1) & 1; }
  // (lane group g, register v) holding D[i][.]
  static __device__ __forceinline__ int out_row(int g, int v) { return 4 * g + v; }
};
template <>
struct MfmaTraits<double2> {
  typedef double scalar;
  typedef double acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mma(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row_l(int i) { return 2 * (i & 3) + ((i >> 2) & 1); }
  static __device__ __forceinline__ int row_a(int i) { return i >> 3; }
  static __device__ __forceinline__ int out_row(int g, int v) { return 4 * v + g; }
};

template <typename T>
__global__ __launch_bounds__(256) void k_theta_mfma(const ThetaTask* tasks, int ntasks) {
  typedef MfmaTraits<T> M;
  typedef typename M::scalar S;
  typedef typename M::acc A4;
  constexpr int KC = 16;  // contraction chunk staged in LDS
  __shared__ T sAi[TH_L][2][KC + 1];
  __shared__ T sAj[KC][2][TH_R + 1];
  const int t = find_task(tasks, ntasks, (int)blockIdx.x, [](const ThetaTask& x) { return x.tile_begin; });
  const ThetaTask& task = tasks[t];
  const int tile = blockIdx.x - task.tile_begin;
  if (tile >= task.tiles_l * task.tiles_r) return;
  const int l0 = (tile / task.tiles_r) * TH_L, r0 = (tile % task.tiles_r) * TH_R;
  const int cl = task.cl, cm = task.cm, cr = task.cr;
  const T* Ai = (const T*)task.Ai;
  const T* Aj = (const T*)task.Aj;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, k4 = lane >> 4;
  const int wl = (wave >> 1) * 8, wr = (wave & 1) * 16;  // this wave's l and r offsets in the tile
  const int my_l = wl + M::row_l(l16), my_a = M::row_a(l16);  // A operand row of this lane
  A4 re0 = {0, 0, 0, 0}, im0 = {0, 0, 0, 0}, re1 = {0, 0, 0, 0}, im1 = {0, 0, 0, 0};
  for (int m0 = 0; m0 < cm; m0 += KC) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int e = tid + 256 * q;  // 512 = 16 l x 2 a x 16 k
      const int l = e >> 5, a = (e >> 4) & 1, k = e & 15;
      T v = T{0, 0};
      if (l0 + l < cl && m0 + k < cm) v = Ai[((size_t)(l0 + l) * 2 + a) * cm + m0 + k];
      sAi[l][a][k] = v;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = tid + 256 * q;  // 1024 = 16 k x 2 b x 32 r
      const int k = e >> 6, b = (e >> 5) & 1, rr = e & 31;
      T v = T{0, 0};
      if (m0 + k < cm && r0 + rr < cr) v = Aj[((size_t)(m0 + k) * 2 + b) * cr + r0 + rr];
      sAj[k][b][rr] = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KC / 4; ++kk) {
      const T x = sAi[my_l][my_a][kk * 4 + k4];            // A[i][k], i = l16
      const T y0 = sAj[kk * 4 + k4][0][wr + l16];          // B[k][j], b = 0
      const T y1 = sAj[kk * 4 + k4][1][wr + l16];          // b = 1
      const S xr = x.x, xi = x.y, nxi = -x.y;
      re0 = M::mma(xr, y0.x, re0);
      re0 = M::mma(nxi, y0.y, re0);
      im0 = M::mma(xr, y0.y, im0);
      im0 = M::mma(xi, y0.x, im0);
      re1 = M::mma(xr, y1.x, re1);
      re1 = M::mma(nxi, y1.y, re1);
      im1 = M::mma(xr, y1.y, im1);
      im1 = M::mma(xi, y1.x, im1);
    }
    __syncthreads();
  }
  // registers v and v + 2 of this lane hold a = 0, 1 of one l; re0/im0 b = 0, re1/im1 b = 1
  const int r = r0 + wr + l16;
  const size_t ldt = (size_t)2 * cr;
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    const int l = l0 + wl + M::row_l(M::out_row(k4, v));
    if (l >= cl || r >= cr) continue;
    double2 x[4];  // (a', b') = (0,0), (0,1), (1,0), (1,1)
    x[0] = make_double2(re0[v], im0[v]);
    x[1] = make_double2(re1[v], im1[v]);
    x[2] = make_double2(re0[v + 2], im0[v + 2]);
    x[3] = make_double2(re1[v + 2], im1[v + 2]);
#pragma unroll
    for (int ab = 0; ab < 4; ++ab) {
      double2 o = make_double2(0, 0);
#pragma unroll
      for (int k = 0; k < 4; ++k) o = cfma(task.G[ab * 4 + k], x[k], o);
      // stabilizeTensorBody: |x| < 1e-100 -> 0 (ExaTnMpsVisitor.cpp:141-161)
      if (cabs2(o) < 1e-200) o = make_double2(0, 0);
      const int a = ab >> 1, b = ab & 1;
      task.theta[((size_t)l * 2 + a) * ldt + (size_t)b * cr + r] = o;
    }
  }
}

hipError_t launch_theta(const ThetaTask* d_tasks, int ntasks, int total_tiles, int fp32, hipStream_t s) {
  if (total_tiles <= 0) return hipSuccess;
  if (fp32)
    hipLaunchKernelGGL(k_theta_mfma<float2>, dim3(total_tiles), dim3(256), 0, s, d_tasks, ntasks);
  else
    hipLaunchKernelGGL(k_theta_mfma<double2>, dim3(total_tiles), dim3(256), 0, s, d_tasks, ntasks);
  return hipGetLastError();
}

// ------------------------------------------------------------------ Jacobi: prepare Y
// Y = X with X = theta (m <= n) or theta^H (m > n); rows r..r_pad-1 are zero.
__global__ __launch_bounds__(256) void k_jacobi_prep(const SplitTask* sp, const JacTask* jt) {
  __shared__ double2 tile[32][33];
  const SplitTask& S = sp[blockIdx.y];
  const JacTask& J = jt[blockIdx.y];
  const int tiles_c = (J.c_tot + 31) / 32;
  const int tiles_r = J.r_pad / 32;
  const int bt = blockIdx.x;
  if (bt >= tiles_c * tiles_r) return;
  const int i0 = (bt / tiles_c) * 32, c0 = (bt % tiles_c) * 32;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;  // 32 x 8
  if (!S.transposed) {
    for (int y = ty; y < 32; y += 8) {
      int i = i0 + y, c = c0 + tx;
      if (c < J.c_tot) {
        double2 v = make_double2(0, 0);
        if (i < J.r && c < J.c) v = S.theta[(size_t)i * S.n + c];
        J.Y[(size_t)i * J.ldy + c] = v;
      }
    }
  } else {
    // Y[i][c] = conj(theta[c][i]); read theta rows coalesced along i
    for (int y = ty; y < 32; y += 8) {
      int c = c0 + y, i = i0 + tx;
      double2 v = make_double2(0, 0);
      if (c < J.c && i < J.r) v = cconj(S.theta[(size_t)c * S.n + i]);
      tile[y][tx] = v;
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
      int i = i0 + y, c = c0 + tx;
      if (c < J.c_tot) J.Y[(size_t)i * J.ldy + c] = tile[tx][y];
    }
  }
}

hipError_t launch_jacobi_prep(const SplitTask* d_split, const JacTask* d_jac, int ntasks, int max_rows,
                              int max_cols, hipStream_t s) {  // max_cols: largest c + r
  int tr = (max_rows + 31) / 32, tc = (max_cols + 31) / 32;
  hipLaunchKernelGGL(k_jacobi_prep, dim3(tr * tc, ntasks), dim3(256), 0, s, d_split, d_jac);
  return hipGetLastError();
}

// ------------------------------------------------------------------ Jacobi: one round
// One workgroup per block pair (the rows of two JB-row blocks).  Round-robin ("circle")
// ordering: slot 0 holds block 0, slot s>0 holds block 1 + (s-1+round) mod (nb-1); pair
// i couples slots i and nb-1-i, so every unordered block pair meets once per sweep.  The
// same ordering, with 2*JB single rows in place of blocks, drives the inner sweep.
//
// For the 2*JB rows:  Gram  Gam[i][j] = sum_c conj(Y[i][c]) Y[j][c]
//                     Gam ~ W Lambda W^H  by one cyclic two-sided Jacobi sweep (FP64)
//                     Y' = W^T Y          (rows become mutually orthogonal)
// A value moved one lane along its row of 16 lanes: from the next lane (lane 15 keeps `edge`) or from
// the previous one (lane 0 keeps `edge`).
template <int CTRL>
__device__ __forceinline__ double dpp_move(double edge, double v) {
  const long long e = __double_as_longlong(edge), x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)e, (int)x, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(e >> 32), (int)(x >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double2 flip_im(double2 v, int sign) {  // sign: 0, or the sign bit
  const long long y = __double_as_longlong(v.y) ^ ((long long)sign << 32);
  return make_double2(v.x, __longlong_as_double(y));
}
__device__ __forceinline__ double2 from_next(double2 edge, double2 v) {
  return make_double2(dpp_move<0x101>(edge.x, v.x), dpp_move<0x101>(edge.y, v.y));  // row_shl:1
}
__device__ __forceinline__ double2 from_next_cyclic(double2 v) {  // lane 15 takes lane 0's
  return make_double2(dpp_move<0x12f>(v.x, v.x), dpp_move<0x12f>(v.y, v.y));  // row_ror:15
}
__device__ __forceinline__ double2 from_prev(double2 edge, double2 v) {
  return make_double2(dpp_move<0x111>(edge.x, v.x), dpp_move<0x111>(edge.y, v.y));  // row_shr:1
}

// The two orderings of the inner sweep.  G is held by slot: at every step, pair k is slots k and
// JP-1-k.
//   full (CROSS = false): the circle ordering, 31 steps, every pair of the 32 rows once.  From one
//     step to the next a row moves from slot x to x-1, slot 1 to JP-1, slot 0 stays.
//   cross (CROSS = true): 16 steps, every row of the first block with every row of the second.  The
//     first block's rows keep their slots k, the second's move from pair k to pair k-1 (mod 16).
// A sweep over all block pairs that uses the full ordering everywhere rotates the pairs within a
// block nb-1 times; the cross ordering in most rounds leaves those out (jacobi_full_round).
template <bool CROSS>
constexpr int inner_next_slot(int x) {
  return CROSS ? (x < JB ? x : (x == JP - 1 ? JB : x + 1)) : (x == 0 ? 0 : (x == 1 ? JP - 1 : x - 1));
}

// The 120 blocks (k, l), k < l, of rotation pairs that the threads 0..119 update, packed k << 4 | l.
// The next step's pair j is formed from one entry of one block -- full: (0, 1) for pair 0, (j - 1,
// j + 1), (14, 15) for pair 15; cross: (j, j + 1), (0, 15) for pair 15 -- and these 16 blocks come
// first (wave 0, so that wave 1 skips the rotation), the others in row order.
struct InnerBlockMap {
  unsigned char v[128];
};
template <bool CROSS>
constexpr int inner_owner_block(int j) {
  const int k = CROSS ? (j < 15 ? j : 0) : (j == 0 ? 0 : j - 1);
  const int l = CROSS ? (j < 15 ? j + 1 : 15) : (j == 0 ? 1 : (j == 15 ? 15 : j + 1));
  return k << 4 | l;
}
template <bool CROSS>
constexpr InnerBlockMap make_inner_block_map() {
  InnerBlockMap m{};
  int n = 0;
  for (; n < 16; ++n) m.v[n] = (unsigned char)inner_owner_block<CROSS>(n);
  for (int k = 0; k < 16; ++k)
    for (int l = k + 1; l < 16; ++l) {
      bool owner = false;
      for (int j = 0; j < 16; ++j) owner = owner || inner_owner_block<CROSS>(j) == (k << 4 | l);
      if (!owner) m.v[n++] = (unsigned char)(k << 4 | l);
    }
  for (; n < 128; ++n) m.v[n] = 1;  // threads 120..127 (see inner_sweep)
  return m;
}
__constant__ InnerBlockMap c_inner_full = make_inner_block_map<false>();
__constant__ InnerBlockMap c_inner_cross = make_inner_block_map<true>();

// Rounds of a sweep whose inner sweep is the full ordering: every 2nd for SVDs of up to 4 blocks,
// every 4th up to 14, every 8th above.  In an emulation on preconditioned 64 x 64 to 256 x 256
// matrices (random, and theta' of decaying spectra; tolerances 1e-13 and 1e-8) these periods keep
// the sweep count within one of the full ordering's with 16 to 41% fewer inner steps; once a sweep
// takes one more sweep, and twice as often gains nothing.
__device__ __forceinline__ bool jacobi_full_round(int round, int nb) {
  return round % (nb <= 4 ? 2 : (nb < 16 ? 4 : 8)) == 0;
}

struct InnerShared {
  double2 G[2][JP][JP + 1];
  double2 tau[2][JB];  // rotations of the current / next step
  double c[2][JB];
  double d[2][JP];     // diagonal by slot, rotated
  int rot[8];          // per wave: an entry of the Gram is above the tolerance
};

// One cyclic two-sided Jacobi sweep on the Hermitian S.G[0]; leaves W (its rotations) in S.G[0].
// Waves 0 and 1 hold one 2x2 block each of rotation pairs k < l (the other half is its conjugate,
// a rotated diagonal block is diag(d) with a zero off-diagonal entry), waves 2 and 3 hold W.
// Further waves only keep the barriers.
template <bool CROSS>
__device__ __forceinline__ void inner_sweep(InnerShared& S, double itol, double floor2) {
  const int tid = threadIdx.x, wave = tid >> 6, l16 = tid & 15;
  if (tid < JB) {
    double alpha = S.G[0][tid][tid].x, beta = S.G[0][JP - 1 - tid][JP - 1 - tid].x, c;
    double2 tau;
    jacobi_rotation(alpha, beta, S.G[0][tid][JP - 1 - tid], itol, floor2, c, tau);
    S.c[0][tid] = c;
    S.tau[0][tid] = tau;
    S.d[0][tid] = alpha;
    S.d[0][JP - 1 - tid] = beta;
  }
  __syncthreads();
  constexpr int STEPS = CROSS ? JB : JP - 1;
  constexpr int LDG = JP + 1;
  if (wave < 2) {
    const int blk = CROSS ? c_inner_cross.v[tid] : c_inner_full.v[tid];
    const int bk = blk >> 4, bl = blk & 15;
    // where this thread's four entries go: the next step's slots, in the half with the smaller pair
    // first, conjugated (sign bit) where that swaps row and column.  The entry that becomes a
    // pair's own off-diagonal goes to the unused column JP.  Threads 120..127 write the zeros that
    // the rotated off-diagonal entries of two pairs each become.
    const bool zeros = tid >= 120;
    int dst[4], flip[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int x = (e & 2) ? JP - 1 - bk : bk, y = (e & 1) ? JP - 1 - bl : bl;
      if (zeros) {
        x = 2 * (tid - 120) + (e & 1);
        y = JP - 1 - x;
      }
      const int dx = inner_next_slot<CROSS>(x), dy = inner_next_slot<CROSS>(y);
      const int px = dx < JB ? dx : JP - 1 - dx, py = dy < JB ? dy : JP - 1 - dy;
      dst[e] = px == py ? dx * LDG + JP : (px < py ? dx * LDG + dy : dy * LDG + dx);
      flip[e] = px > py ? (int)0x80000000 : 0;
    }
    // owners (threads 0..15): slots of the next pair's members, which entry of the block couples
    // them and whether it is stored conjugated
    const bool owner = tid < JB;
    int xa, xb;
    bool conj_g, e10 = false, e11 = false;
    if (CROSS) {
      xa = tid & 15;
      xb = JP - 1 - ((tid + 1) & 15);
      e10 = conj_g = tid == 15;
    } else {
      xa = tid == 0 ? 0 : (tid == 15 ? JB : (tid + 1) & 15);
      xb = tid == 0 ? 1 : JP - 1 - ((tid - 1) & 15);
      conj_g = tid != 0;
      e11 = tid == 15;
      e10 = conj_g && !e11;
    }
    double2* gA = &S.G[0][0][0];
    double2* gB = &S.G[1][0][0];
    const int pk = bk * LDG, qk = (JP - 1 - bk) * LDG, pl = bl, ql = JP - 1 - bl;
#pragma unroll 1
    for (int st = 0; st < STEPS; ++st) {
      const int buf = st & 1;
      const double2 tl = S.tau[buf][bl];
      const double2 b00 = gA[pk + pl], b01 = gA[pk + ql], b10 = gA[qk + pl], b11 = gA[qk + ql];
      const double2 tk = S.tau[buf][bk];
      const double ck = S.c[buf][bk], cl = S.c[buf][bl];
      double alpha = 0.0, beta = 0.0;
      if (wave == 0) {
        alpha = S.d[buf][xa];
        beta = S.d[buf][xb];
      }
      const double rho = zeros ? 0.0 : ck * cl;
      // block B' = Jk^H B Jl
      const double2 ntl = make_double2(-tl.x, tl.y);
      const double2 m00 = cfma(b01, ntl, b00), m01 = cfma(b00, tl, b01);
      const double2 m10 = cfma(b11, ntl, b10), m11 = cfma(b10, tl, b11);
      const double2 ntk = make_double2(-tk.x, -tk.y), ctk = cconj(tk);
      const double2 n00 = cscale(cfma(ntk, m10, m00), rho), n01 = cscale(cfma(ntk, m11, m01), rho);
      const double2 n10 = cscale(cfma(ctk, m00, m10), rho), n11 = cscale(cfma(ctk, m01, m11), rho);
      gB[dst[0]] = flip_im(n00, flip[0]);
      gB[dst[1]] = flip_im(n01, flip[1]);
      gB[dst[2]] = flip_im(n10, flip[2]);
      gB[dst[3]] = flip_im(n11, flip[3]);
      if (wave == 0) {  // the next step's rotations
        double cn;
        double2 tau;
        double2 gam = CROSS ? (e10 ? n10 : n01) : (e10 ? n10 : (e11 ? n11 : n00));
        gam = flip_im(gam, conj_g ? (int)0x80000000 : 0);
        jacobi_rotation(alpha, beta, gam, itol, floor2, cn, tau);
        if (owner) {
          S.tau[buf ^ 1][tid] = tau;
          S.c[buf ^ 1][tid] = cn;
          S.d[buf ^ 1][tid] = alpha;
          S.d[buf ^ 1][JP - 1 - tid] = beta;
        }
      }
      __syncthreads();
      double2* tmp = gA;
      gA = gB;
      gB = tmp;
    }
    __syncthreads();  // W is in place
  } else if (wave >= 4) {
#pragma unroll 1
    for (int st = 0; st <= STEPS; ++st) __syncthreads();
  } else {
    // W rows wr .. wr + 3 at slots l16 (t) and JP-1-l16 (b)
    const int wr = 4 * ((tid - 128) >> 4);
    double2 t[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      t[i] = make_double2(wr + i == l16 ? 1.0 : 0.0, 0.0);
      b[i] = make_double2(wr + i == JP - 1 - l16 ? 1.0 : 0.0, 0.0);
    }
#pragma unroll 1
    for (int st = 0; st < STEPS; ++st) {
      const double c = S.c[st & 1][l16];
      const double2 tau = S.tau[st & 1][l16], ntau = make_double2(-tau.x, tau.y);
      // W' = W J, then to the next step's slots; full: the top slot of pair k takes pair k + 1's top
      // (pair 15: its own bottom, pair 0 keeps its top), the bottom slot pair k - 1's bottom (pair
      // 0: pair 1's top)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double2 u = cscale(cfma(b[i], ntau, t[i]), c), d = cscale(cfma(t[i], tau, b[i]), c);
        if (CROSS) {
          t[i] = u;
          b[i] = from_next_cyclic(d);
        } else {
          const double2 x = from_next(d, u);
          b[i] = from_prev(x, d);
          t[i] = l16 == 0 ? u : x;
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      S.G[0][wr + i][l16] = t[i];
      S.G[0][wr + i][JP - 1 - l16] = b[i];
    }
    __syncthreads();
  }
}

// Design notes (gfx950):
//  * Gram and apply stream their MFMA operands straight from memory into registers; no
//    LDS staging and no barriers in either loop.  The Gram is Hermitian, so only tiles
//    (0,0), (0,1), (1,1) are formed; each wave covers every fourth 4-column unit and the
//    four partial Grams are summed once in LDS.
//  * In the apply each wave owns whole 32-row x 16-column tiles, so the in-place update
//    never overwrites a column another wave still reads.
//  * Inner sweep: a thread owns the 2x2 block of rotation pairs k < l and updates it two-sided
//    in one pass (B' = Jk^H B Jl, G double-buffered in LDS); when an entry of it couples the
//    members of a next step's pair, it also forms that pair's rotation from values it already
//    holds and the rotated diagonal entries, which travel with the rotations.  One barrier per
//    step; every LDS read of a step is issued before any arithmetic.  Each step writes its
//    rotated blocks where the next step reads them, so every G address is fixed per thread; after
//    the last step the slots are back in row order.
//  * W stays in registers of two waves of its own, each thread four rows at the two slots of one
//    pair: the slots' move to the next step is a shift by one lane within a row of 16 lanes.
//  A step is bound by its serial chain (LDS read, block update, rotation, LDS write, barrier) and
//  by LDS bandwidth: the whole G and W in LDS (20 16-byte accesses a thread and step, all four
//  waves) took 1590 clocks a step, a half of G on two waves and W in registers 1200.
//  Measured, 768 workgroups on 32 rows x 512 columns (three per CU): 156 us a launch before
//  (inner sweep 93k clocks), 143 us with the full ordering, 126 us with the cross one, which is
//  4.8 TB/s over its three passes, 115 us with the diagonal tiles' products left out of cross rounds.
//  * A launch that leaves CUs idle is bound by one workgroup's chain.  At 32 x 256, four waves: Gram
//    26.7k clocks (1700 a unit of 9 MFMA, 576 of them MFMA: two loads in flight do not cover the
//    latency), inner 20.6k, apply 19.3k.  Eight waves with four loads in flight and cross rounds of
//    three MFMA a unit: 12.5k, 20.6k, 16.6k; 35.2 -> 29.4 -> 26.8 us a launch (512 columns:
//    54.4 -> 43.5 -> 37.3).
// BLK is the block size JB (a template parameter: the kernel's register allocation on
// gfx950 comes out at 128 VGPRs with four waves, four waves per SIMD, in the tiled form).
template <int BLK, bool TILED, int NW>
__global__ __launch_bounds__(64 * NW, NW == 4 && TILED ? 4 : 2) void k_jacobi_round(const JacTask* tasks, int ntasks,
                                                                                    int sweep, int round) {
  static_assert(BLK == 16 && JB == BLK && JP == 2 * BLK && NW % 4 == 0, "rotation-pair blocks of the inner sweep");
  constexpr int NT = 64 * NW;
  __shared__ InnerShared S;
  double2 (*sG)[JP + 1] = S.G[0];
  double2 (*sG2)[JP + 1] = S.G[1];

  const int t = find_task(tasks, ntasks, (int)blockIdx.x, [](const JacTask& x) { return x.pair_begin; });
  const JacTask& T = tasks[t];
  const int pi = blockIdx.x - T.pair_begin;
  const int nb = T.nb;
  if (pi >= nb / 2 || round >= nb - 1) return;
  int* counts = T.counts + sweep % JAC_COUNT_SLOTS * T.cstride;
  if (sweep > T.gram32 && T.counts[(sweep - 1) % JAC_COUNT_SLOTS * T.cstride] == 0) return;  // converged in the sweep before
  const int ba = circle_slot(pi, round, nb), bb = circle_slot(nb - 1 - pi, round, nb);
  const int C = T.c, CT = T.c_tot;
  const size_t ld = T.ldy;
  const double tol = T.tol;
  const double floor2 = T.fro2 ? JAC_FLOOR2 * *T.fro2 : 0.0;
  double2* Y = TILED ? T.Yt : T.Y;
  const int ntc = T.ntc;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, k4 = lane >> 4;
  // element (row, col) of the row-major layout
  auto at = [&](int row, int col) -> size_t { return (size_t)row * ld + col; };
  const int rowa = ba * JB + l16, rowb = bb * JB + l16;  // pair rows l16 and 16 + l16

  // ---- Gram tiles (0,0), (0,1), (1,1), or in a cross round (0,1) and the diagonal ----
  // FP64 MFMA, or in the early sweeps of large SVDs FP32 MFMA at twice the rate: the rotations
  // they give are still applied in FP64 and are unitary, so the rows only lose the accuracy of
  // the rotation angles, which the FP64 sweeps that end every SVD make up for.
  // Eight partial sums whatever NW is, over the 4-column units u = vw, vw + 8, ..., added in the same order:
  // an SVD's result does not depend on what else is in its launch.  Four waves take two of them each, one
  // after the other.
  // Tiled rows (c = c_tot, the last tile's missing columns zero): unit vw + 8 d is a quarter of
  // tile (vw / 4) + 2 d, so both operands advance by two tiles a step; row-major rows are
  // bounded by their columns.
  const int nd = ((TILED ? ntc : (((C + 3) >> 2) + 3) >> 2) + 1) / 2;
  const double2* ga = TILED ? Y + (size_t)ba * ntc * 256 + (l16 >> 2) * 64 + (wave & 3) * 16 + (l16 & 3) * 4 + k4 : Y;
  const double2* gb = TILED ? Y + (size_t)bb * ntc * 256 + (l16 >> 2) * 64 + (wave & 3) * 16 + (l16 & 3) * 4 + k4 : Y;
  constexpr int PD = NW == 4 ? 2 : 4;
  int vw = wave;
  // The loads are not conditional, past the end they repeat the last tile or column: behind a load that may
  // not have been issued, the wait for an older one is a wait for all.
  auto ld_unit = [&](int d, double2& v0, double2& v1) __attribute__((always_inline)) {
    const int col = min(4 * (vw + 8 * d) + k4, C - 1), tile = min((vw >> 2) + 2 * d, ntc - 1);
    v0 = gld(TILED ? ga + (size_t)tile * 256 : Y + at(rowa, col));
    v1 = gld(TILED ? gb + (size_t)tile * 256 : Y + at(rowb, col));
  };
  auto skip_unit = [&](int d) { return TILED && (vw >> 2) + 2 * d >= ntc; };
  auto unit = [&](int d, double2 v) __attribute__((always_inline)) {  // row-major: nothing past the columns
    return TILED || 4 * (vw + 8 * d) + k4 < C ? v : make_double2(0, 0);
  };
  // Complex products on real MFMA with three real products each instead of four:
  //  * diagonal tiles (Hermitian): Re = Ar Ar^T + Ai Ai^T, and Im = X - X^T with X = Ar Ai^T;
  //  * off-diagonal tile conj(A) B^T (Gauss): K1 = (Ar - Ai) Br^T, K2 = Ar (Bi - Br)^T,
  //    K3 = -Ai (Br + Bi)^T;  Re = K1 - K3, Im = K1 + K2.
  // A cross round takes only the rows' norms of the diagonal tiles, three products a unit instead of
  // nine: what its sweep leaves out there is second order (see jacobi_full_round).
  // Each partial sum of the waves goes to LDS as (Re, X) for the diagonal tiles and
  // (Re, Im) for the off-diagonal one; Im of the diagonal tiles is formed after the sum.
  // to_lds(value of the tile entry v of this lane, its row): sums 0, 1 store, then 2, 3 (and so on) add
  const bool full = jacobi_full_round(round, nb);
  double n0 = 0.0, n1 = 0.0;  // cross: squared norms of the rows l16 and 16 + l16 over this lane's columns
  auto to_lds = [&](auto row, auto e00, auto e01, auto e11) __attribute__((always_inline)) {
    if (!full) {
      n0 += __shfl_xor(n0, 16);
      n1 += __shfl_xor(n1, 16);
      n0 += __shfl_xor(n0, 32);
      n1 += __shfl_xor(n1, 32);
    }
    for (int w = vw - wave; w < vw - wave + NW; w += 2) {
      if ((vw & ~1) == w) {
        double2 (*P)[JP + 1] = S.G[vw & 1];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = row(v), j = l16;
          const double2 g01 = e01(v);
          P[i][JB + j] = w ? cadd(g01, P[i][JB + j]) : g01;
          if (full) {
            const double2 g00 = e00(v), g11 = e11(v);
            P[i][j] = w ? cadd(g00, P[i][j]) : g00;
            P[JB + i][JB + j] = w ? cadd(g11, P[JB + i][JB + j]) : g11;
          }
        }
        if (!full && k4 == 0) {
          P[l16][l16].x = w ? P[l16][l16].x + n0 : n0;
          P[JB + l16][JB + l16].x = w ? P[JB + l16][JB + l16].x + n1 : n1;
        }
      }
      __syncthreads();
    }
  };
#pragma unroll 1
  for (; vw < 8; vw += NW) {
    n0 = n1 = 0.0;
    if (sweep >= T.gram32) {
      mfma_d4 k1 = {0, 0, 0, 0}, k2 = {0, 0, 0, 0}, k3 = {0, 0, 0, 0};
      mfma_d4 a00r = {0, 0, 0, 0}, a00x = {0, 0, 0, 0}, a11r = {0, 0, 0, 0}, a11x = {0, 0, 0, 0};
      auto products = [&](auto diag) __attribute__((always_inline)) {
        double2 x0[PD], x1[PD];
#pragma unroll
        for (int d = 0; d < PD; ++d) ld_unit(d, x0[d], x1[d]);
#pragma unroll 1
        for (int e0 = 0; e0 < nd; e0 += PD) {
#pragma unroll
          for (int d = 0; d < PD; ++d) {
            const double2 v0 = unit(e0 + d, x0[d]), v1 = unit(e0 + d, x1[d]);
            ld_unit(e0 + d + PD, x0[d], x1[d]);
            if (skip_unit(e0 + d)) continue;
            if (diag) {
              a00r = mfma64(v0.x, v0.x, a00r);
              a11r = mfma64(v1.x, v1.x, a11r);
              a00x = mfma64(v0.x, v0.y, a00x);
              a11x = mfma64(v1.x, v1.y, a11x);
            } else {
              n0 = fma(v0.x, v0.x, fma(v0.y, v0.y, n0));
              n1 = fma(v1.x, v1.x, fma(v1.y, v1.y, n1));
            }
            k1 = mfma64(v0.x - v0.y, v1.x, k1);
            k2 = mfma64(v0.x, v1.y - v1.x, k2);
            k3 = mfma64(-v0.y, v1.x + v1.y, k3);
            if (diag) {
              a00r = mfma64(v0.y, v0.y, a00r);
              a11r = mfma64(v1.y, v1.y, a11r);
            }
          }
        }
      };
      if (full) products(std::true_type());
      else products(std::false_type());
      // f64 D[i][j]: lane j + 16 (i % 4), register i / 4
      to_lds([&](int v) { return 4 * v + k4; }, [&](int v) { return make_double2(a00r[v], a00x[v]); },
             [&](int v) { return make_double2(k1[v] - k3[v], k1[v] + k2[v]); },
             [&](int v) { return make_double2(a11r[v], a11x[v]); });
    } else {
      typedef float mfma_f4 __attribute__((ext_vector_type(4)));
      mfma_f4 h1 = {0, 0, 0, 0}, h2 = {0, 0, 0, 0}, h3 = {0, 0, 0, 0};
      mfma_f4 b00r = {0, 0, 0, 0}, b00x = {0, 0, 0, 0}, b11r = {0, 0, 0, 0}, b11x = {0, 0, 0, 0};
      auto products = [&](auto diag) __attribute__((always_inline)) {
        double2 x0[PD], x1[PD];
#pragma unroll
        for (int d = 0; d < PD; ++d) ld_unit(d, x0[d], x1[d]);
#pragma unroll 1
        for (int e0 = 0; e0 < nd; e0 += PD) {
#pragma unroll
          for (int d = 0; d < PD; ++d) {
            const double2 v0 = unit(e0 + d, x0[d]), v1 = unit(e0 + d, x1[d]);
            const float p0 = (float)v0.x, q0 = (float)v0.y, p1 = (float)v1.x, q1 = (float)v1.y;
            ld_unit(e0 + d + PD, x0[d], x1[d]);
            if (skip_unit(e0 + d)) continue;
            if (diag) {
              b00r = __builtin_amdgcn_mfma_f32_16x16x4f32(p0, p0, b00r, 0, 0, 0);
              b11r = __builtin_amdgcn_mfma_f32_16x16x4f32(p1, p1, b11r, 0, 0, 0);
              b00x = __builtin_amdgcn_mfma_f32_16x16x4f32(p0, q0, b00x, 0, 0, 0);
              b11x = __builtin_amdgcn_mfma_f32_16x16x4f32(p1, q1, b11x, 0, 0, 0);
            } else {
              n0 = fma(v0.x, v0.x, fma(v0.y, v0.y, n0));
              n1 = fma(v1.x, v1.x, fma(v1.y, v1.y, n1));
            }
            h1 = __builtin_amdgcn_mfma_f32_16x16x4f32(p0 - q0, p1, h1, 0, 0, 0);
            h2 = __builtin_amdgcn_mfma_f32_16x16x4f32(p0, q1 - p1, h2, 0, 0, 0);
            h3 = __builtin_amdgcn_mfma_f32_16x16x4f32(-q0, p1 + q1, h3, 0, 0, 0);
            if (diag) {
              b00r = __builtin_amdgcn_mfma_f32_16x16x4f32(q0, q0, b00r, 0, 0, 0);
              b11r = __builtin_amdgcn_mfma_f32_16x16x4f32(q1, q1, b11r, 0, 0, 0);
            }
          }
        }
      };
      if (full) products(std::true_type());
      else products(std::false_type());
      // f32 D[i][j]: lane j + 16 (i / 4), register i % 4; the waves' partial tiles are summed in FP64
      to_lds([&](int v) { return 4 * k4 + v; }, [&](int v) { return make_double2((double)b00r[v], (double)b00x[v]); },
             [&](int v) {
               return make_double2((double)h1[v] - (double)h3[v], (double)h1[v] + (double)h2[v]);
             },
             [&](int v) { return make_double2((double)b11r[v], (double)b11x[v]); });
    }
  }
  {
    // the two partial sums; Im of the diagonal tiles from X (X[i][j] - X[j][i]), or nothing but the
    // diagonal in a cross round; and the lower off-diagonal tile
    const int i = (tid >> 4) & 15, j = tid & 15;
    double2 g00 = make_double2(0, 0), g11 = make_double2(0, 0);
    if (full) {
      g00 = cadd(sG[i][j], sG2[i][j]);
      g11 = cadd(sG[JB + i][JB + j], sG2[JB + i][JB + j]);
      g00.y -= sG[j][i].y + sG2[j][i].y;
      g11.y -= sG[JB + j][JB + i].y + sG2[JB + j][JB + i].y;
    } else if (i == j) {
      g00.x = sG[i][i].x + sG2[i][i].x;
      g11.x = sG[JB + i][JB + i].x + sG2[JB + i][JB + i].x;
    }
    const double2 g01 = cadd(sG[i][JB + j], sG2[i][JB + j]), g10 = cadd(sG[j][JB + i], sG2[j][JB + i]);
    __syncthreads();
    if (tid < 256) {
      sG[i][j] = g00;
      sG[JB + i][JB + j] = g11;
      sG[i][JB + j] = g01;
      sG[JB + i][j] = cconj(g10);
    }
  }
  __syncthreads();
  // ---- convergence test of this block pair: |G_ij|^2 > tol^2 G_ii G_jj for some i < j ----
  {
    int above = 0;
    const double tol2 = tol * tol;
    for (int e = tid; e < JP * JP; e += NT) {
      const int i = e / JP, j = e % JP;
      const double aii = sG[i][i].x, ajj = sG[j][j].x;
      if (i < j && aii > floor2 && ajj > floor2 && cabs2(sG[i][j]) > tol2 * (aii * ajj)) above = 1;
    }
    above = __any(above);
    if (lane == 0) S.rot[wave] = above;
    __syncthreads();
  }
  if (tid == 0) atomicAdd(counts + 1, 1);
  int any = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) any |= S.rot[w];
  if (!any) return;

  // ---- apply prefetch: this wave's first column tile, all 32 rows ----
  // element (4 kk + k4, column l16 of the tile) of the pair's rows, kk = 0..7
  const int nt = TILED ? ntc : (CT + 15) >> 4;
  double2* ya = TILED ? Y + (size_t)ba * ntc * 256 + (l16 >> 2) * 16 + k4 * 4 + (l16 & 3) : Y + at(ba * JB + k4, l16);
  double2* yb = TILED ? Y + (size_t)bb * ntc * 256 + (l16 >> 2) * 16 + k4 * 4 + (l16 & 3) : Y + at(bb * JB + k4, l16);
  const size_t step_row = TILED ? 64 : 4 * ld, step_tile = TILED ? 256 : 16;
  auto ok_tile = [&](int ctile) { return TILED ? ctile < nt : ctile < nt && ctile * 16 + l16 < CT; };
  auto elem = [&](int kk, int ctile) {
    return (kk < 4 ? ya + kk * step_row : yb + (kk - 4) * step_row) + ctile * step_tile;
  };
  double2 bq[8];
  auto first_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) bq[kk] = ok_tile(wave) ? gld(elem(kk, wave)) : make_double2(0, 0);
  };
  if (NW != 4) first_tile();
  if (full) inner_sweep<false>(S, tol * 0.25, floor2);
  else inner_sweep<true>(S, tol * 0.25, floor2);
  if (NW == 4) first_tile();
  double2 (*sW)[JP + 1] = S.G[0];

  // Several workgroups share a CU where NW = 4 and cover each other's phases: there 128 registers for four
  // of them beat the first tile's loads ahead of the inner sweep, W in registers and both row tiles at a
  // time (three per CU): 1024 workgroups on 32 x 256 95 -> 81 us, on 32 x 512 154 -> 145 us.
  constexpr int RT = NW == 4 ? 1 : 2;  // 16-row tiles at a time
  // ---- apply Y' = W^T Y; wave owns column tiles wave, wave + NW, ... (all 32 rows) ----
#pragma unroll 1
  for (int ctile = wave; ctile < nt; ctile += NW) {
    if (NW == 4) asm volatile("" ::: "memory");  // W from LDS for each tile, not held in registers over the tiles
    // (A + iB)(C + iD) with three real products (Gauss): K1 = (A + B) C, K2 = A (D - C),
    // K3 = B (C + D); Re = K1 - K3, Im = K1 + K2
    const bool ok = ok_tile(ctile), nok = ok_tile(ctile + NW);
#pragma unroll
    for (int h = 0; h < 2; h += RT) {
      mfma_d4 e[RT], f[RT], g[RT];
#pragma unroll
      for (int q = 0; q < RT; ++q) e[q] = f[q] = g[q] = mfma_d4{0, 0, 0, 0};
#pragma unroll
      for (int kk = 0; kk < 8; ++kk) {
        const double2 b = bq[kk];
        double2 w[RT];
#pragma unroll
        for (int q = 0; q < RT; ++q) w[q] = sW[kk * 4 + k4][16 * (h + q) + l16];  // A[i][k] = W[k][i]
        if (h + RT == 2) bq[kk] = nok ? gld(elem(kk, ctile + NW)) : make_double2(0, 0);
        const double dmc = b.y - b.x, cpd = b.x + b.y;
#pragma unroll
        for (int q = 0; q < RT; ++q) {
          e[q] = mfma64(w[q].x + w[q].y, b.x, e[q]);
          f[q] = mfma64(w[q].x, dmc, f[q]);
          g[q] = mfma64(w[q].y, cpd, g[q]);
        }
      }
      if (ok) {
#pragma unroll
        for (int q = 0; q < RT; ++q)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            gst(elem(4 * (h + q) + v, ctile), make_double2(e[q][v] - g[q][v], e[q][v] + f[q][v]));
      }
    }
  }
  if (tid == 0) atomicAdd(counts, 1);
}

// Bound by the read of theta'; one workgroup a task took 2.5 ms at 1536 x 1536 and 220 us a wave of 512 x 512.
// The partial sums are added by a launch of their own: the last workgroup to finish doing so, found by a
// device-scope atomic, made every workgroup write back its XCD's L2 (126 us a wave of an uneven batch).
__global__ __launch_bounds__(256) void k_fro2(const SplitTask* sp, double* part) {
  __shared__ double red[4];
  const SplitTask& S = sp[blockIdx.y];
  const size_t n = (size_t)S.m * S.n;
  const double2* x = S.theta;
  double a = 0.0;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)FRO_BLOCKS * 256) a += cabs2(gld(x + e));
  a = wave_sum(a);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) part[(size_t)blockIdx.y * FRO_BLOCKS + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void k_fro2_sum(const JacTask* jt, const double* part, int ntasks) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= ntasks) return;
  double a = 0.0;
  for (int b = 0; b < FRO_BLOCKS; ++b) a += part[(size_t)t * FRO_BLOCKS + b];
  *jt[t].fro2 = a;
}

hipError_t launch_fro2(const SplitTask* d_split, const JacTask* d_jac, double* part, int ntasks, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fro2, dim3(FRO_BLOCKS, ntasks), dim3(256), 0, s, d_split, part);
  hipLaunchKernelGGL(k_fro2_sum, dim3((ntasks + 255) / 256), dim3(256), 0, s, d_jac, part, ntasks);
  return hipGetLastError();
}

// Launches of at most one workgroup per CU take eight waves each: 256 workgroups on 32 x 512 took 71 us
// with four waves and 56 with eight; from two per CU on, the second one's waves do the same.
constexpr int JAC_WIDE_PAIRS = 256;
hipError_t launch_jacobi_round(const JacTask* d_tasks, int ntasks, int total_pairs, int sweep, int round,
                               hipStream_t s, bool tiled) {
  if (total_pairs <= 0) return hipSuccess;
  const dim3 grid(total_pairs);
  if (total_pairs <= JAC_WIDE_PAIRS) {
    if (tiled) hipLaunchKernelGGL((k_jacobi_round<JB, true, 8>), grid, dim3(512), 0, s, d_tasks, ntasks, sweep, round);
    else hipLaunchKernelGGL((k_jacobi_round<JB, false, 8>), grid, dim3(512), 0, s, d_tasks, ntasks, sweep, round);
  } else {
    if (tiled) hipLaunchKernelGGL((k_jacobi_round<JB, true, 4>), grid, dim3(256), 0, s, d_tasks, ntasks, sweep, round);
    else hipLaunchKernelGGL((k_jacobi_round<JB, false, 4>), grid, dim3(256), 0, s, d_tasks, ntasks, sweep, round);
  }
  return hipGetLastError();
}

// One 16 x 16 tile per workgroup (blockIdx.x = 16-row block * max_ntc + tile column, blockIdx.y =
// task); thread (i, j) = (tid / 16, tid % 16) moves element (16 b + i, 16 t + j).
template <bool TO>
__global__ __launch_bounds__(256) void k_tiles(const JacTask* tasks, int max_ntc) {
  const JacTask& T = tasks[blockIdx.y];
  const int b = blockIdx.x / max_ntc, t = blockIdx.x % max_ntc;
  if (b >= T.r_pad / 16 || t >= T.ntc) return;
  const int row = 16 * b + (threadIdx.x >> 4), col = 16 * t + (threadIdx.x & 15);
  const size_t o = jac_tile_offset(row, col, T.ntc);
  if (TO) T.Yt[o] = col < T.c_tot ? T.Y[(size_t)row * T.ldy + col] : make_double2(0, 0);
  else if (col < T.c_tot) T.Y[(size_t)row * T.ldy + col] = T.Yt[o];
}

hipError_t launch_to_tiles(const JacTask* d_tasks, int ntasks, int max_blocks, int max_ntc, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_tiles<true>, dim3(max_blocks * max_ntc, ntasks), dim3(256), 0, s, d_tasks, max_ntc);
  return hipGetLastError();
}

hipError_t launch_from_tiles(const JacTask* d_tasks, int ntasks, int max_blocks, int max_ntc, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_tiles<false>, dim3(max_blocks * max_ntc, ntasks), dim3(256), 0, s, d_tasks, max_ntc);
  return hipGetLastError();
}

// ------------------------------------------------------------------ row norms
__global__ __launch_bounds__(256) void k_rownorm(const SplitTask* sp) {
  const SplitTask& S = sp[blockIdx.y];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int i = blockIdx.x * 4 + wave;
  if (i >= S.r) return;
  double a = 0.0;
  const double2* row = S.Y + (size_t)i * S.ldy;
  for (int c = lane; c < S.c; c += 64) a += cabs2(row[c]);
  for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off, 64);
  if (lane == 0) S.rownorm[i] = sqrt(a);
}

hipError_t launch_rownorm(const SplitTask* d_split, int ntasks, int max_r, hipStream_t s) {
  hipLaunchKernelGGL(k_rownorm, dim3((max_r + 3) / 4, ntasks), dim3(256), 0, s, d_split);
  return hipGetLastError();
}

// ------------------------------------------------------------------ sort + truncation rule
// Singular values sorted descending (bitonic in LDS, ties by row index).  Truncation
// follows truncateSvdTensors (ExaTnMpsVisitor.cpp:2424-2445): with the sqrt(S) split
// both partial norms of bond index k equal sigma_k (squared definition) or
// sqrt(sigma_k) (2-norm definition); K = i+1 for the first i whose norm is below the
// cutoff (the sub-threshold index itself is kept), else K0; then K = min(K, max_bond).
constexpr int SEL_MAX = 4096;
__global__ __launch_bounds__(256) void k_select(const SplitTask* sp) {
  __shared__ double key[SEL_MAX];
  __shared__ int idx[SEL_MAX];
  __shared__ double red[256];
  __shared__ int s_first;
  const SplitTask& S = sp[blockIdx.x];
  const int r = S.r;
  int P = 1;
  while (P < r) P <<= 1;
  const int tid = threadIdx.x;
  __shared__ int s_bad;
  if (tid == 0) {
    s_first = r;
    s_bad = 0;
  }
  __syncthreads();
  // a NaN or Inf singular value (non-finite input or overflow) is sorted as 0 and flagged:
  // the keys of real rows then stay >= 0 > -1 (the padding), so the first r indices of the
  // sorted order are always rows of Y
  for (int i = tid; i < P; i += 256) {
    double v = -1.0;
    if (i < r) {
      v = S.rownorm[i];
      if (!(v >= 0.0 && v <= DBL_MAX)) {
        v = 0.0;
        s_bad = 1;
      }
    }
    key[i] = v;
    idx[i] = i;
  }
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < P; i += 256) {
        int ixj = i ^ j;
        if (ixj > i) {
          bool desc = (i & k) == 0;
          double a = key[i], b = key[ixj];
          int ia = idx[i], ib = idx[ixj];
          // "a before b" in descending order with index tie-break
          bool a_first = (a > b) || (a == b && ia < ib);
          bool swap = desc ? !a_first : a_first;
          if (swap) {
            key[i] = b; key[ixj] = a;
            idx[i] = ib; idx[ixj] = ia;
          }
        }
      }
      __syncthreads();
    }
  }
  // first sub-threshold index
  // partial norm of index i: across a sqrt(S) split each factor carries sqrt(sigma_i), so
  // sigma_i (squared norm) or sqrt(sigma_i) (2-norm); a Kraus vector sigma_i v_i carries
  // sigma_i^2 or sigma_i
  for (int i = tid; i < r; i += 256) {
    const double sg = key[i];
    double pn = S.keep_rule ? (S.pn_l2 ? sg : sg * sg) : (S.pn_l2 ? sqrt(sg) : sg);
    if (pn < S.cutoff) atomicMin(&s_first, i);
  }
  __syncthreads();
  int K = s_first < r ? (S.keep_rule ? s_first : s_first + 1) : r;
  if (K > S.max_bond) K = S.max_bond;
  if (K < 1) K = 1;
  // kept / discarded weights (FP64)
  double kept = 0.0, disc = 0.0;
  for (int i = tid; i < r; i += 256) {
    double w = key[i] * key[i];
    if (i < K) kept += w; else disc += w;
  }
  red[tid] = kept;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) { if (tid < w) red[tid] += red[tid + w]; __syncthreads(); }
  kept = red[0];
  __syncthreads();
  red[tid] = disc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) { if (tid < w) red[tid] += red[tid + w]; __syncthreads(); }
  disc = red[0];
  __syncthreads();
  // sum of all singular values: the squared Frobenius norm of either sqrt(S) factor
  // before truncation, for the post-SVD norm validation (ExaTnMpsVisitor.cpp:1634-1661)
  double ssum = 0.0;
  for (int i = tid; i < r; i += 256) ssum += key[i];
  red[tid] = ssum;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) { if (tid < w) red[tid] += red[tid + w]; __syncthreads(); }
  ssum = red[0];
  double f = 1.0;
  if (S.renorm && kept > 0.0) f = sqrt((kept + disc) / kept);
  // scales: left factor U (s)^aL, right factor (s)^aR V^H with s = f * sigma.
  // Row k of Y (sigma_k xh_k^H) gives the factor on the X-row side (times sigma^-1);
  // the other factor is a unit vector recovered by a GEMM and scaled to (s)^a.
  const double aL = S.absorb == 0 ? 0.5 : 0.0, aR = 1.0 - aL;
  const double a_y = S.transposed ? aL : aR;
  const double a_w = S.transposed ? aR : aL;
  for (int k = tid; k < r; k += 256) {
    S.sig[k] = key[k];
    S.perm[k] = idx[k];
    if (k < K) {
      double sg = key[k];
      double gy = 0.0, gw = 0.0, is = 0.0;
      if (sg > 1e-150) {
        double sf = sg * f;
        gy = pow(sf, a_y) / sg;
        gw = pow(sf, a_w);
        is = 1.0 / sg;
      }
      S.scale_y[k] = gy;
      S.scale_w[k] = gw;
      S.inv_sig[k] = is;
    }
  }
  if (tid == 0) {
    *S.K = K;
    S.wstats[0] = disc;
    S.wstats[1] = kept;
    S.wstats[2] = kept + disc;
    S.wstats[3] = f;
    S.wstats[4] = ssum;
    S.wstats[5] = s_bad ? 1.0 : 0.0;
  }
}

hipError_t launch_select(const SplitTask* d_split, int ntasks, hipStream_t s) {
  hipLaunchKernelGGL(k_select, dim3(ntasks), dim3(256), 0, s, d_split);
  return hipGetLastError();
}

// ------------------------------------------------------------------ factor from Y rows
// not transposed (X = theta):  Aj[k][j] = Y[perm k][j] * scale_y[k]         (K x n)
// transposed (X = theta^H):    Ai[i][k] = conj(Y[perm k][i]) * scale_y[k]   (m x K)
template <typename T>
__global__ __launch_bounds__(256) void k_gather(const SplitTask* sp) {
  __shared__ double2 tile[32][33];
  const SplitTask& S = sp[blockIdx.y];
  const int K = *S.K;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;
  const int bt = blockIdx.x;
  if (!S.transposed) {
    const int len = S.n;
    const int tiles_c = (len + 31) / 32;
    const int k0 = (bt / tiles_c) * 32, c0 = (bt % tiles_c) * 32;
    if (k0 >= K) return;
    T* out = (T*)S.Aj;
    for (int y = ty; y < 32; y += 8) {
      int k = k0 + y, c = c0 + tx;
      if (k < K && c < len) {
        double2 v = S.Y[(size_t)S.perm[k] * S.ldy + c];
        st(out, (size_t)k * len + c, cscale(v, S.scale_y[k]));
      }
    }
  } else {
    const int len = S.m;
    const int tiles_i = (len + 31) / 32;
    const int k0 = (bt / tiles_i) * 32, i0 = (bt % tiles_i) * 32;
    if (k0 >= K) return;
    T* out = (T*)S.Ai;
    for (int y = ty; y < 32; y += 8) {
      int k = k0 + y, i = i0 + tx;
      double2 v = make_double2(0, 0);
      if (k < K && i < len) v = cscale(cconj(S.Y[(size_t)S.perm[k] * S.ldy + i]), S.scale_y[k]);
      tile[y][tx] = v;
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
      int i = i0 + y, k = k0 + tx;
      if (i < len && k < K) st(out, (size_t)i * K + k, tile[tx][y]);
    }
  }
}

hipError_t launch_gather(const SplitTask* d_split, int ntasks, int max_k, int max_len, int fp32,
                         hipStream_t s) {
  int tiles = ((max_k + 31) / 32) * ((max_len + 31) / 32);
  if (fp32)
    hipLaunchKernelGGL(k_gather<float2>, dim3(tiles, ntasks), dim3(256), 0, s, d_split);
  else
    hipLaunchKernelGGL(k_gather<double2>, dim3(tiles, ntasks), dim3(256), 0, s, d_split);
  return hipGetLastError();
}

// ------------------------------------------------------------------ normalise recovered factor
// not transposed: columns k of Ai (m x K) scaled to norm scale_w[k];
// transposed:     rows k of Aj (K x n) scaled to norm scale_w[k].
// A vector that came out exactly zero stays zero.
template <typename T>
__global__ __launch_bounds__(256) void k_normalize(const SplitTask* sp) {
  __shared__ double part[8][33];
  __shared__ double fac[32];
  const SplitTask& S = sp[blockIdx.y];
  const int K = *S.K;
  const int k0 = blockIdx.x * 32;
  if (k0 >= K) return;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;
  if (!S.transposed) {
    T* A = (T*)S.Ai;
    const int k = k0 + tx;
    double a = 0.0;
    if (k < K)
      for (int i = ty; i < S.m; i += 8) a += cabs2(ld(A, (size_t)i * K + k));
    part[ty][tx] = a;
    __syncthreads();
    if (ty == 0) {
      double t = 0.0;
      for (int q = 0; q < 8; ++q) t += part[q][tx];
      fac[tx] = (k < K && t > 0.0) ? S.scale_w[k] / sqrt(t) : 0.0;
    }
    __syncthreads();
    if (k < K)
      for (int i = ty; i < S.m; i += 8) {
        size_t o = (size_t)i * K + k;
        st(A, o, cscale(ld(A, o), fac[tx]));
      }
  } else {
    T* A = (T*)S.Aj;
    // 8 rows per block pass, 32 threads per row
    for (int kr = ty; kr < 32; kr += 8) {
      const int k = k0 + kr;
      double a = 0.0;
      if (k < K)
        for (int j = tx; j < S.n; j += 32) a += cabs2(ld(A, (size_t)k * S.n + j));
      for (int off = 16; off > 0; off >>= 1) a += __shfl_xor(a, off, 32);
      const double fk = (k < K && a > 0.0) ? S.scale_w[k] / sqrt(a) : 0.0;
      if (k < K)
        for (int j = tx; j < S.n; j += 32) {
          size_t o = (size_t)k * S.n + j;
          st(A, o, cscale(ld(A, o), fk));
        }
    }
  }
}

hipError_t launch_normalize(const SplitTask* d_split, int ntasks, int max_k, int fp32, hipStream_t s) {
  dim3 grid((max_k + 31) / 32, ntasks);
  if (fp32)
    hipLaunchKernelGGL(k_normalize<float2>, grid, dim3(256), 0, s, d_split);
  else
    hipLaunchKernelGGL(k_normalize<double2>, grid, dim3(256), 0, s, d_split);
  return hipGetLastError();
}

// ------------------------------------------------------------------ generic batched GEMM
// C[i][j] = rowscale_i * colscale_j * sum_k a(i,k) b(k,j)
//   a(i,k): N  A[gA(i)*lda + k]   C conj(A[gA(i)*lda + k])
//           H  conj(A[k*lda + i]) T A[k*lda + i]
//   b(k,j): N  B[k*ldb + j]       T B[gB(j)*ldb + k]   H conj(B[gB(j)*ldb + k])
// optional diagonal operator diag(kd0, kd1) on a(i,k), selected by the physical index
// (k / sign_div) & 1 (Z, projectors, ... inserted on the contracted physical leg).
//
// FP64 MFMA, complex64 operands converted on the way in.  A workgroup owns a 32 x 16 tile of C and its
// four waves split K (unit u of 4 to wave u mod 4, so that the four waves read whole lines of a row of
// A), each streaming its operands from memory into MFMA registers, GEMM_PD units in flight; the four
// partial tiles are summed in LDS in a fixed order.  No LDS staging and no barrier in the loop: the
// operands of these products (environments, sites) are L2-resident, and a chain of them is bound by
// each product's latency.  Split K and the small tile put a 256 x 512 x 256 product, one step of an
// environment sweep at bond 256, on all 256 CUs (32 x 32 tiles through LDS on vector FMA took 38 to 60
// us a step and half of the CUs).
constexpr int GEMM_PD = 4;

template <typename TA, typename TB, typename TC, int OPA, int OPB>
__global__ __launch_bounds__(256) void k_gemm(const GemmTask* tasks, int ntasks, int tile_base) {
  __shared__ double2 sC[4][GEMM_TM][GEMM_TN + 1];
  const int block = tile_base + (int)blockIdx.x;
  const int t = find_task(tasks, ntasks, block, [](const GemmTask& x) { return x.tile_begin; });
  const GemmTask& T = tasks[t];
  const int tile = block - T.tile_begin;
  if (tile >= T.tiles_m * T.tiles_n) return;
  int M = T.M, N = T.N;
  if (T.Mdyn) M = min(M, *T.Mdyn);
  if (T.Ndyn) N = min(N, *T.Ndyn);
  const int i0 = (tile / T.tiles_n) * GEMM_TM, j0 = (tile % T.tiles_n) * GEMM_TN;
  if (i0 >= M || j0 >= N) return;
  const int K = T.K;
  const int ldc = T.ldc > 0 ? T.ldc : N;
  const size_t lda = T.lda, ldb = T.ldb;
  const TA* A = (const TA*)T.A;
  const TB* B = (const TB*)T.B;
  const int sign_div = T.sign_div;
  const double kd0 = T.kd0, kd1 = T.kd1;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, k4 = lane >> 4;
  // rows of A and columns of B of this lane; past the end: a repeat, not stored
  const int ia = min(i0 + l16, M - 1), ib = min(i0 + 16 + l16, M - 1), jb = min(j0 + l16, N - 1);
  const bool a_rows = OPA == 0 || OPA == 1;
  const TA* pa = A + (a_rows ? (size_t)(T.gatherA ? T.gatherA[ia] : ia) * lda : (size_t)ia);
  const TA* pb = A + (a_rows ? (size_t)(T.gatherA ? T.gatherA[ib] : ib) * lda : (size_t)ib);
  const TB* pj = B + (OPB == 0 ? (size_t)jb : (size_t)(T.gatherB ? T.gatherB[jb] : jb) * ldb);
  const size_t sa = a_rows ? 1 : lda, sb = OPB == 0 ? ldb : 1;
  const int nu = (K + 3) >> 2, nd = (nu - wave + 3) >> 2;  // this wave's units wave, wave + 4, ...
  // past the end of K a load repeats the last element: behind a load that may not have been issued, the wait
  // for an older one is a wait for all
  auto load = [&](int d, double2& x0, double2& x1, double2& y) __attribute__((always_inline)) {
    const int kc = min(4 * (wave + 4 * d) + k4, K - 1);
    x0 = ld(pa, (size_t)kc * sa);
    x1 = ld(pb, (size_t)kc * sa);
    y = ld(pj, (size_t)kc * sb);
  };
  mfma_d4 re0 = {0, 0, 0, 0}, im0 = {0, 0, 0, 0}, re1 = {0, 0, 0, 0}, im1 = {0, 0, 0, 0};
  double2 x0[GEMM_PD], x1[GEMM_PD], y[GEMM_PD];
#pragma unroll
  for (int d = 0; d < GEMM_PD; ++d) load(d, x0[d], x1[d], y[d]);
#pragma unroll 1
  for (int d0 = 0; d0 < nd; d0 += GEMM_PD) {
#pragma unroll
    for (int d = 0; d < GEMM_PD; ++d) {
      double2 a0 = x0[d], a1 = x1[d];
      const double2 b = y[d];
      load(d0 + d + GEMM_PD, x0[d], x1[d], y[d]);
      if (d0 + d < nd) {
        const int k0 = 4 * (wave + 4 * (d0 + d));
        if (k0 + 4 > K || sign_div > 0) {
          const int k = k0 + k4;
          double f = k < K ? 1.0 : 0.0;
          if (sign_div > 0) f *= ((k / sign_div) & 1) ? kd1 : kd0;
          a0 = cscale(a0, f);
          a1 = cscale(a1, f);
        }
        // conj(A) (OPA 1, 2): -a.y for a.y; conj(B) (OPB 2): -b.y for b.y
        const double a0y = OPA == 1 || OPA == 2 ? -a0.y : a0.y, a1y = OPA == 1 || OPA == 2 ? -a1.y : a1.y;
        const double by = OPB == 2 ? -b.y : b.y;
        re0 = mfma64(a0.x, b.x, re0);
        im0 = mfma64(a0.x, by, im0);
        re1 = mfma64(a1.x, b.x, re1);
        im1 = mfma64(a1.x, by, im1);
        re0 = mfma64(-a0y, by, re0);
        im0 = mfma64(a0y, b.x, im0);
        re1 = mfma64(-a1y, by, re1);
        im1 = mfma64(a1y, b.x, im1);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    sC[wave][4 * v + k4][l16] = make_double2(re0[v], im0[v]);
    sC[wave][16 + 4 * v + k4][l16] = make_double2(re1[v], im1[v]);
  }
  __syncthreads();
  TC* Cp = (TC*)T.C;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int li = (tid >> 4) + 16 * q, i = i0 + li, j = j0 + l16;
    if (i >= M || j >= N) continue;
    double2 v = cadd(cadd(sC[0][li][l16], sC[1][li][l16]), cadd(sC[2][li][l16], sC[3][li][l16]));
    const double s = (T.rowscale ? T.rowscale[i] : 1.0) * (T.colscale ? T.colscale[j] : 1.0);
    v = cscale(v, s);
    const size_t o = (size_t)i * ldc + j;
    if (T.accumulate) v = cadd(v, ld(Cp, o));
    st(Cp, o, v);
  }
}

template <int OPA, int OPB>
static hipError_t gemm_types(const GemmTask* d, int nt, int tiles, int ta, int tb, int tc, hipStream_t s) {
  constexpr int CHUNK = 1 << 23;  // a dispatch holds at most 2^32 work-items
#define HIPMPS_GEMM_CASE(A_, B_, C_, a, b_, c)                                                   \
  if (ta == a && tb == b_ && tc == c) {                                                          \
    for (int t0 = 0; t0 < tiles; t0 += CHUNK)                                                    \
      hipLaunchKernelGGL((k_gemm<A_, B_, C_, OPA, OPB>), dim3(std::min(CHUNK, tiles - t0)), dim3(256), 0, s, d, nt, t0); \
    return hipGetLastError();                                                                    \
  }
  HIPMPS_GEMM_CASE(double2, double2, double2, 0, 0, 0)
  HIPMPS_GEMM_CASE(double2, double2, float2, 0, 0, 1)
  HIPMPS_GEMM_CASE(float2, double2, double2, 1, 0, 0)
  HIPMPS_GEMM_CASE(double2, float2, double2, 0, 1, 0)
  HIPMPS_GEMM_CASE(float2, float2, double2, 1, 1, 0)
#undef HIPMPS_GEMM_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_gemm(const GemmTask* d_tasks, int ntasks, int total_tiles, int opa, int opb, int ta, int tb,
                       int tc, hipStream_t s) {
  if (total_tiles <= 0) return hipSuccess;
#define HIPMPS_OP_CASE(a, b)                                                                     \
  if (opa == a && opb == b) return gemm_types<a, b>(d_tasks, ntasks, total_tiles, ta, tb, tc, s);
  HIPMPS_OP_CASE(0, 0)
  HIPMPS_OP_CASE(0, 2)
  HIPMPS_OP_CASE(0, 3)
  HIPMPS_OP_CASE(1, 3)
  HIPMPS_OP_CASE(2, 0)
#undef HIPMPS_OP_CASE
  return hipErrorInvalidValue;
}

// ------------------------------------------------------------------ chain step (amplitudes / slices)
// amplitude: vout[r][row] = sum_l vin[l][row] A[l][bits[row][site]][r]
// slice:     vout[r][o]   = sum_l vin[l][o % rows_in] A[l][p][r], p = open ? o / rows_in : bit
//
// FP64 MFMA.  A workgroup owns CHAIN_ROWS rows x 16 columns: it lists its rows with p = 0 and then those
// with p = 1, so that each 16-row tile takes one of the two matrices A[.][p][.] (at most one tile more than
// the rows alone need), and its eight waves split l (unit u of 4 to wave u mod 8).  The vectors lie with the
// rows together; a wave reads them in whole lines, CHAIN_PD units ahead, and picks its tiles' rows through
// LDS of its own, without a barrier.  The partial tiles are summed in LDS in a fixed order.
// Measured, 1000 strings at bond 256, a site: a thread a column with l in series 54 us; tiles read straight
// from rows of vectors, a gather of 64-byte pieces with two units in flight, 24 us; this 21 us, of which
// the MFMA of five tiles for 64 rows take 9.
template <typename T>
__global__ __launch_bounds__(512) void k_chain(const ChainTask* tasks, int ntasks) {
  constexpr int NTILE = CHAIN_ROWS / 16 + 1, PD = 4, NW = 8;
  __shared__ int s_row[16 * NTILE];  // of the tiles' rows: the workgroup's row, or -1
  __shared__ double2 sV[NW][2][4][CHAIN_ROWS];
  __shared__ double2 sC[NW / 2][NTILE][16][17];
  __shared__ int s_tiles[2];
  const int t = find_task(tasks, ntasks, (int)blockIdx.x, [](const ChainTask& x) { return x.block_begin; });
  const ChainTask& C = tasks[t];
  const int b = blockIdx.x - C.block_begin;
  if (b >= C.blocks) return;
  const int cl = C.cl, cr = C.cr, rows_in = C.rows_in;
  // blocks of the same rows 8 apart in launch order: on one XCD, which reads an eighth of the vectors, those
  // it wrote at the site before, and all of A (the other way round: all vectors, an eighth of A)
  const int rblocks = (C.rows_out + CHAIN_ROWS - 1) / CHAIN_ROWS;
  const int r0 = b % rblocks * CHAIN_ROWS, j0 = b / rblocks * 16;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15,
            k4 = lane >> 4;
  const T* A = (const T*)C.A + min(j0 + l16, cr - 1);
  static_assert(CHAIN_ROWS == 64, "a lane a row");
  const int row = min(r0 + lane, C.rows_out - 1);
  const double2* v = C.vin + (C.mode == 0 ? row : row % rows_in);
  const int nu = (cl + 3) >> 2, nd = (nu - wave + NW - 1) / NW;
  double2 x[PD][4], y[PD][2];  // a unit's vectors (a row a lane) and rows of A (p = 0, 1)
  auto load = [&](int d, double2 (&xs)[4], double2 (&ys)[2]) __attribute__((always_inline)) {
    const int l0 = 4 * (wave + NW * d);
#pragma unroll
    for (int i = 0; i < 4; ++i) xs[i] = gld(v + (size_t)min(l0 + i, cl - 1) * rows_in);
    const size_t at = (size_t)min(l0 + k4, cl - 1) * 2 * cr;
    ys[0] = ld(A, at);
    ys[1] = ld(A, at + cr);
  };
#pragma unroll
  for (int d = 0; d < PD; ++d) load(d, x[d], y[d]);
  if (wave == 0) {
    const bool in = r0 + lane < C.rows_out;
    int p = 0;
    if (in) p = C.mode == 0 ? C.bits[(size_t)row * C.n + C.site] : (C.slice_bit < 0 ? row / rows_in : C.slice_bit);
    const unsigned long long m0 = __ballot(in && p == 0), m1 = __ballot(in && p != 0);
    const unsigned long long below = (1ull << lane) - 1;
    const int t0 = (__popcll(m0) + 15) / 16 * 16;
    for (int e = lane; e < 16 * NTILE; e += 64) s_row[e] = -1;
    __builtin_amdgcn_wave_barrier();
    if (in) s_row[p == 0 ? __popcll(m0 & below) : t0 + __popcll(m1 & below)] = lane;
    if (lane == 0) {
      s_tiles[0] = t0 / 16;
      s_tiles[1] = t0 / 16 + (__popcll(m1) + 15) / 16;
    }
  }
  __syncthreads();
  const int n0 = __builtin_amdgcn_readfirstlane(s_tiles[0]);  // tiles with p = 0
  const int nt = __builtin_amdgcn_readfirstlane(s_tiles[1]);  // all tiles
  int pick[NTILE];  // past the end of a tile: any row, not stored
#pragma unroll
  for (int q = 0; q < NTILE; ++q) pick[q] = max(s_row[16 * q + l16], 0);
  mfma_d4 re[NTILE], im[NTILE];
#pragma unroll
  for (int q = 0; q < NTILE; ++q) re[q] = im[q] = mfma_d4{0, 0, 0, 0};
  // the loads are not conditional, past the end they repeat the last row: a wait for one unit's would
  // otherwise be a wait for all that may have followed
#pragma unroll 1
  for (int d0 = 0; d0 < nd; d0 += PD) {
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      const int l0 = 4 * (wave + NW * (d0 + d));
      double2 (*mine)[CHAIN_ROWS] = sV[wave][d & 1];
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[i][lane] = l0 + i < cl ? x[d][i] : make_double2(0, 0);
      const double2 b0 = y[d][0], b1 = y[d][1];
      load(d0 + d + PD, x[d], y[d]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (l0 < cl) {
        double2 a[NTILE];
#pragma unroll
        for (int q = 0; q < NTILE; ++q) a[q] = mine[k4][pick[q]];
#pragma unroll
        for (int q = 0; q < NTILE; ++q)
          if (q < nt) {
            re[q] = mfma64(a[q].x, q < n0 ? b0.x : b1.x, re[q]);
            im[q] = mfma64(a[q].x, q < n0 ? b0.y : b1.y, im[q]);
          }
#pragma unroll
        for (int q = 0; q < NTILE; ++q)
          if (q < nt) {
            re[q] = mfma64(-a[q].y, q < n0 ? b0.y : b1.y, re[q]);
            im[q] = mfma64(a[q].y, q < n0 ? b0.x : b1.x, im[q]);
          }
      }
    }
  }
  // sums of the eight waves: the upper four to the lower, then those four; no barrier after a store
  auto put = [&](int w) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NTILE; ++q)
      if (q < nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sC[w][q][4 * i + k4][l16] = make_double2(re[q][i], im[q][i]);
  };
  if (wave >= 4) put(wave - 4);
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int q = 0; q < NTILE; ++q)
      if (q < nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const double2 x = sC[wave][q][4 * i + k4][l16];
          re[q][i] += x.x;
          im[q][i] += x.y;
        }
    put(wave);  // where this wave read
  }
  __syncthreads();
  for (int e = tid; e < 256 * nt; e += 64 * NW) {
    const int q = e >> 8, j = (e >> 4) & 15, i = e & 15, mine = s_row[16 * q + i];
    if (mine < 0 || j0 + j >= cr) continue;
    const double2 o = cadd(cadd(sC[0][q][i][j], sC[1][q][i][j]), cadd(sC[2][q][i][j], sC[3][q][i][j]));
    gst(C.vout + (size_t)(j0 + j) * C.rows_out + r0 + mine, o);
  }
}

hipError_t launch_chain(const ChainTask* d_tasks, int ntasks, int total_blocks, int fp32, hipStream_t s) {
  if (total_blocks <= 0) return hipSuccess;
  if (fp32)
    hipLaunchKernelGGL(k_chain<float2>, dim3(total_blocks), dim3(512), 0, s, d_tasks, ntasks);
  else
    hipLaunchKernelGGL(k_chain<double2>, dim3(total_blocks), dim3(512), 0, s, d_tasks, ntasks);
  return hipGetLastError();
}

// ------------------------------------------------------------------ sum_{ij} a_ij b_ij
__global__ __launch_bounds__(256) void k_trace_prod(const double2* const* a, const double2* const* b,
                                                    const int* dims, double2* out) {
  __shared__ double2 red[256];
  const int t = blockIdx.x;
  const size_t n = (size_t)dims[t] * dims[t];
  double2 acc = make_double2(0, 0);
  for (size_t e = threadIdx.x; e < n; e += 256) acc = cfma(a[t][e], b[t][e], acc);
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = cadd(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[t] = red[0];
}

hipError_t launch_trace_prod(const double2* const* d_a, const double2* const* d_b, const int* d_dims,
                             double2* d_out, int ntasks, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_trace_prod, dim3(ntasks), dim3(256), 0, s, d_a, d_b, d_dims, d_out);
  return hipGetLastError();
}

// ------------------------------------------------------------------ one measured site of the sampling
// One wave per shot: the rows' products, the choice and the copy of the chosen rows (bound by the read
// of X and U, 2 rho d chi_r complex128 per shot; the choice stays on the device, so that a site costs
// no round trip to the host).
__global__ __launch_bounds__(256) void k_sample_pick(SampleTask T) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T.shots) return;
  const int half = T.kap * T.cr, per = T.rho * half;  // elements of one outcome: of a row group, of a shot
  const size_t base = (size_t)t * 2 * per;
  double p[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    double acc = 0.0;
    for (int e = lane; e < per; e += 64) {
      const size_t o = base + (size_t)(e / half) * 2 * half + (size_t)b * half + e % half;
      const double2 x = T.X[o], u = T.U[o];
      acc += fma(u.x, x.x, u.y * x.y);
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    p[b] = acc * T.f[t];
    if (fabs(p[b]) < 1e-12) p[b] = 0.0;
  }
  const int bit = T.draws[(size_t)t * T.stride] <= p[0] ? 0 : 1;
  const double pb = bit ? p[1] : p[0];
  if (lane == 0) {
    T.out[(size_t)t * T.stride] = bit ? '1' : '0';
    if (pb > 0.0) T.f[t] /= pb;
  }
  for (int e = lane; e < per; e += 64)
    T.V[(size_t)t * per + e] = T.X[base + (size_t)(e / half) * 2 * half + (size_t)bit * half + e % half];
}

hipError_t launch_sample_pick(const SampleTask& task, hipStream_t s) {
  if (task.shots <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sample_pick, dim3((task.shots + 3) / 4), dim3(256), 0, s, task);
  return hipGetLastError();
}

// ------------------------------------------------------------------ sum_e z_e a_e conj(b_e), real part
__global__ __launch_bounds__(256) void k_dot(const DotTask* tasks, double* out) {
  __shared__ double red[4];
  const DotTask& T = tasks[blockIdx.x];
  const size_t per = (size_t)T.d * T.cr, n = (size_t)T.rows * per, half = per / 2;
  double acc0 = 0.0, acc1 = 0.0;
  for (size_t e = (size_t)blockIdx.y * 256 + threadIdx.x; e < n; e += (size_t)DOT_BLOCKS * 256) {
    const double2 a = gld(T.a + e), b = gld(T.b + e);
    const double v = fma(a.x, b.x, a.y * b.y);
    if (e % per < half) acc0 += v;
    else acc1 += v;
  }
  double acc = T.z0 * acc0 + T.z1 * acc1;
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[(size_t)blockIdx.x * DOT_BLOCKS + blockIdx.y] = (red[0] + red[1]) + (red[2] + red[3]);
}

hipError_t launch_dot(const DotTask* d_tasks, double* d_out, int ntasks, hipStream_t s) {
  if (ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_dot, dim3(ntasks, DOT_BLOCKS), dim3(256), 0, s, d_tasks, d_out);
  return hipGetLastError();
}

// ------------------------------------------------------------------ misc
__global__ void k_check_finite(const double* p, size_t n, int* flag) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n && !isfinite(p[i])) atomicOr(flag, 1);
}
__global__ void k_check_finite_f(const float* p, size_t n, int* flag) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n && !isfinite(p[i])) atomicOr(flag, 1);
}
hipError_t launch_check_finite(const void* p, size_t n_complex, int fp32, int* d_flag, hipStream_t s) {
  size_t n = 2 * n_complex;
  if (n == 0) return hipSuccess;
  dim3 g((unsigned)((n + 255) / 256));
  if (fp32) hipLaunchKernelGGL(k_check_finite_f, g, dim3(256), 0, s, (const float*)p, n, d_flag);
  else hipLaunchKernelGGL(k_check_finite, g, dim3(256), 0, s, (const double*)p, n, d_flag);
  return hipGetLastError();
}

__global__ void k_fill_identity1(double2* p) { p[0] = make_double2(1.0, 0.0); }
hipError_t launch_fill_identity1(double2* p, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_identity1, dim3(1), dim3(1), 0, s, p);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fill_c(double2* p, size_t n, double2 v) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}
hipError_t launch_fill_c(double2* p, size_t n, double2 v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_c, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

// density-matrix readout: label A holds, in base-4 digit t, the ket (2s) and bra (1s) component
// of the t-th measured site; element A goes to out[x + 2^k x'] with x, x' the components placed
// at the bits P.pos[t]
__global__ __launch_bounds__(256) void k_rdm_scatter(const double2* __restrict__ E, double2* __restrict__ out,
                                                     size_t count, RdmPerm P) {
  for (size_t a = (size_t)blockIdx.x * 256 + threadIdx.x; a < count; a += (size_t)gridDim.x * 256) {
    size_t x = 0, xb = 0;
    for (int t = 0; t < P.k; ++t) {
      const size_t d = (a >> (2 * t)) & 3;
      x |= (d >> 1) << P.pos[t];
      xb |= (d & 1) << P.pos[t];
    }
    out[x + (xb << P.k)] = E[a];
  }
}

hipError_t launch_rdm_scatter(const double2* E, double2* out, const RdmPerm& P, hipStream_t s) {
  const size_t count = (size_t)1 << (2 * P.k);
  const unsigned blocks = (unsigned)std::min<size_t>((count + 255) / 256, 65536);
  hipLaunchKernelGGL(k_rdm_scatter, dim3(blocks), dim3(256), 0, s, E, out, count, P);
  return hipGetLastError();
}

}  // namespace hipmps
