// Ladder sums through the part of the matrix that the q-points of a (channel, w) group share.
//
// A(q) = chi0^-1(q) delta_vv' + (Gamma - U_r - V_r(q)) / beta^2. Gamma, by far the largest part, is
// the same for every q of a group, and chi0^-1(q) differs little from its mean over q. With
//   A0 = mean_q A(q),   D(q) = A(q) - A0   (blocks of nb^2 x nb^2 on the v = v' diagonal, and a
//                                           rank-nb^2 term of V_r(q) - mean V_r),
// and P = A0^-1 formed once per group, P A(q) = 1 + P D(q) is close to 1 (spectral radius of P D(q)
// 0.01 ... 0.8 on the synthetic models of 1 to 3 orbitals, beta = 5 ... 40, U = 2 ... 8), and every
// column of every q is solved by GMRES on it. One iteration of all q and right-hand sides of a
// group is one n x n by n x (nq nb^2) product on the matrix cores plus one pass over the Krylov
// basis, where the LU factors an own n x n matrix for every q: at n = 720 and 91 q-points 15
// products of 3.4 GF per group against 91 factorisations of 1.0 GF that stream 47.8 GB.
//
// Each cycle runs up to SH_M iterations from the residual of the current X, B - A0 X - D(q) X, formed
// in FP64 from A0 and D(q) themselves, so the error of P only slows the convergence down; X ends as
// an LU solution with a step of iterative refinement does. The mixed forms hold the basis, P and D(q) in
// complex64 and multiply P on the FP32 or (split) BF16 matrix cores: 62 groups at n = 720 with 91 q-points
// 80 ms in complex128, 40 in split BF16 (LU: 235 and 94). Every column has its own Hessenberg matrix and
// status on the device; tiles of 64 columns (SH_TN) without an active column are skipped by the
// products and the basis kernels, and no value is read by the host, so a call can be captured.
// Problems with a column that does not converge (a singular or nearly singular A(q), a NaN), and those of a
// group whose matrices may be singular in a way that the right-hand sides do not show (shared_equal_rows), are
// collected on the device and solved by the LU with partial pivoting, whose info they report.
#include <algorithm>
#include <cstdlib>
#include <string>
#include <type_traits>

#include "dgami.h"
#include "dgami_internal.hpp"
#include "dgami_launch.hpp"
#include "ladder_common.hpp"
#include "ladder_shared.hpp"
#include "ladder_tune.hpp"
#include "cgemm.hpp"
#include "zgemm.hpp"

namespace dgami {

int ladder_col_variant(int n, int nrhs);
int ladder_col_launch(int variant, const LadderArgs& a, hipStream_t stream);
int ladder_blocked_fp64(const LadderArgs& a, int variant, hipStream_t stream);

constexpr int SH_TN = ZG_TN;       // columns of a workgroup, and of a tile of the products
constexpr int SH_WAVES = 4;        // wavefronts of a workgroup, which share the rows of its columns

// S: type of the Krylov basis and of what it is multiplied with.
template <typename S>
struct SharedArgs : SharedGroups {
  typedef S Scalar;
  int ntile;              // tiles of SH_TN columns
  size_t cols;            // columns of the batch
  const S* ps;            // P and D(q) in S (the originals where S is double2)
  const __bf16* pb;       // P split for the BF16 matrix cores (cgemm.hpp) in place of ps, or null
  const S* ds;
  S* V;                   // [SH_M + 1][groups][n][N] Krylov basis
  S* u;                   // operand of the products [groups][n][N]
  S* g;                   // their result
  double2* ax;            // A0 X [groups][n][N] (where S is double2: g)
  double2* X;             // solution
  double2* sums;          // [groups][T][N] sums over v of the vector D(q) is applied to (with dv)
  // per column, column fastest
  double* rc;             // [SH_M] rotations
  double2* rs;
  double2* R;             // [SH_ROT] triangular factor, column j at j (j + 1) / 2
  double2* gv;            // [SH_M + 1] rotated residual
  double* beta0;
  double* target;
  double* xnorm;
  int* kdim;              // vectors of the current cycle
  int* live;              // 1 while the column iterates in the current cycle
  int* tile_run;          // [groups][ntile] 1 while the tile has a running column
  int* tile_live;         // [groups][ntile] 1 while the tile has a column iterating in this cycle
};

// Ends of a cycle and of the iteration, by the type of the basis (ladder_shared.hpp).
template <typename S>
struct SharedTol {
  static constexpr double cycle = SH_CYCLE_TOL, done = SH_DONE_TOL, trust = SH_TRUST;
  static constexpr double lowest = SH_NORM_MIN, highest = SH_NORM_MAX;
};
template <>
struct SharedTol<float2> {
  static constexpr double cycle = SH_CYCLE_TOL_C64, done = SH_DONE_TOL_C64, trust = SH_TRUST_C64;
  static constexpr double lowest = SH_NORM_MIN_C64, highest = SH_NORM_MAX_C64;
};

__device__ __forceinline__ double2 sh_wide(double2 x) { return x; }
__device__ __forceinline__ double2 sh_wide(float2 x) { return make_double2(x.x, x.y); }
template <typename S>
__device__ __forceinline__ S sh_narrow(double2 x) {
  if constexpr (std::is_same<S, float2>::value)
    return make_float2(static_cast<float>(x.x), static_cast<float>(x.y));
  else
    return x;
}
__device__ __forceinline__ float2 sh_zero(float2*) { return make_float2(0.f, 0.f); }
__device__ __forceinline__ double2 sh_zero(double2*) { return make_double2(0.0, 0.0); }

// Complex64 copy.
__global__ void __launch_bounds__(256) shared_narrow_kernel(const double2* __restrict__ in, float2* __restrict__ out,
                                                            size_t count) {
  const size_t i = blockIdx.x * static_cast<size_t>(256) + threadIdx.x;
  if (i < count) out[i] = sh_narrow<float2>(in[i]);
}

// ---------------------------------------------------------------------------
// D(q) = chi0^-1(q) - mean over q and the mean, one wavefront per (w, block, v); zero [nw][T][nv]: whether an element
// of a diagonal block vanishes.
__global__ void __launch_bounds__(256) shared_mean_kernel(const double2* __restrict__ ci, double2* __restrict__ mean,
                                                          double2* __restrict__ dd, int rows, int nq, int T, int nv,
                                                          int* __restrict__ zero, int* __restrict__ count) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *count = 0;  // of the unconverged problems
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const double2* src = ci + static_cast<size_t>(row) * nq;
  double2 s = make_double2(0.0, 0.0);
  bool none = false;
  for (int q = lane; q < nq; q += 64) {
    const double2 x = src[q];
    s = cadd(s, x);
    none |= x.x == 0.0 && x.y == 0.0;
  }
  for (int o = 32; o > 0; o >>= 1) s = cadd(s, make_double2(__shfl_xor(s.x, o), __shfl_xor(s.y, o)));
  s = cscale(s, 1.0 / nq);
  for (int q = lane; q < nq; q += 64) dd[static_cast<size_t>(row) * nq + q] = csub(src[q], s);
  const bool any = __any(none);
  if (lane == 0) {
    mean[row] = s;
    const int blk = row / nv % (T * T), c = blk / T;
    if (blk == c * T + c) zero[(row / nv / (T * T) * T + c) * nv + row % nv] = any;
  }
}

// The same for V_r [nchan][nq][T*T]: one wavefront per (chan, block); dv is scaled by 1 / beta^2.
__global__ void __launch_bounds__(64) shared_vmean_kernel(LadderArgs a, double2* __restrict__ mean,
                                                          double2* __restrict__ dv) {
  const int TT = a.T * a.T, chan = blockIdx.x / TT, e = blockIdx.x - chan * TT, lane = threadIdx.x;
  const double2* src = a.v_r + static_cast<size_t>(chan) * a.nq * TT + e;
  double2 s = make_double2(0.0, 0.0);
  for (int q = lane; q < a.nq; q += 64) s = cadd(s, src[static_cast<size_t>(q) * TT]);
  for (int o = 32; o > 0; o >>= 1) s = cadd(s, make_double2(__shfl_xor(s.x, o), __shfl_xor(s.y, o)));
  s = cscale(s, 1.0 / a.nq);
  double2* dst = dv + static_cast<size_t>(chan) * a.nq * TT + e;
  for (int q = lane; q < a.nq; q += 64)
    dst[static_cast<size_t>(q) * TT] = cscale(csub(src[static_cast<size_t>(q) * TT], s), a.inv_beta2);
  if (lane == 0) mean[blockIdx.x] = s;
}

// z0 = P B: sums of P over the frequencies of every orbital pair. One wavefront per (group, row); in the last
// s.groups workgroups the look for equal rows of the groups (n uint4 of LDS).
__global__ void __launch_bounds__(256) shared_rhs_kernel(SharedGroups s, double2* __restrict__ z0) {
  const int n = s.a.n, T = s.a.T, nv = s.a.nv, rows = s.groups * n, grp = blockIdx.x - (gridDim.x - s.groups);
  if (grp >= 0) {
    extern __shared__ uint4 s_hash[];
    const bool equal = shared_equal_rows(s, grp, s_hash);
    if (threadIdx.x == 0) s.equal[grp] = equal;
    return;
  }
  const double2* P = s.P;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  for (int t = 0; t < T; ++t) {
    const double2* src = P + static_cast<size_t>(row) * n + t * nv;
    double2 s = make_double2(0.0, 0.0);
    for (int v = lane; v < nv; v += 64) s = cadd(s, src[v]);
    for (int o = 32; o > 0; o >>= 1) s = cadd(s, make_double2(__shfl_xor(s.x, o), __shfl_xor(s.y, o)));
    if (lane == 0) z0[static_cast<size_t>(row) * T + t] = s;
  }
}

// ---------------------------------------------------------------------------
// Workgroups of the kernels below: one tile of SH_TN columns of one group; thread (wave, lane) owns
// column `lane` of the tile and the rows i = wave + SH_WAVES k, so that a row of the tile is one 1 KiB
// run. They are bound by the reads of the basis.
struct SharedTile {
  int grp, e, q, t, wave, lane;  // batch-local group, column (clamped), its q and right-hand side
  bool in;
  size_t base, col;              // offset of the column in a [groups][n][N] vector, column of the batch
};

template <typename S>
__device__ __forceinline__ SharedTile shared_tile(const SharedArgs<S>& s) {
  SharedTile x;
  x.grp = blockIdx.x / s.ntile;
  const int tile = blockIdx.x - x.grp * s.ntile;
  x.lane = threadIdx.x & 63;
  x.wave = threadIdx.x >> 6;
  const int e = tile * SH_TN + x.lane;
  x.in = e < s.N;
  x.e = x.in ? e : s.N - 1;
  x.q = x.e / s.a.T;
  x.t = x.e - x.q * s.a.T;
  x.base = static_cast<size_t>(x.grp) * s.a.n * s.N + x.e;
  x.col = static_cast<size_t>(x.grp) * s.N + x.e;
  return x;
}

// Sum over the wavefronts of a workgroup of one value per column.
__device__ __forceinline__ double2 wave_sum(double2 (&sh)[SH_WAVES][SH_TN], double2 v, const SharedTile& x) {
  __syncthreads();
  sh[x.wave][x.lane] = v;
  __syncthreads();
  double2 r = sh[0][x.lane];
#pragma unroll
  for (int k = 1; k < SH_WAVES; ++k) r = cadd(r, sh[k][x.lane]);
  return r;
}

// D(q) of a column's frequency-diagonal part for nb = 1 (row i = v).
template <typename S>
__device__ __forceinline__ const double2* shared_diag(const SharedArgs<S>& s, const SharedTile& x) {
  const int w = (s.group0 + x.grp) % s.a.nw;
  return s.dd + static_cast<size_t>(w) * s.a.n * s.a.nq + x.q;
}

// Start of a cycle: b = z0 (first) or P r (in s.g); V_0 = b / |b| and the column's state. DIAG
// (one orbital, no V_r): u = D(q) V_0 here too.
template <typename S, bool DIAG>
__global__ void __launch_bounds__(256) shared_start_kernel(SharedArgs<S> s, int first) {
  const int tile_id = blockIdx.x;
  if (!first && s.tile_run[tile_id] == 0) return;
  __shared__ double2 sh[SH_WAVES][SH_TN];
  const SharedTile x = shared_tile(s);
  const int n = s.a.n;
  const double2* b = s.z0 + static_cast<size_t>(x.grp) * n * s.a.T + x.t;
  const S* g = s.g + x.base;
  auto at = [&](int i) { return first ? b[static_cast<size_t>(i) * s.a.T] : sh_wide(g[static_cast<size_t>(i) * s.N]); };
  double nrm = 0.0;
#pragma unroll 4
  for (int i = x.wave; i < n; i += SH_WAVES) {
    const double2 y = at(i);
    nrm = fma(y.x, y.x, fma(y.y, y.y, nrm));
  }
  nrm = sqrt(wave_sum(sh, make_double2(nrm, 0.0), x).x);
  const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
  const double2* dd = shared_diag(s, x);
#pragma unroll 4
  for (int i = x.wave; i < n; i += SH_WAVES) {
    const double2 v = cscale(at(i), inv);
    const size_t o = x.base + static_cast<size_t>(i) * s.N;
    if (x.in) s.V[o] = sh_narrow<S>(v);
    if constexpr (DIAG) {
      if (x.in) s.u[o] = sh_narrow<S>(cmul(dd[static_cast<size_t>(i) * s.a.nq], v));
    }
  }
  if (x.wave == 0) {
    int st = first ? SH_RUN : s.state[x.col];
    const double xn = first ? nrm : s.xnorm[x.col];
    if (!(nrm <= 1e300)) st = SH_FAIL;  // infinite or NaN
    if (first && !(nrm >= SharedTol<S>::lowest && nrm <= SharedTol<S>::highest)) st = SH_FAIL;
    if (st == SH_RUN && nrm <= SharedTol<S>::done * xn) st = SH_DONE;
    if (st == SH_RUN && !first && nrm > SH_STAGNATION * xn) st = SH_FAIL;  // P is no inverse
    const int live = x.in && st == SH_RUN;
    if (x.in) {
      s.state[x.col] = st;
      s.live[x.col] = live;
      s.beta0[x.col] = nrm;
      s.target[x.col] = fmax(SharedTol<S>::cycle * nrm, SharedTol<S>::done * xn);
      s.kdim[x.col] = 0;
      s.gv[x.col] = make_double2(nrm, 0.0);
    }
    const unsigned long long any = __ballot(live);
    if (x.lane == 0) s.tile_live[tile_id] = any != 0;
  }
}

// Iteration k: w = P u (in s.g) is orthogonalised against V_0 .. V_k (KC = k + 1 rounded up to even;
// the pointer of an index beyond k is that of V_k and its coefficient 0), V_(k+1) is written (with
// DIAG u = D(q) V_(k+1) too), and the column's Hessenberg matrix (1 + P D(q) projected) and
// residual are updated. |w - projection| comes from |w|^2 - sum |h|^2: w = P D(q) V_k itself is
// orthogonalised, not V_k + w, so little cancels, and V and the Hessenberg matrix stay consistent.
template <typename S, bool DIAG, int KC>
__global__ void __launch_bounds__(256) shared_step_kernel(SharedArgs<S> s, int k) {
  const int tile_id = blockIdx.x;
  if (s.tile_live[tile_id] == 0) return;
  __shared__ double2 sh[SH_WAVES][SH_TN];
  const SharedTile x = shared_tile(s);
  const int n = s.a.n, N = s.N;
  const size_t vec = static_cast<size_t>(s.groups) * n * N;
  const S* Vp[KC];
#pragma unroll
  for (int j = 0; j < KC; ++j) Vp[j] = s.V + static_cast<size_t>(j <= k ? j : k) * vec + x.base;
  const S* w = s.g + x.base;
  double2 h[KC];
#pragma unroll
  for (int j = 0; j < KC; ++j) h[j] = make_double2(0.0, 0.0);
  double nrm = 0.0;
#pragma unroll 2
  for (int i = x.wave; i < n; i += SH_WAVES) {
    const size_t o = static_cast<size_t>(i) * N;
    const double2 y = sh_wide(w[o]);
    S p[KC];
#pragma unroll
    for (int j = 0; j < KC; ++j) p[j] = Vp[j][o];
    nrm = fma(y.x, y.x, fma(y.y, y.y, nrm));
#pragma unroll
    for (int j = 0; j < KC; ++j) h[j] = cfma(h[j], cconj(sh_wide(p[j])), y);
  }
  nrm = wave_sum(sh, make_double2(nrm, 0.0), x).x;
  double left = nrm;
#pragma unroll
  for (int j = 0; j < KC; ++j) {
    h[j] = wave_sum(sh, h[j], x);
    if (j > k) h[j] = make_double2(0.0, 0.0);
    left -= h[j].x * h[j].x + h[j].y * h[j].y;
  }
  if constexpr (std::is_same<S, float2>::value) left = fmax(left, SH_LOSS_C64 * nrm);
  const double hn = sqrt(fmax(left, 0.0));
  const double inv = hn > 1e-150 ? 1.0 / hn : 0.0;
  const double2* dd = shared_diag(s, x);
  S* Vn = s.V + static_cast<size_t>(k + 1) * vec + x.base;
  S* un = s.u + x.base;
#pragma unroll 2
  for (int i = x.wave; i < n; i += SH_WAVES) {
    const size_t o = static_cast<size_t>(i) * N;
    double2 y = sh_wide(w[o]);
    S p[KC];
#pragma unroll
    for (int j = 0; j < KC; ++j) p[j] = Vp[j][o];
#pragma unroll
    for (int j = 0; j < KC; ++j) y = cfms(y, h[j], sh_wide(p[j]));
    y = cscale(y, inv);
    if (x.in) Vn[o] = sh_narrow<S>(y);
    if constexpr (DIAG) {
      if (x.in) un[o] = sh_narrow<S>(cmul(dd[static_cast<size_t>(i) * s.a.nq], y));
    }
  }
  if (x.wave == 0) {
    int live = x.in && s.live[x.col];
    if (live) {
      const size_t cols = s.cols, col = x.col;
#pragma unroll
      for (int j = 0; j < KC; ++j)
        if (j == k) h[j].x += 1.0;
#pragma unroll
      for (int j = 0; j + 1 < KC; ++j) {
        if (j < k) {
          const double c = s.rc[j * cols + col];
          const double2 sn = s.rs[j * cols + col];
          const double2 t = cfma(cscale(h[j], c), sn, h[j + 1]);
          h[j + 1] = cfms(cscale(h[j + 1], c), cconj(sn), h[j]);
          h[j] = t;
        }
      }
      double2 hk = make_double2(0.0, 0.0);
#pragma unroll
      for (int j = 0; j < KC; ++j)
        if (j == k) hk = h[j];
      const double ah = hypot(hk.x, hk.y), r = hypot(ah, hn);
      const double c = r > 0.0 ? ah / r : 1.0;
      const double2 ph = ah > 0.0 ? cscale(hk, 1.0 / ah) : make_double2(1.0, 0.0);
      const double2 sn = cscale(ph, r > 0.0 ? hn / r : 0.0);
      s.rc[k * cols + col] = c;
      s.rs[k * cols + col] = sn;
      const size_t rk = static_cast<size_t>(k) * (k + 1) / 2;
#pragma unroll
      for (int j = 0; j < KC; ++j)
        if (j < k) s.R[(rk + j) * cols + col] = h[j];
      s.R[(rk + k) * cols + col] = cscale(ph, r);
      const double2 gk = s.gv[k * cols + col];
      s.gv[k * cols + col] = cscale(gk, c);
      const double2 gn = cmul(make_double2(-sn.x, sn.y), gk);
      s.gv[(k + 1) * cols + col] = gn;
      s.kdim[col] = k + 1;
      const double res = hypot(gn.x, gn.y);
      // converged, broken down, or not a number: the column waits for the end of the cycle
      live = res > s.target[col] && hn > 0.0 && k + 1 < SH_M;
      s.live[col] = live;
    }
    const unsigned long long any = __ballot(live);
    if (x.lane == 0) s.tile_live[tile_id] = any != 0;
  }
}

// End of a cycle: X (+)= sum_j y_j V_j with the y of the column's triangular factor, and its state. With a
// complex64 basis the residual sum_j rho_j V_j is formed in the same pass (rho: the rotated residual turned
// back; one more vector is read).
template <typename S>
__global__ void __launch_bounds__(256) shared_update_kernel(SharedArgs<S> s, int cycle, int last) {
  const int tile_id = blockIdx.x;
  if (cycle > 0 && s.tile_run[tile_id] == 0) return;
  __shared__ double2 sh[SH_WAVES][SH_TN];
  __shared__ int s_kmax;
  const SharedTile x = shared_tile(s);
  const int n = s.a.n, N = s.N;
  const size_t vec = static_cast<size_t>(s.groups) * n * N, cols = s.cols, col = x.col;
  const bool run = s.state[col] == SH_RUN;
  const int kd = run ? s.kdim[col] : 0;
  double2 y[SH_M];
#pragma unroll
  for (int j = SH_M - 1; j >= 0; --j) {
    y[j] = make_double2(0.0, 0.0);
    if (j < kd) {
      double2 r = s.gv[j * cols + col];
#pragma unroll
      for (int l = j + 1; l < SH_M; ++l)
        if (l < kd) r = cfms(r, s.R[(static_cast<size_t>(l) * (l + 1) / 2 + j) * cols + col], y[l]);
      y[j] = cmul(r, cinv(s.R[(static_cast<size_t>(j) * (j + 1) / 2 + j) * cols + col]));
    }
  }
  constexpr bool C64 = std::is_same<S, float2>::value;
  double2 rho[C64 ? SH_M : 1], end = make_double2(0.0, 0.0);  // end: of V_kd
  double ynrm = 0.0;
  if constexpr (C64) {
    double2 cur = kd > 0 ? s.gv[static_cast<size_t>(kd) * cols + col] : end;
#pragma unroll
    for (int j = SH_M; j > 0; --j) {
      if (j < SH_M) rho[j] = make_double2(0.0, 0.0);
      if (j <= kd) {
        const double2 e = cscale(cur, s.rc[(j - 1) * cols + col]);
        if (j < SH_M) rho[j] = e;
        if (j == kd) end = e;
        const double2 sn = s.rs[(j - 1) * cols + col];
        cur = cmul(make_double2(-sn.x, -sn.y), cur);
      }
    }
    rho[0] = cur;
#pragma unroll
    for (int j = 0; j < SH_M; ++j) ynrm = fma(y[j].x, y[j].x, fma(y[j].y, y[j].y, ynrm));
    ynrm = sqrt(ynrm);
  }
  if (x.wave == 0) {
    int km = kd;
    for (int o = 32; o > 0; o >>= 1) km = max(km, __shfl_xor(km, o));
    if (x.lane == 0) s_kmax = km;
  }
  __syncthreads();
  const int kmax = s_kmax;
  double nrm = 0.0, left = 0.0;  // |X|^2 and, with a complex64 basis, the residual's square
  auto pass = [&](auto kc_tag) {
    constexpr int KC = decltype(kc_tag)::value;
#pragma unroll 2
    for (int i = x.wave; i < n; i += SH_WAVES) {
      const size_t o = x.base + static_cast<size_t>(i) * N;
      S p[KC];
#pragma unroll
      for (int j = 0; j < KC; ++j) p[j] = s.V[static_cast<size_t>(j < kmax ? j : 0) * vec + o];
      double2 acc = cycle > 0 ? s.X[o] : make_double2(0.0, 0.0);
      if constexpr (C64) {
        const double2 v = sh_wide(s.V[static_cast<size_t>(kmax) * vec + o]);
        double2 r = kd == kmax ? cmul(end, v) : make_double2(0.0, 0.0);
#pragma unroll
        for (int j = 0; j < KC; ++j)
          if (j <= kd && j < kmax) r = cfma(r, rho[j], sh_wide(p[j]));
        left = fma(r.x, r.x, fma(r.y, r.y, left));
      }
#pragma unroll
      for (int j = 0; j < KC; ++j)
        if (j < kd) acc = cfma(acc, y[j], sh_wide(p[j]));
      nrm = fma(acc.x, acc.x, fma(acc.y, acc.y, nrm));
      if (x.in) s.X[o] = acc;
    }
  };
  switch ((kmax + 1) / 2) {
    case 0:
    case 1: pass(std::integral_constant<int, 2>{}); break;
    case 2: pass(std::integral_constant<int, 4>{}); break;
    case 3: pass(std::integral_constant<int, 6>{}); break;
    case 4: pass(std::integral_constant<int, 8>{}); break;
    default: pass(std::integral_constant<int, SH_M>{}); break;
  }
  const double2 norms = wave_sum(sh, make_double2(nrm, left), x);
  const double xn = sqrt(norms.x);
  if (x.wave == 0) {
    int st = s.state[col];
    if (run) {
      const double2 g = s.gv[static_cast<size_t>(kd) * cols + col];
      const double b0 = s.beta0[col], res = C64 ? sqrt(norms.y) : hypot(g.x, g.y);
      if (!(xn <= 1e300) || !(res <= 1e300))
        st = SH_FAIL;
      else if (cycle > 0 && res <= 2.0 * SharedTol<S>::done * xn && fmax(b0, ynrm) <= SharedTol<S>::trust * xn)
        st = SH_DONE;
      else if (last || !(res <= SH_STAGNATION * b0))
        st = SH_FAIL;
    }
    if (x.in) {
      s.state[col] = st;
      s.xnorm[col] = xn;
    }
    const unsigned long long any = __ballot(x.in && st == SH_RUN);
    if (x.lane == 0) s.tile_run[tile_id] = any != 0;
  }
}

// ---------------------------------------------------------------------------
// Sums over v of every orbital pair's rows of v ([groups][T][N], for the V_r term). One workgroup per tile.
template <int T, typename S, typename V>
__global__ void __launch_bounds__(256) shared_sums_kernel(SharedArgs<S> s, const V* __restrict__ v,
                                                          const int* __restrict__ tiles) {
  if (tiles[blockIdx.x] == 0) return;
  __shared__ double2 sh[SH_WAVES][SH_TN];
  const SharedTile x = shared_tile(s);
  const int nv = s.a.nv, N = s.N;
  for (int c = 0; c < T; ++c) {
    double2 sv = make_double2(0.0, 0.0);
    for (int vi = x.wave; vi < nv; vi += SH_WAVES) sv = cadd(sv, sh_wide(v[x.base + static_cast<size_t>(c * nv + vi) * N]));
    sv = wave_sum(sh, sv, x);
    if (x.in && x.wave == 0) s.sums[(static_cast<size_t>(x.grp) * T + c) * N + x.e] = sv;
  }
}

// u = D(q) v, or (RESIDUAL, in FP64 throughout) u = B - A0 v - D(q) v with A0 v in s.ax. grid (tiles, ceil(nv / 4)), one
// frequency per wavefront. The blocks of the tile's q-points are staged in LDS, coalesced over q; read
// by every column from global memory they made this step 5 times slower than its traffic.
template <int T, bool RESIDUAL, typename S>
__global__ void __launch_bounds__(256) shared_apply_kernel(
    SharedArgs<S> s, const typename std::conditional<RESIDUAL, double2, S>::type* __restrict__ v,
    const int* __restrict__ tiles) {
  typedef typename std::conditional<RESIDUAL, double2, S>::type V;
  if (tiles[blockIdx.x] == 0) return;
  constexpr int QT = (63 + T - 1) / T + 1;  // most q-points of a tile
  __shared__ V s_d[SH_WAVES][T * T][QT];
  const SharedTile x = shared_tile(s);
  const int nv = s.a.nv, nq = s.a.nq, N = s.N;
  const int vi = blockIdx.y * SH_WAVES + x.wave;
  const int g = s.group0 + x.grp, w = g % s.a.nw, chan = g / s.a.nw;
  const int q0 = (blockIdx.x - x.grp * s.ntile) * SH_TN / T;
  V y[T];
  if (vi < nv) {
    const V* dd;
    if constexpr (RESIDUAL)
      dd = s.dd;
    else
      dd = s.ds;
    dd += (static_cast<size_t>(w) * T * T * nv + vi) * nq;
    for (int e = x.lane; e < T * T * QT; e += 64) {
      const int blk = e / QT, qq = e - blk * QT;
      if (q0 + qq < nq) s_d[x.wave][blk][qq] = dd[static_cast<size_t>(blk) * nv * nq + q0 + qq];
    }
#pragma unroll
    for (int c = 0; c < T; ++c) y[c] = v[x.base + static_cast<size_t>(c * nv + vi) * N];
  }
  __syncthreads();
  if (vi >= nv || !x.in) return;
  const int qq = x.q - q0;
#pragma unroll
  for (int r = 0; r < T; ++r) {
    V sum = sh_zero(static_cast<V*>(nullptr));
#pragma unroll
    for (int c = 0; c < T; ++c) sum = cfma(sum, s_d[x.wave][r * T + c][qq], y[c]);
    double2 acc = sh_wide(sum);
    if (s.dv) {
      const double2* dv = s.dv + (static_cast<size_t>(chan) * nq + x.q) * T * T + r * T;
      for (int c = 0; c < T; ++c) acc = cfms(acc, dv[c], s.sums[(static_cast<size_t>(x.grp) * T + c) * N + x.e]);
    }
    const size_t o = x.base + static_cast<size_t>(r * nv + vi) * N;
    if constexpr (RESIDUAL) acc = csub(make_double2(r == x.t ? 1.0 : 0.0, 0.0), cadd(s.ax[o], acc));
    s.u[o] = sh_narrow<S>(acc);
  }
}

// out = X / beta, q fastest. grid (n, groups).
template <typename S>
__global__ void __launch_bounds__(256) shared_output_kernel(SharedArgs<S> s) {
  const LadderArgs& a = s.a;
  const int i = blockIdx.x, grp = blockIdx.y;
  const double2* X = s.X + (static_cast<size_t>(grp) * a.n + i) * s.N;
  const int g = s.group0 + grp, w = g % a.nw, chan = g / a.nw;
  for (int e = threadIdx.x; e < s.N; e += 256) {
    const int t = e / a.nq, q = e - t * a.nq;
    a.out[ladder_out_index(a, chan, w, q, i, t)] = cscale(X[q * a.T + t], a.inv_beta);
  }
}

// info 0 for the converged problems of the batch; the others are appended to the list (in no order: the
// LU of a problem does not depend on its place).
__global__ void __launch_bounds__(256) shared_collect_kernel(SharedGroups s, int* __restrict__ list, int* __restrict__ count) {
  const int i = blockIdx.x * 256 + threadIdx.x, T = s.a.T;
  if (i >= s.groups * s.a.nq) return;
  bool bad = false;
  for (int t = 0; t < T; ++t) bad |= s.state[static_cast<size_t>(i) * T + t] != SH_DONE;
  bad |= s.equal[i / s.a.nq] != 0;
  const int item = s.group0 * s.a.nq + i;
  if (bad)
    list[atomicAdd(count, 1)] = item;
  else if (s.a.info)
    s.a.info[item] = 0;
}

// ---------------------------------------------------------------------------
template <bool DIAG, typename S>
static int shared_step(const SharedArgs<S>& s, int k, hipStream_t stream) {
  const dim3 gd(static_cast<unsigned>(s.groups) * s.ntile), bd(256);
  switch (k / 2) {
    case 0: hipLaunchKernelGGL((shared_step_kernel<S, DIAG, 2>), gd, bd, 0, stream, s, k); break;
    case 1: hipLaunchKernelGGL((shared_step_kernel<S, DIAG, 4>), gd, bd, 0, stream, s, k); break;
    case 2: hipLaunchKernelGGL((shared_step_kernel<S, DIAG, 6>), gd, bd, 0, stream, s, k); break;
    case 3: hipLaunchKernelGGL((shared_step_kernel<S, DIAG, 8>), gd, bd, 0, stream, s, k); break;
    default: hipLaunchKernelGGL((shared_step_kernel<S, DIAG, SH_M>), gd, bd, 0, stream, s, k); break;
  }
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

// u = D(q) v (RESIDUAL: u = B - A v with A0 v in s.ax).
template <int T, bool RESIDUAL, typename S, typename V>
static int shared_apply(const SharedArgs<S>& s, const V* v, const int* tiles, hipStream_t stream) {
  const unsigned nt = static_cast<unsigned>(s.groups) * s.ntile;
  if (s.dv) {
    hipLaunchKernelGGL((shared_sums_kernel<T, S, V>), dim3(nt), dim3(256), 0, stream, s, v, tiles);
    DGAMI_HIP_CHECK(hipGetLastError());
  }
  const dim3 gd(nt, ceil_div(s.a.nv, SH_WAVES)), bd(256);
  hipLaunchKernelGGL((shared_apply_kernel<T, RESIDUAL, S>), gd, bd, 0, stream, s, v, tiles);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

// C = A B of every group's n x n matrix, tiles without work left out.
template <typename G, typename S>
static G shared_operands(const SharedGroups& s, const S* A, const S* B, S* C, const int* tiles) {
  G g;
  g.A = A;
  g.B = B;
  g.C = C;
  g.M = g.K = g.lda = s.a.n;
  g.N = g.ldb = g.ldc = s.N;
  g.sa = static_cast<long long>(s.a.n) * s.a.n;
  g.sb = g.sc = static_cast<long long>(s.a.n) * s.N;
  g.tile_active = tiles;
  return g;
}

static int shared_product(const SharedGroups& s, const double2* A, const double2* B, double2* C, const int* tiles,
                          bool three, hipStream_t stream) {
  ZgemmArgs g = shared_operands<ZgemmArgs>(s, A, B, C, tiles);
  g.alpha = make_double2(1.0, 0.0);
  g.beta = make_double2(0.0, 0.0);
  return three ? launch_zgemm<true>(g, s.groups, stream) : launch_zgemm<false>(g, s.groups, stream);
}

// g = P u.
static int shared_precondition(const SharedArgs<double2>& s, const int* tiles, hipStream_t stream) {
  return shared_product(s, s.ps, s.u, s.g, tiles, true, stream);
}

static int shared_precondition(const SharedArgs<float2>& s, const int* tiles, hipStream_t stream) {
  static_assert(CG_TN == SH_TN, "the tiles whose activity is tracked");
  if (!s.pb) return launch_cgemm(shared_operands<CgemmArgs>(s, s.ps, s.u, s.g, tiles), s.groups, stream);
  CgemmBf16Args g;
  g.A = s.pb;
  g.B = s.u;
  g.C = s.g;
  g.M = g.K = s.a.n;
  g.lda = cgemm_split_lda(s.a.n);
  g.N = g.ldb = g.ldc = s.N;
  g.sb = g.sc = static_cast<long long>(s.a.n) * s.N;
  g.tile_active = tiles;
  return launch_cgemm_bf16x3(g, s.groups, stream);
}

template <int T, typename S>
static int shared_solve(SharedArgs<S>& s, hipStream_t stream) {
  const dim3 gd(static_cast<unsigned>(s.groups) * s.ntile), bd(256);
  const bool diag = T == 1 && !s.dv;
  const size_t vec = static_cast<size_t>(s.groups) * s.a.n * s.N;
  int rc = 0;
#define DGAMI_STEP(x) \
  if ((rc = (x)) != 0) return rc
  for (int cycle = 0; cycle < SH_CYCLES; ++cycle) {
    if (cycle > 0) {
      DGAMI_STEP(shared_product(s, s.A0, s.X, s.ax, s.tile_run, false, stream));
      DGAMI_STEP((shared_apply<T, true>(s, s.X, s.tile_run, stream)));
      DGAMI_STEP(shared_precondition(s, s.tile_run, stream));
    }
    if (diag)
      hipLaunchKernelGGL((shared_start_kernel<S, true>), gd, bd, 0, stream, s, cycle == 0 ? 1 : 0);
    else
      hipLaunchKernelGGL((shared_start_kernel<S, false>), gd, bd, 0, stream, s, cycle == 0 ? 1 : 0);
    DGAMI_HIP_CHECK(hipGetLastError());
    for (int k = 0; k < SH_M; ++k) {
      if (!diag) DGAMI_STEP((shared_apply<T, false>(s, s.V + k * vec, s.tile_live, stream)));
      // the first product of a batch, of all columns, is what dgami_profile_* times here
      hipEvent_t start = nullptr;
      const bool prof = cycle == 0 && k == 0 && profile_on();
      if (prof && profile_begin(stream, &start)) return -2;
      DGAMI_STEP(shared_precondition(s, s.tile_live, stream));
      if (prof) {
        const double nn = static_cast<double>(s.a.n) * s.a.n * s.groups;
        if (profile_end(stream, start, (nn + 2.0 * vec) * sizeof(S), 8.0 * nn * s.N)) return -2;
      }
      DGAMI_STEP(diag ? shared_step<true>(s, k, stream) : shared_step<false>(s, k, stream));
    }
    hipLaunchKernelGGL((shared_update_kernel<S>), gd, bd, 0, stream, s, cycle, cycle == SH_CYCLES - 1 ? 1 : 0);
    DGAMI_HIP_CHECK(hipGetLastError());
  }
#undef DGAMI_STEP
  return 0;
}

bool ladder_shared_applies(const LadderArgs& a, int precision) {
  if (a.dense || a.rhs_mode != LADDER_RHS_INDICATOR || a.items) return false;
  if (a.T != 1 && a.T != 4 && a.T != 9 && a.T != 16) return false;
  if (a.n > 1536 || a.nq < 2 || ladder_tune_lu_only()) return false;
  const char* v = getenv("DGAMI_LADDER_SHARED");
  if (v && *v) return std::string(v) == "1";
  if (a.nq < SHARED_MIN_NQ) return false;
  const double ratio = a.n / (3.0 * a.T) + 1.0, work = static_cast<double>(a.nchan) * a.nw * a.nq * ratio;
  if (a.n <= 32) return work >= SHARED_MIN_WORK_N32 && a.T <= SHARED_TILE_T;
  if (a.n <= SHARED_TILE_N && a.T <= SHARED_TILE_T)
    return work >= (a.T == 1 ? SHARED_MIN_WORK_1 : SHARED_MIN_WORK_4)[a.n <= 64 ? 0 : a.n <= 128 ? 1 : 2];
  return precision == DGAMI_PLAIN_FP64 ? ratio >= SHARED_MIN_RATIO && work >= SHARED_MIN_WORK
                                       : ratio >= SHARED_MIN_RATIO_MIXED && work >= SHARED_MIN_WORK_MIXED;
}

// A batch by one launch per product and per pass over the basis: vec and st hold the vectors and the
// columns' data of ng groups. With a complex64 basis (c64) A0 X has its own vector, and P and D(q) are
// there in complex64 too (in `narrow`: P or its split form, then D(q)).
static size_t large_vectors(const LadderArgs& a, size_t groups, int N, bool c64) {
  const size_t vec = static_cast<size_t>(a.n) * groups * N, sums = a.v_r ? static_cast<size_t>(a.T) * groups * N : 0;
  return c64 ? vec * ((SH_M + 3) * sizeof(float2) + 2 * sizeof(double2)) + sums * sizeof(double2)
             : (vec * (SH_M + 4) + sums) * sizeof(double2);
}
static size_t shared_narrow_p(const LadderArgs& a, size_t groups) {
  return groups * a.n * cgemm_split_lda(a.n);
}

static size_t large_state(size_t groups, int N) {
  const size_t per_col = sizeof(double2) * (SH_M + SH_ROT + SH_M + 1) + sizeof(double) * (SH_M + 3) + 2 * sizeof(int);
  return groups * (N * per_col + 2 * ceil_div(N, SH_TN) * sizeof(int));
}

template <typename S>
static int shared_large_solve(const SharedGroups& sg, char* vec, void* st, float2* narrow, const float2* ds, bool bf16,
                              hipStream_t stream) {
  SharedArgs<S> s{};
  static_cast<SharedGroups&>(s) = sg;
  const size_t cols = static_cast<size_t>(s.groups) * s.N, used = cols * s.a.n;
  s.ntile = static_cast<int>(ceil_div(s.N, SH_TN));
  s.cols = cols;
  s.X = reinterpret_cast<double2*>(vec);
  s.sums = s.X + used;
  double2* end = s.sums + (s.a.v_r ? cols * s.a.T : 0);
  if constexpr (std::is_same<S, float2>::value) {
    s.ax = end;
    end += used;
    const size_t nn = static_cast<size_t>(s.groups) * s.a.n * s.a.n;
    s.ds = ds;
    if (bf16) {
      const int ldp = cgemm_split_lda(s.a.n);
      __bf16* p = reinterpret_cast<__bf16*>(narrow);
      hipLaunchKernelGGL(cgemm_split_kernel, dim3(ceil_div(static_cast<size_t>(s.a.n) * ldp, 256), s.groups), dim3(256), 0,
                         stream, s.P, p, s.a.n, ldp);
      s.pb = p;
    } else {
      hipLaunchKernelGGL(shared_narrow_kernel, dim3(ceil_div(nn, 256)), dim3(256), 0, stream, s.P, narrow, nn);
      s.ps = narrow;
    }
    DGAMI_HIP_CHECK(hipGetLastError());
  } else {
    s.ds = s.dd;
    s.ps = s.P;
  }
  s.V = reinterpret_cast<S*>(end);
  s.u = s.V + used * (SH_M + 1);
  s.g = s.u + used;
  if constexpr (std::is_same<S, double2>::value) s.ax = s.g;
  s.rs = static_cast<double2*>(st);
  s.R = s.rs + SH_M * cols;
  s.gv = s.R + SH_ROT * cols;
  s.rc = reinterpret_cast<double*>(s.gv + (SH_M + 1) * cols);
  s.beta0 = s.rc + SH_M * cols;
  s.target = s.beta0 + cols;
  s.xnorm = s.target + cols;
  s.kdim = reinterpret_cast<int*>(s.xnorm + cols);
  s.live = s.kdim + cols;
  s.tile_run = s.live + cols;
  s.tile_live = s.tile_run + static_cast<size_t>(s.groups) * s.ntile;
  int rc = 0;
  switch (s.a.T) {
    case 1: rc = shared_solve<1>(s, stream); break;
    case 4: rc = shared_solve<4>(s, stream); break;
    case 9: rc = shared_solve<9>(s, stream); break;
    default: rc = shared_solve<16>(s, stream); break;
  }
  if (rc) return rc;
  hipLaunchKernelGGL((shared_output_kernel<S>), dim3(s.a.n, s.groups), dim3(256), 0, stream, s);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

int ladder_solve_shared(const LadderArgs& a, int precision, hipStream_t stream, int slot_offset) {
  const int n = a.n, T = a.T, nq = a.nq, TT = T * T, N = nq * T;
  const size_t G = static_cast<size_t>(a.nchan) * a.nw, nn = static_cast<size_t>(n) * n;
  const size_t items = G * nq;
  const bool tiles = n <= SHARED_TILE_N && T <= SHARED_TILE_T;
  const bool c64 = !tiles && precision != DGAMI_PLAIN_FP64;
  const size_t pk = tiles ? shared_packed(n) : 0;
  // groups per batch: matrices and, for large sizes, vectors of at most 24 GiB, fewer where the device holds less
  const size_t per_group = (2 * (nn + pk) + shared_inverse_workspace(n)) * sizeof(double2) + (tiles ? 0 : large_vectors(a, 1, N, c64)) +
                           (c64 ? shared_narrow_p(a, 1) * sizeof(float2) : 0);
  size_t gb = std::max<size_t>(1, std::min<size_t>({(size_t(24) << 30) / per_group, G, 65535}));
  SharedGroups s{};
  s.a = a;
  s.N = N;
  const size_t rows = static_cast<size_t>(a.nw) * TT * a.nv;
  const size_t vsz = a.v_r ? static_cast<size_t>(a.nchan) * TT : 0, dvsz = vsz * nq;
  double2* mean = nullptr;
  char *vec = nullptr, *st = nullptr;
  for (;; gb = (gb + 1) / 2) {
    s.groups = static_cast<int>(gb);
    const size_t szc = rows + rows * nq + vsz + dvsz + gb * ((nn + pk) * 2 + n * T + shared_inverse_workspace(n));
    const size_t nsz = c64 ? shared_narrow_p(a, gb) + rows * nq : 0;
    const size_t ints = gb * N + NUM_XCD + items + 1 + gb + static_cast<size_t>(a.nw) * n;
    mean = static_cast<double2*>(workspace(WS_SHARED + slot_offset, szc * sizeof(double2) + nsz * sizeof(float2)));
    vec = static_cast<char*>(workspace(
        WS_SHARED_VEC + slot_offset, tiles ? shared_tile_workspace(s) * sizeof(double2) : large_vectors(a, gb, N, c64)));
    st = static_cast<char*>(workspace(WS_SHARED_STATE + slot_offset, (tiles ? 0 : large_state(gb, N)) + ints * sizeof(int)));
    if (mean && vec && st) break;
    if (gb == 1) return SHARED_NO_SPACE;
  }
  double2* dd = mean + rows;
  double2* vmean = dd + rows * nq;
  double2* dv = vmean + vsz;
  double2* A0 = dv + dvsz;
  double2* P = A0 + gb * nn;
  double2* pack = P + gb * nn;
  double2* z0 = pack + 2 * gb * pk;
  double2* inv = z0 + gb * n * T;
  float2* narrow = reinterpret_cast<float2*>(inv + gb * shared_inverse_workspace(n));  // P, D(q) in complex64
  float2* ds = narrow + shared_narrow_p(a, gb);
  s.dd = dd;
  s.dv = a.v_r ? dv : nullptr;
  s.A0 = A0;
  s.P = P;
  s.z0 = z0;
  s.state = reinterpret_cast<int*>(st + (tiles ? 0 : large_state(gb, N)));
  int* next = s.state + gb * N;
  int* list = next + NUM_XCD;
  int* count = list + items;
  s.equal = count + 1;
  int* zero = s.equal + gb;
  s.zero = zero;

  hipLaunchKernelGGL(shared_mean_kernel, dim3(ceil_div(rows, 4)), dim3(256), 0, stream, a.chi0_inv, mean, dd,
                     static_cast<int>(rows), nq, T, a.nv, zero, count);
  DGAMI_HIP_CHECK(hipGetLastError());
  if (a.v_r) {
    hipLaunchKernelGGL(shared_vmean_kernel, dim3(static_cast<unsigned>(vsz)), dim3(64), 0, stream, a, vmean, dv);
    DGAMI_HIP_CHECK(hipGetLastError());
  }
  if (c64) {
    hipLaunchKernelGGL(shared_narrow_kernel, dim3(ceil_div(rows * nq, 256)), dim3(256), 0, stream, dd, ds, rows * nq);
    DGAMI_HIP_CHECK(hipGetLastError());
  }
  for (size_t g0 = 0; g0 < G; g0 += gb) {
    const int ng = static_cast<int>(std::min(gb, G - g0));
    s.group0 = static_cast<int>(g0);
    s.groups = ng;
    int rc = 0;
    rc = shared_inverse(s, mean, a.v_r ? vmean : nullptr, A0, P, inv, stream);
    if (rc) return rc;
    if (tiles) {
      rc = shared_tile_solve(s, pack, z0, reinterpret_cast<double2*>(vec), next, stream);
    } else {
      hipLaunchKernelGGL(shared_rhs_kernel, dim3(ceil_div(static_cast<size_t>(ng) * n, 4) + ng), dim3(256),
                         n * sizeof(uint4), stream, s, z0);
      DGAMI_HIP_CHECK(hipGetLastError());
      rc = c64 ? shared_large_solve<float2>(s, vec, st, narrow, ds, precision == DGAMI_MIXED_BF16X3_IR, stream)
               : shared_large_solve<double2>(s, vec, st, nullptr, nullptr, false, stream);
    }
    if (rc) return rc;
    hipLaunchKernelGGL(shared_collect_kernel, dim3(ceil_div(static_cast<size_t>(ng) * nq, 256)), dim3(256), 0, stream, s, list,
                       count);
    DGAMI_HIP_CHECK(hipGetLastError());
  }
  // The problems that did not converge, by the LU: its kernels are launched for every problem and return at once
  // beyond the device count. Up to n = 128 the column kernel, whose one launch costs 4 us where the list is empty
  // (the blocked LU's twenty about 90), though it is slower where all problems fail: with the cycles before it
  // 1890 problems of n = 40 take 0.93 ms (LU alone 0.29; with the register kernel 0.86), 6426 of n = 120 10.9 (3.8).
  LadderArgs f = a;
  f.items = list;
  f.nitems = count;
  const int v = ladder_col_variant(n, T);
  return v >= 0 ? ladder_col_launch(v, f, stream) : ladder_blocked_fp64(f, -1, stream);
}

}  // namespace dgami
