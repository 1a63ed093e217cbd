// Inverses of the mean matrices A0 that the q-points of a group share (ladder_shared.hip).
//
// Up to n = SHARED_SMALL_N one workgroup per group holds the matrix in registers; above, Gauss-Jordan
// steps over blocks of 64 rows (three launches per block). The inverse only has to be good enough for the
// iteration on it: its error shows in the residuals that the iteration forms from A0 itself, and a group
// whose inverse fails is solved by the LU with partial pivoting. The blocked steps therefore pivot inside
// their diagonal blocks only. Measured against the LU with n right-hand sides that they replace: 24
// matrices of n = 216 0.39 against 1.1 ms, 62 of n = 720 6.2 against 14 ms.
#include "dgami_internal.hpp"
#include "dgami_launch.hpp"
#include "ladder_common.hpp"
#include "ladder_shared.hpp"
#include "zmma.hpp"

namespace dgami {

constexpr int GJ_NB = 64;  // rows of a block, and of a tile of its updates
constexpr int GJ_TK = 8;

template <int RA, int CB>
struct GjLds {
  double2 col[2][32 * RA];
  double2 row[2][16 * CB];
  unsigned key[2][32];
  int idx[2][32];
  int prow[16 * CB], krow[32 * RA];
};

// Inverts the n x n matrix (n <= 32 RA, n <= 16 CB) that a workgroup of 512 holds in registers (thread (tr, tc)
// the elements (tr + 32 a, tc + 16 b)) in place, by Gauss-Jordan steps with partial pivoting, two barriers each:
// the owners of column k publish it and their best candidate, every wavefront picks the pivot row p from
// the 32 candidates, its owners publish it. Rows are not moved: row p of step k ends as row k of the
// inverse, column j as its column p_j (sh.krow, sh.prow). Column k and row p are set to zero when they are
// published and row p's factor to -1, so that the update is one complex FMA per element everywhere (with selects
// between it and the special cases 122 matrices of n = 120 took 440 us, now 238, and 42 of n = 40 58 us, now
// 45). Bound by the chain of n steps: 1 us each at n = 64.
// Returns whether a step found no finite pivot.
template <int RA, int CB>
__device__ __forceinline__ bool gj_invert(double2 (&x)[RA][CB], int n, GjLds<RA, CB>& sh) {
  const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15, lane = tid & 63;
  unsigned used = 0;
  bool bad = false;
#pragma unroll
  for (int r = 0; r < RA; ++r)
    if (tr + 32 * r >= n) used |= 1u << r;
#pragma unroll
  for (int b = 0; b < CB; ++b) {
#pragma unroll 1
    for (int kk = 0; kk < 16; ++kk) {
      const int k = 16 * b + kk, buf = k & 1;
      if (k >= n) break;
      if (tc == kk) {
        unsigned best = 0;
        int idx = tr;
#pragma unroll
        for (int r = 0; r < RA; ++r) {
          sh.col[buf][tr + 32 * r] = x[r][b];
          x[r][b] = make_double2(0.0, 0.0);  // column k of the update starts from zero
          const double m = cabs1(sh.col[buf][tr + 32 * r]);
          const unsigned key = pivot_key(m, !((used >> r) & 1u) && m <= 1.7e308);
          if (key > best) {
            best = key;
            idx = tr + 32 * r;
          }
        }
        sh.key[buf][tr] = best;
        sh.idx[buf][tr] = idx;
      }
      __syncthreads();
      const unsigned key = sh.key[buf][lane & 31], wkey = wave_max_u32(key);
      const int first = __ffsll(static_cast<long long>(__ballot(key == wkey))) - 1;
      const int p = __builtin_amdgcn_readlane(sh.idx[buf][lane & 31], first);
      bad |= wkey == 0u;  // no finite candidate
      if (tr == (p & 31)) {
#pragma unroll
        for (int r = 0; r < RA; ++r)
          if (r == p >> 5) {
            used |= 1u << r;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
              sh.row[buf][tc + 16 * c] = x[r][c];
              x[r][c] = make_double2(0.0, 0.0);
            }
          }
      }
      if (tid == 0) {
        sh.prow[k] = p;
        sh.krow[p] = k;
      }
      const double2 pinv = cinv(sh.col[buf][p]);
      double2 f[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r) f[r] = tr + 32 * r == p ? make_double2(-1.0, 0.0) : sh.col[buf][tr + 32 * r];
      __syncthreads();
      double2 rv[CB];
#pragma unroll
      for (int c = 0; c < CB; ++c) rv[c] = cmul(sh.row[buf][tc + 16 * c], pinv);
      if (tc == kk) rv[b] = pinv;
#pragma unroll
      for (int r = 0; r < RA; ++r)
#pragma unroll
        for (int c = 0; c < CB; ++c) x[r][c] = cfms(x[r][c], f[r], rv[c]);
    }
  }
  __syncthreads();
  return bad;
}

// Element (i, j) of the result goes to row krow[i] and column prow[j]; a singular or non-finite matrix is NaN, so
// that no column of its group converges.
template <int RA, int CB>
__device__ __forceinline__ void gj_store(const double2 (&x)[RA][CB], const GjLds<RA, CB>& sh, double2* P, int n, int ld,
                                         bool bad) {
  const int tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  const double nan = __longlong_as_double(0x7ff8000000000000ll);
#pragma unroll
  for (int r = 0; r < RA; ++r)
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int i = tr + 32 * r, j = tc + 16 * b;
      if (i >= n || j >= n) continue;
      if (bad)
        P[static_cast<size_t>(i) * ld + j] = make_double2(nan, nan);
      else
        P[static_cast<size_t>(sh.krow[i]) * ld + sh.prow[j]] = x[r][b];
    }
}

// A0 of the groups [g0, g0 + groups) and a copy: grid (ceil(n*n/256), groups).
__global__ void __launch_bounds__(256) shared_matrix_kernel(LadderArgs a, const double2* __restrict__ mean,
                                                            const double2* __restrict__ vmean, double2* __restrict__ A0,
                                                            double2* __restrict__ W, int g0) {
  const size_t nn = static_cast<size_t>(a.n) * a.n;
  const size_t e = blockIdx.x * static_cast<size_t>(256) + threadIdx.x;
  if (e >= nn) return;
  const int grp = g0 + blockIdx.y, chan = grp / a.nw, w = grp - chan * a.nw;
  const int i = static_cast<int>(e / a.n), j = static_cast<int>(e - static_cast<size_t>(i) * a.n);
  const int ri = i / a.nv, vi = i - ri * a.nv, cj = j / a.nv, vj = j - cj * a.nv;
  double2 uv = a.u_r[chan * a.T * a.T + ri * a.T + cj];
  if (vmean) uv = cadd(uv, vmean[chan * a.T * a.T + ri * a.T + cj]);
  double2 x = cscale(csub(a.gamma[grp * nn + e], uv), a.inv_beta2);
  if (vi == vj) x = cadd(x, mean[(static_cast<size_t>(w) * a.T * a.T + ri * a.T + cj) * a.nv + vi]);
  A0[blockIdx.y * nn + e] = x;
  W[blockIdx.y * nn + e] = x;
}

// Mean matrices of the groups and their inverses for n <= 32 RA, n <= 16 CB.
template <int RA, int CB>
__global__ void __launch_bounds__(512) shared_invert_kernel(LadderArgs a, const double2* __restrict__ mean,
                                                            const double2* __restrict__ vmean, double2* __restrict__ A0,
                                                            double2* __restrict__ P, int g0) {
  __shared__ GjLds<RA, CB> sh;
  const int n = a.n, T = a.T, nv = a.nv, tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  const int grp = g0 + blockIdx.x, chan = grp / a.nw, w = grp - chan * a.nw;
  const size_t mat = blockIdx.x * static_cast<size_t>(n) * n;
  const double2* G = a.gamma + static_cast<size_t>(grp) * n * n;
  double2 x[RA][CB];
#pragma unroll
  for (int r = 0; r < RA; ++r) {
    const int i = tr + 32 * r, ri = i / nv, vi = i - ri * nv;
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int j = tc + 16 * b, cj = j / nv, vj = j - cj * nv;
      x[r][b] = make_double2(0.0, 0.0);
      if (i < n && j < n) {
        double2 uv = a.u_r[chan * T * T + ri * T + cj];
        if (vmean) uv = cadd(uv, vmean[chan * T * T + ri * T + cj]);
        double2 v = cscale(csub(G[static_cast<size_t>(i) * n + j], uv), a.inv_beta2);
        if (vi == vj) v = cadd(v, mean[(static_cast<size_t>(w) * T * T + ri * T + cj) * nv + vi]);
        x[r][b] = v;
        A0[mat + static_cast<size_t>(i) * n + j] = v;
      }
    }
  }
  const bool bad = gj_invert(x, n, sh);
  gj_store(x, sh, P + mat, n, n, bad);
}

// Blocked form: step kb inverts the diagonal block D = W[k, k] of every group's matrix W.
struct GjArgs {
  double2* W;  // [groups][n][n], in place
  double2* D;  // [groups][64][64] inverse of the diagonal block
  double2* R;  // [groups][64][n] D W[k, :], with D itself in the columns of the block
  double2* C;  // [groups][n][64] -W[:, k]
  int n, groups, tiles, kb;
};

__global__ void __launch_bounds__(512) gj_diag_kernel(GjArgs g) {
  __shared__ GjLds<2, 4> sh;
  const int n = g.n, k0 = g.kb * GJ_NB, nb = min(GJ_NB, n - k0), tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  const double2* W = g.W + (static_cast<size_t>(blockIdx.x) * n + k0) * n + k0;
  double2 x[2][4];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = tr + 32 * r, j = tc + 16 * b;
      x[r][b] = i < nb && j < nb ? W[static_cast<size_t>(i) * n + j] : make_double2(0.0, 0.0);
    }
  const bool bad = gj_invert(x, nb, sh);
  gj_store(x, sh, g.D + static_cast<size_t>(blockIdx.x) * GJ_NB * GJ_NB, nb, GJ_NB, bad);
}

// acc += A B of one 64 x 64 tile with a depth of kn <= 64: A [64][lda] rows below rows, B [kn][ldb] columns
// below cols; what lies beyond reads zero.
__device__ __forceinline__ void gj_product(ZmmaAcc<2, 2>& acc, const double2* __restrict__ A, int lda, int rows,
                                           const double2* __restrict__ B, int ldb, int cols, int kn) {
  __shared__ double2 s_a[GJ_NB][GJ_TK + 1];
  __shared__ double2 s_b[GJ_TK][GJ_NB + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ar = tid / GJ_TK, ak = tid % GJ_TK, bk = tid / GJ_NB, bc = tid % GJ_NB;
  double2 ra[2], rb[2];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = ar + 32 * u, k = k0 + bk + 4 * u;
      ra[u] = r < rows && k0 + ak < kn ? A[static_cast<size_t>(r) * lda + k0 + ak] : make_double2(0.0, 0.0);
      rb[u] = bc < cols && k < kn ? B[static_cast<size_t>(k) * ldb + bc] : make_double2(0.0, 0.0);
    }
  };
  load(0);
  for (int k0 = 0; k0 < kn; k0 += GJ_TK) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s_a[ar + 32 * u][ak] = ra[u];
      s_b[bk + 4 * u][bc] = rb[u];
    }
    __syncthreads();
    if (k0 + GJ_TK < kn) load(k0 + GJ_TK);
    zmma_chunk<2, 2, GJ_NB, GJ_NB, GJ_TK>(acc, s_a, s_b, 32 * (wave >> 1), 32 * (wave & 1), lane);
    __syncthreads();
  }
}

// Row panel R = D W[k, :] and column panel C = -W[:, k]; grid xcd_grid(groups, tiles).
__global__ void __launch_bounds__(256, 3) gj_panel_kernel(GjArgs g) {
  int b, t;
  if (!xcd_tile(blockIdx.x, g.groups, g.tiles, b, t)) return;
  const int n = g.n, k0 = g.kb * GJ_NB, nb = min(GJ_NB, n - k0), c0 = t * GJ_NB, nc = min(GJ_NB, n - c0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double2* W = g.W + static_cast<size_t>(b) * n * n;
  const double2* D = g.D + static_cast<size_t>(b) * GJ_NB * GJ_NB;
  double2* R = g.R + static_cast<size_t>(b) * GJ_NB * n + c0;
  double2* C = g.C + (static_cast<size_t>(b) * n + c0) * GJ_NB;
  for (int e = tid; e < nc * GJ_NB; e += 256) {
    const int i = e / GJ_NB, j = e % GJ_NB;
    if (j < nb) {
      const double2 x = W[static_cast<size_t>(c0 + i) * n + k0 + j];
      C[static_cast<size_t>(i) * GJ_NB + j] = make_double2(-x.x, -x.y);
    }
  }
  if (t == g.kb) {
    for (int e = tid; e < nb * GJ_NB; e += 256) {
      const int i = e / GJ_NB, j = e % GJ_NB;
      if (j < nb) R[static_cast<size_t>(i) * n + j] = D[i * GJ_NB + j];
    }
    return;
  }
  ZmmaAcc<2, 2> acc;
  zmma_zero(acc);
  gj_product(acc, D, GJ_NB, nb, W + static_cast<size_t>(k0) * n + c0, n, nc, nb);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int r = 32 * (wave >> 1) + 16 * i + zmma_row(lane, r4), c = 32 * (wave & 1) + 16 * j + (lane & 15);
        if (r < nb && c < nc) R[static_cast<size_t>(r) * n + c] = zmma_value(acc, i, j, r4);
      }
}

// W[i, j] = (j in the block ? 0 : W[i, j]) + C[i] R[:, j] for the rows outside the block, R for those
// inside; grid xcd_grid(groups, tiles^2). Bound by the FP64 matrix cores (a depth of 64 against one
// read and one write of the tile).
__global__ void __launch_bounds__(256, 3) gj_update_kernel(GjArgs g) {
  int b, t;
  if (!xcd_tile(blockIdx.x, g.groups, g.tiles * g.tiles, b, t)) return;
  const int tm = t / g.tiles, tn = t - tm * g.tiles;
  const int n = g.n, nb = min(GJ_NB, n - g.kb * GJ_NB), r0 = tm * GJ_NB, c0 = tn * GJ_NB;
  const int nr = min(GJ_NB, n - r0), nc = min(GJ_NB, n - c0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double2* W = g.W + (static_cast<size_t>(b) * n + r0) * n + c0;
  const double2* R = g.R + static_cast<size_t>(b) * GJ_NB * n + c0;
  if (tm == g.kb) {
    for (int e = tid; e < nr * GJ_NB; e += 256) {
      const int i = e / GJ_NB, j = e % GJ_NB;
      if (j < nc) W[static_cast<size_t>(i) * n + j] = R[static_cast<size_t>(i) * n + j];
    }
    return;
  }
  ZmmaAcc<2, 2> acc;
  zmma_zero(acc);
  const int wr = 32 * (wave >> 1) + (lane >> 4), wc = 32 * (wave & 1) + (lane & 15);
  if (tn != g.kb) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int r = wr + 16 * i + 4 * r4, c = wc + 16 * j;
          if (r < nr && c < nc) {
            const double2 x = W[static_cast<size_t>(r) * n + c];
            acc.re[i][j][r4] = x.x;
            acc.im[i][j][r4] = x.y;
          }
        }
  }
  gj_product(acc, g.C + (static_cast<size_t>(b) * n + r0) * GJ_NB, GJ_NB, nr, R, n, nc, nb);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int r = wr + 16 * i + 4 * r4, c = wc + 16 * j;
        if (r < nr && c < nc) W[static_cast<size_t>(r) * n + c] = zmma_value(acc, i, j, r4);
      }
}

size_t shared_inverse_workspace(int n) {
  return n <= SHARED_SMALL_N ? 0 : static_cast<size_t>(GJ_NB) * (2 * n + GJ_NB);
}

int shared_inverse(const SharedGroups& s, const double2* mean, const double2* vmean, double2* A0, double2* P,
                   double2* work, hipStream_t stream) {
  const int n = s.a.n;
  if (n <= SHARED_SMALL_N) {
    const dim3 gd(s.groups), bd(512);
    if (n <= 64)
      hipLaunchKernelGGL((shared_invert_kernel<2, 4>), gd, bd, 0, stream, s.a, mean, vmean, A0, P, s.group0);
    else
      hipLaunchKernelGGL((shared_invert_kernel<4, 8>), gd, bd, 0, stream, s.a, mean, vmean, A0, P, s.group0);
    DGAMI_HIP_CHECK(hipGetLastError());
    return 0;
  }
  const size_t nn = static_cast<size_t>(n) * n;
  hipLaunchKernelGGL(shared_matrix_kernel, dim3(ceil_div(nn, 256), s.groups), dim3(256), 0, stream, s.a, mean, vmean, A0, P,
                     s.group0);
  DGAMI_HIP_CHECK(hipGetLastError());
  GjArgs g;
  g.W = P;
  g.D = work;
  g.R = g.D + static_cast<size_t>(s.groups) * GJ_NB * GJ_NB;
  g.C = g.R + static_cast<size_t>(s.groups) * GJ_NB * n;
  g.n = n;
  g.groups = s.groups;
  g.tiles = static_cast<int>(ceil_div(n, GJ_NB));
  const size_t gp = xcd_grid(s.groups, g.tiles), gu = gp * g.tiles;
  DGAMI_ARG_CHECK(gu < (size_t(1) << 31), "ladder: too many groups in one batch");
  for (g.kb = 0; g.kb < g.tiles; ++g.kb) {
    hipLaunchKernelGGL(gj_diag_kernel, dim3(s.groups), dim3(512), 0, stream, g);
    DGAMI_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(gj_panel_kernel, dim3(static_cast<unsigned>(gp)), dim3(256), 0, stream, g);
    DGAMI_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(gj_update_kernel, dim3(static_cast<unsigned>(gu)), dim3(256), 0, stream, g);
    DGAMI_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

}  // namespace dgami
