// Batched complex128 GEMM on LDS tiles and the FP64 matrix cores, C = alpha A B + beta C.
// Row-major operands with leading dimensions and batch strides (elements).
#pragma once

#include "dgami_internal.hpp"
#include "zmma.hpp"

namespace dgami {

struct ZgemmArgs {
  const double2* A;
  const double2* B;
  double2* C;
  int M, N, K;
  int lda, ldb, ldc;
  long long sa, sb, sc;  // batch strides
  double2 alpha, beta;
  const int* active = nullptr;  // [batch] or null: batch entries with active[b] == 0 are skipped
};

constexpr int ZG_TM = 64, ZG_TN = 64, ZG_TK = 16;
static_assert(ZG_TM * ZG_TK == 4 * 256 && ZG_TK * ZG_TN == 4 * 256, "four operand elements per thread");

// grid: xcd_grid(batch, tiles_m * tiles_n); block 256 (all tiles of one batch entry on one XCD). Each
// wavefront owns a 32 x 32 quarter of the tile. Bound by the FP64 matrix cores (zmma.hpp): the
// refinement's residual products 4.90 -> 3.85 ms, the double-counting product 2.5 -> 2.0 ms.
static __global__ void __launch_bounds__(256) zgemm_kernel(ZgemmArgs g, int batch, int tiles_n, int tiles_m) {
  int b, t;
  if (!xcd_tile(blockIdx.x, batch, tiles_m * tiles_n, b, t)) return;
  if (g.active && g.active[b] == 0) return;
  const double2* A = g.A + b * g.sa;
  const double2* B = g.B + b * g.sb;
  double2* C = g.C + b * g.sc;
  const int tm = t / tiles_n, tn = t - (t / tiles_n) * tiles_n;
  const int m0 = tm * ZG_TM, n0 = tn * ZG_TN;
  __shared__ double2 s_a[ZG_TM][ZG_TK + 1];
  __shared__ double2 s_b[ZG_TK][ZG_TN + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = 32 * (wave >> 1), wn = 32 * (wave & 1);
  ZmmaAcc<2, 2> acc;
  zmma_zero(acc);
  // the next k-tile's operands are loaded into registers while the current one is used
  double2 ra[4], rb[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + 256 * u;
      const int r = e / ZG_TK, s = e % ZG_TK;
      ra[u] = (m0 + r < g.M && k0 + s < g.K) ? A[static_cast<size_t>(m0 + r) * g.lda + k0 + s]
                                              : make_double2(0.0, 0.0);
      const int s2 = e / ZG_TN, c = e % ZG_TN;
      rb[u] = (k0 + s2 < g.K && n0 + c < g.N) ? B[static_cast<size_t>(k0 + s2) * g.ldb + n0 + c]
                                               : make_double2(0.0, 0.0);
    }
  };
  load(0);
  for (int k0 = 0; k0 < g.K; k0 += ZG_TK) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = tid + 256 * u;
      s_a[e / ZG_TK][e % ZG_TK] = ra[u];
      s_b[e / ZG_TN][e % ZG_TN] = rb[u];
    }
    __syncthreads();
    if (k0 + ZG_TK < g.K) load(k0 + ZG_TK);
    zmma_chunk<2, 2, ZG_TM, ZG_TN, ZG_TK>(acc, s_a, s_b, wm, wn, lane);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int r = m0 + wm + 16 * i + zmma_row(lane, r4), c = n0 + wn + 16 * j + (lane & 15);
        if (r >= g.M || c >= g.N) continue;
        double2* e = C + static_cast<size_t>(r) * g.ldc + c;
        double2 val = cmul(g.alpha, make_double2(acc.re[i][j][r4], acc.im[i][j][r4]));
        if (g.beta.x != 0.0 || g.beta.y != 0.0) val = cfma(val, g.beta, *e);
        *e = val;
      }
}

inline int launch_zgemm(const ZgemmArgs& g, int batch, hipStream_t stream) {
  if (g.M <= 0 || g.N <= 0 || batch <= 0) return 0;
  const int tn = ceil_div(g.N, ZG_TN), tm = ceil_div(g.M, ZG_TM);
  const size_t grid = xcd_grid(batch, static_cast<size_t>(tn) * tm);
  DGAMI_ARG_CHECK(grid < (size_t(1) << 31), "zgemm: grid too large");
  hipLaunchKernelGGL(zgemm_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, g, batch, tn, tm);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace dgami
