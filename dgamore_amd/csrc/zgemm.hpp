// Batched complex128 GEMM on LDS tiles and the FP64 matrix cores, C = alpha A B + beta C.
// Row-major operands with leading dimensions and batch strides (elements); A may be stored transposed
// ([K][M]), and the columns of C may lie in groups of their own stride.
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
  int cgroup = 0;  // > 0: column c of C is at (c / cgroup) * sgroup + c % cgroup
  long long sgroup = 0;
  const int* tile_active = nullptr;  // [batch][column tiles] or null: tiles of ZG_TN columns with 0 are skipped
};

constexpr int ZG_TM = 64, ZG_TN = 64, ZG_TK = 8;
static_assert(ZG_TM * ZG_TK == 2 * 256 && ZG_TK * ZG_TN == 2 * 256, "two operand elements per thread");

// grid: xcd_grid(batch, tiles_m * tiles_n); block 256 (all tiles of one batch entry on one XCD). Each
// wavefront owns a 32 x 32 quarter of the tile. Bound by the FP64 matrix cores (zmma.hpp). Rows and
// columns past the edge are clamped, not predicated (their results are not stored; a per-load
// predicate cost 8%), and only the last k-chunk zeroes its tail. Measured on 62 products of 768 x 832
// x 768: chunks of 8 at three workgroups per CU 3.76 ms (64.8 TF/s), of 16 3.84, of 32 3.93; the
// vector-FMA tile ran at 32 TF/s.
// THREE: complex products from three real ones, (re, im) = (t1 - t2, t3 - t1 - t2) with t1 = re re,
// t2 = im im, t3 = (re + im)(re + im): a quarter fewer matrix instructions (3.12 ms), with an error
// bounded by |A| |B| instead of per part (for the products of an iteration whose residual is formed
// apart). Chunks of 16 left it one workgroup per CU (4.22 ms).
// TRANS: A is stored [K][M]; a chunk is then read along M.
template <bool THREE, bool TRANS>
static __global__ void __launch_bounds__(256, THREE ? 2 : 3) zgemm_kernel(ZgemmArgs g, int batch, int tiles_n, int tiles_m) {
  int b, t;
  if (!xcd_tile(blockIdx.x, batch, tiles_m * tiles_n, b, t)) return;
  if (g.active && g.active[b] == 0) return;
  const int tm = t / tiles_n, tn = t - (t / tiles_n) * tiles_n;
  if (g.tile_active && g.tile_active[b * tiles_n + tn] == 0) return;
  const int m0 = tm * ZG_TM, n0 = tn * ZG_TN;
  __shared__ double2 s_a[ZG_TM][ZG_TK + 1];
  __shared__ double2 s_b[ZG_TK][ZG_TN + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = 32 * (wave >> 1), wn = 32 * (wave & 1);
  // thread: element (ar + 32 u, ak) of the A chunk (TRANS: (ar, ak + 4 u)) and (bk + 4 u, bc) of the B chunk
  const int ar = TRANS ? tid % ZG_TM : tid / ZG_TK, ak = TRANS ? tid / ZG_TM : tid % ZG_TK;
  const int bk = tid / ZG_TN, bc = tid % ZG_TN;
  constexpr int DR = TRANS ? 0 : 32, DK = TRANS ? 4 : 0;
  const size_t da = TRANS ? g.lda : 1;  // from one k of A to the next
  const double2* A[2];
  const double2* B = g.B + b * g.sb + static_cast<size_t>(bk) * g.ldb + min(n0 + bc, g.N - 1);
#pragma unroll
  for (int u = 0; u < 2; ++u)
    A[u] = g.A + b * g.sa + static_cast<size_t>(min(m0 + ar + DR * u, g.M - 1)) * (TRANS ? 1 : g.lda) + (ak + DK * u) * da;
  ZmmaAcc<2, 2, THREE> acc;
  zmma_zero(acc);
  // the next k-chunk's operands are loaded into registers while the current one is used
  double2 ra[2], rb[2];
  auto load = [&](int k0) {
    if (k0 + ZG_TK <= g.K) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        ra[u] = A[u][k0 * da];
        rb[u] = B[static_cast<size_t>(k0 + 4 * u) * g.ldb];
      }
    } else {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        ra[u] = k0 + ak + DK * u < g.K ? A[u][k0 * da] : make_double2(0.0, 0.0);
        rb[u] = k0 + bk + 4 * u < g.K ? B[static_cast<size_t>(k0 + 4 * u) * g.ldb] : make_double2(0.0, 0.0);
      }
    }
  };
  load(0);
  for (int k0 = 0; k0 < g.K; k0 += ZG_TK) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s_a[ar + DR * u][ak + DK * u] = ra[u];
      s_b[bk + 4 * u][bc] = rb[u];
    }
    __syncthreads();
    if (k0 + ZG_TK < g.K) load(k0 + ZG_TK);
    zmma_chunk<2, 2, ZG_TM, ZG_TN, ZG_TK>(acc, s_a, s_b, wm, wn, lane);
    __syncthreads();
  }
  double2* C = g.C + b * g.sc;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const int r = m0 + wm + 16 * i + zmma_row(lane, r4), c = n0 + wn + 16 * j + (lane & 15);
        if (r >= g.M || c >= g.N) continue;
        double2* e = C + static_cast<size_t>(r) * g.ldc;
        e += g.cgroup > 0 ? c / g.cgroup * g.sgroup + c % g.cgroup : c;
        double2 val = cmul(g.alpha, zmma_value(acc, i, j, r4));
        if (g.beta.x != 0.0 || g.beta.y != 0.0) val = cfma(val, g.beta, *e);
        *e = val;
      }
}

template <bool THREE = false, bool TRANS = false>
inline int launch_zgemm(const ZgemmArgs& g, int batch, hipStream_t stream) {
  if (g.M <= 0 || g.N <= 0 || batch <= 0) return 0;
  const int tn = ceil_div(g.N, ZG_TN), tm = ceil_div(g.M, ZG_TM);
  const size_t grid = xcd_grid(batch, static_cast<size_t>(tn) * tm);
  DGAMI_ARG_CHECK(grid < (size_t(1) << 31), "zgemm: grid too large");
  hipLaunchKernelGGL((zgemm_kernel<THREE, TRANS>), dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, g, batch, tn, tm);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace dgami
