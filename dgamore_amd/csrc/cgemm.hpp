// Batched complex64 GEMM on the FP32 matrix cores, C = A B: the products of an iteration in complex64
// whose residuals are formed in FP64 apart. Row-major operands (leading dimensions and batch strides
// in elements).
#pragma once

#include "dgami_internal.hpp"

namespace dgami {

struct CgemmArgs {
  const float2* A;
  const float2* B;
  float2* C;
  int M, N, K;
  int lda, ldb, ldc;
  long long sa, sb, sc;
  const int* tile_active = nullptr;  // [batch][column tiles] or null: tiles of CG_TN columns with 0 are skipped
};

constexpr int CG_TM = 128, CG_TN = 64, CG_TK = 16;

// grid: xcd_grid(batch, tiles_m * tiles_n); block 256 (all tiles of one batch entry on one XCD). A
// wavefront owns 64 x 32 of the tile in blocks of 16 x 16, each a complex product from three real
// ones: (re, im) = (t1 - t2, t3 - t1 - t2) with t1 = re re, t2 = im im, t3 = (re + im)(re + im).
// Operand layout of the 16x16x4 FP32 form (lane l): a = A[l%16][l/16], b = B[l/16][l%16],
// d[e] = D[4 (l/16) + e][l%16]. Rows of B are 80 apart in LDS, so that the two rows that 32 lanes read
// lie 32 banks apart. Edges are clamped (their results are not stored); the last k-chunk is zeroed.
static __global__ void __launch_bounds__(256, 2) cgemm_kernel(CgemmArgs g, int batch, int tiles_n, int tiles_m) {
  typedef float V4 __attribute__((ext_vector_type(4)));
  constexpr int MI = 4, NJ = 2, LA = CG_TM * CG_TK / 256, LB = CG_TK * CG_TN / 256;
  int b, t;
  if (!xcd_tile(blockIdx.x, batch, tiles_m * tiles_n, b, t)) return;
  const int tm = t / tiles_n, tn = t - tm * tiles_n;
  if (g.tile_active && g.tile_active[b * tiles_n + tn] == 0) return;
  const int m0 = tm * CG_TM, n0 = tn * CG_TN;
  __shared__ float2 s_a[CG_TM][CG_TK + 1];
  __shared__ float2 s_b[CG_TK][CG_TN + 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = 64 * (wave >> 1), wn = 32 * (wave & 1), l16 = lane & 15, kg = lane >> 4;
  // thread: elements (ar + 16 u, ak) of the A chunk and (bk + 4 u, bc) of the B chunk
  const int ar = tid / CG_TK, ak = tid % CG_TK, bk = tid / CG_TN, bc = tid % CG_TN;
  const float2* A[LA];
#pragma unroll
  for (int u = 0; u < LA; ++u) A[u] = g.A + b * g.sa + static_cast<size_t>(min(m0 + ar + 16 * u, g.M - 1)) * g.lda + ak;
  const float2* B = g.B + b * g.sb + static_cast<size_t>(bk) * g.ldb + min(n0 + bc, g.N - 1);
  V4 t1[MI][NJ], t2[MI][NJ], t3[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) t1[i][j] = t2[i][j] = t3[i][j] = V4{0.f, 0.f, 0.f, 0.f};
  float2 ra[LA], rb[LB];
  auto load = [&](int k0) {
    if (k0 + CG_TK <= g.K) {
#pragma unroll
      for (int u = 0; u < LA; ++u) ra[u] = A[u][k0];
#pragma unroll
      for (int u = 0; u < LB; ++u) rb[u] = B[static_cast<size_t>(k0 + 4 * u) * g.ldb];
    } else {
#pragma unroll
      for (int u = 0; u < LA; ++u) ra[u] = k0 + ak < g.K ? A[u][k0] : make_float2(0.f, 0.f);
#pragma unroll
      for (int u = 0; u < LB; ++u)
        rb[u] = k0 + bk + 4 * u < g.K ? B[static_cast<size_t>(k0 + 4 * u) * g.ldb] : make_float2(0.f, 0.f);
    }
  };
  load(0);
  for (int k0 = 0; k0 < g.K; k0 += CG_TK) {
#pragma unroll
    for (int u = 0; u < LA; ++u) s_a[ar + 16 * u][ak] = ra[u];
#pragma unroll
    for (int u = 0; u < LB; ++u) s_b[bk + 4 * u][bc] = rb[u];
    __syncthreads();
    if (k0 + CG_TK < g.K) load(k0 + CG_TK);
#pragma unroll
    for (int k = 0; k < CG_TK; k += 4) {
      float2 av[MI], bv[NJ];
      float as[MI], bs[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        av[i] = s_a[wm + 16 * i + l16][k + kg];
        as[i] = av[i].x + av[i].y;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        bv[j] = s_b[k + kg][wn + 16 * j + l16];
        bs[j] = bv[j].x + bv[j].y;
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          t1[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i].x, bv[j].x, t1[i][j], 0, 0, 0);
          t2[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i].y, bv[j].y, t2[i][j], 0, 0, 0);
          t3[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(as[i], bs[j], t3[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  }
  float2* C = g.C + b * g.sc;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = m0 + wm + 16 * i + 4 * kg + e, c = n0 + wn + 16 * j + l16;
        if (r < g.M && c < g.N)
          C[static_cast<size_t>(r) * g.ldc + c] =
              make_float2(t1[i][j][e] - t2[i][j][e], t3[i][j][e] - t1[i][j][e] - t2[i][j][e]);
      }
}

inline int launch_cgemm(const CgemmArgs& g, int batch, hipStream_t stream) {
  if (g.M <= 0 || g.N <= 0 || batch <= 0) return 0;
  const int tn = ceil_div(g.N, CG_TN), tm = ceil_div(g.M, CG_TM);
  const size_t grid = xcd_grid(batch, static_cast<size_t>(tn) * tm);
  DGAMI_ARG_CHECK(grid < (size_t(1) << 31), "cgemm: grid too large");
  hipLaunchKernelGGL(cgemm_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, g, batch, tn, tm);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace dgami
