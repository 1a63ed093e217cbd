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

// ---------------------------------------------------------------------------
// The same product on the BF16 matrix cores: every float x = hi + lo with hi = bf16(x), lo = bf16(x - hi), and
// a b ~ hi hi + hi lo + lo hi with FP32 accumulation (relative error about 2^-16 per product). A is split
// once, into planes [batch][4][M][lda] of re hi, re lo, im hi, im lo with lda a multiple of CB_TK and zeros from
// K on (16-byte aligned); B is split when it is staged. Operand layout of the 16x16x32 BF16 form
// (lane l): a[i] = A[l%16][8 (l/16) + i], b[i] = B[8 (l/16) + i][l%16], d[e] = D[4 (l/16) + e][l%16]; both
// operands lie along k in LDS, rows 40 apart, so that 16 lanes read 16 different bank groups.
// Bound by LDS and the staging rather than by the matrix cores (192 of 1536 cycles of the FP32 form).
// 62 products of 720 x 819 x 720: 1.59 ms in the FP32 form, 0.75 here.
// ---------------------------------------------------------------------------
constexpr int CB_TK = 32;

struct CgemmBf16Args {
  const __bf16* A;
  const float2* B;
  float2* C;
  int M, N, K;
  int lda, ldb, ldc;
  long long sb, sc;
  const int* tile_active = nullptr;
};

// Planes of complex128 matrices [batch][n][n]; grid (ceil(n lda / 256), batch).
static __global__ void __launch_bounds__(256) cgemm_split_kernel(const double2* __restrict__ in, __bf16* __restrict__ out,
                                                                 int n, int lda) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= n * lda) return;
  const int r = e / lda, k = e - r * lda;
  const double2 x = k < n ? in[(static_cast<size_t>(blockIdx.y) * n + r) * n + k] : make_double2(0.0, 0.0);
  const size_t plane = static_cast<size_t>(n) * lda;
  __bf16* dst = out + blockIdx.y * 4 * plane + e;
  const float re = static_cast<float>(x.x), im = static_cast<float>(x.y);
  const __bf16 rh = static_cast<__bf16>(re), ih = static_cast<__bf16>(im);
  dst[0] = rh;
  dst[plane] = static_cast<__bf16>(re - static_cast<float>(rh));
  dst[2 * plane] = ih;
  dst[3 * plane] = static_cast<__bf16>(im - static_cast<float>(ih));
}

static __global__ void __launch_bounds__(256, 2) cgemm_bf16x3_kernel(CgemmBf16Args g, int batch, int tiles_n, int tiles_m) {
  typedef float V4 __attribute__((ext_vector_type(4)));
  typedef __bf16 B8 __attribute__((ext_vector_type(8)));
  typedef unsigned U4 __attribute__((ext_vector_type(4)));
  constexpr int MI = 4, NJ = 2, LD = CB_TK + 8;
  int b, t;
  if (!xcd_tile(blockIdx.x, batch, tiles_m * tiles_n, b, t)) return;
  const int tm = t / tiles_n, tn = t - tm * tiles_n;
  if (g.tile_active && g.tile_active[b * tiles_n + tn] == 0) return;
  const int m0 = tm * CG_TM, n0 = tn * CG_TN;
  __shared__ __attribute__((aligned(16))) __bf16 s_a[4][CG_TM][LD];
  __shared__ __attribute__((aligned(16))) __bf16 s_b[4][CG_TN][LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = 64 * (wave >> 1), wn = 32 * (wave & 1), l16 = lane & 15, kg = lane >> 4;
  // thread: of A 16 k of one row in every plane, of B 8 k of one column
  const int ar = tid >> 1, ak = (tid & 1) * 16, bc = tid & 63, bk = (tid >> 6) * 8;
  const size_t plane = static_cast<size_t>(g.M) * g.lda;
  const __bf16* A = g.A + b * 4 * plane + static_cast<size_t>(min(m0 + ar, g.M - 1)) * g.lda + ak;
  const float2* B = g.B + b * g.sb + min(n0 + bc, g.N - 1);
  V4 cr[MI][NJ], ci[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) cr[i][j] = ci[i][j] = V4{0.f, 0.f, 0.f, 0.f};
  U4 ra[4][2];
  float2 rb[8];
  auto load = [&](int k0) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int u = 0; u < 2; ++u) ra[p][u] = *reinterpret_cast<const U4*>(A + p * plane + k0 + 8 * u);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 + bk + u;
      const float2 x = B[static_cast<size_t>(min(k, g.K - 1)) * g.ldb];
      rb[u] = k < g.K ? make_float2(x.x, x.y) : make_float2(0.f, 0.f);
    }
  };
  load(0);
  for (int k0 = 0; k0 < g.K; k0 += CB_TK) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int u = 0; u < 2; ++u) *reinterpret_cast<U4*>(&s_a[p][ar][ak + 8 * u]) = ra[p][u];
    B8 sp[4];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const __bf16 rh = static_cast<__bf16>(rb[u].x), ih = static_cast<__bf16>(rb[u].y);
      sp[0][u] = rh;
      sp[1][u] = static_cast<__bf16>(rb[u].x - static_cast<float>(rh));
      sp[2][u] = ih;
      sp[3][u] = static_cast<__bf16>(rb[u].y - static_cast<float>(ih));
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) *reinterpret_cast<B8*>(&s_b[p][bc][bk]) = sp[p];
    __syncthreads();
    if (k0 + CB_TK < g.K) load(k0 + CB_TK);
    B8 bv[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int p = 0; p < 4; ++p) bv[j][p] = *reinterpret_cast<const B8*>(&s_b[p][wn + 16 * j + l16][8 * kg]);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      B8 av[4], ng[2];
#pragma unroll
      for (int p = 0; p < 4; ++p) av[p] = *reinterpret_cast<const B8*>(&s_a[p][wm + 16 * i + l16][8 * kg]);
#pragma unroll
      for (int p = 0; p < 2; ++p) ng[p] = __builtin_bit_cast(B8, __builtin_bit_cast(U4, av[2 + p]) ^ 0x80008000u);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        // small terms first
        cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[1], bv[j][0], cr[i][j], 0, 0, 0);
        ci[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[1], bv[j][2], ci[i][j], 0, 0, 0);
        cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[0], bv[j][1], cr[i][j], 0, 0, 0);
        ci[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[0], bv[j][3], ci[i][j], 0, 0, 0);
        cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ng[1], bv[j][2], cr[i][j], 0, 0, 0);
        ci[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[3], bv[j][0], ci[i][j], 0, 0, 0);
        cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ng[0], bv[j][3], cr[i][j], 0, 0, 0);
        ci[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[2], bv[j][1], ci[i][j], 0, 0, 0);
        cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[0], bv[j][0], cr[i][j], 0, 0, 0);
        ci[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[0], bv[j][2], ci[i][j], 0, 0, 0);
        cr[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ng[0], bv[j][2], cr[i][j], 0, 0, 0);
        ci[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[2], bv[j][0], ci[i][j], 0, 0, 0);
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
        if (r < g.M && c < g.N) C[static_cast<size_t>(r) * g.ldc + c] = make_float2(cr[i][j][e], ci[i][j][e]);
      }
}

inline int cgemm_split_lda(int n) { return (n + CB_TK - 1) / CB_TK * CB_TK; }

inline int launch_cgemm_bf16x3(const CgemmBf16Args& g, int batch, hipStream_t stream) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0 || batch <= 0) return 0;
  DGAMI_ARG_CHECK(g.lda % CB_TK == 0 && g.lda >= g.K, "cgemm: split operand rows");
  const int tn = ceil_div(g.N, CG_TN), tm = ceil_div(g.M, CG_TM);
  const size_t grid = xcd_grid(batch, static_cast<size_t>(tn) * tm);
  DGAMI_ARG_CHECK(grid < (size_t(1) << 31), "cgemm: grid too large");
  hipLaunchKernelGGL(cgemm_bf16x3_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, g, batch, tn, tm);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // namespace dgami
