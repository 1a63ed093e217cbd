// Complex128 tile products on the FP64 matrix cores (v_mfma_f64_16x16x4_f64).
//
// A wavefront owns MI x NJ blocks of 16 x 16 complex results as separate real and imaginary
// accumulators. Operand layout of the 16x16x4 instruction (lane l): a = A[l%16][l/16],
// b = B[l/16][l%16]; the result differs from the FP32 form: d[r] = D[l/16 + 4 r][l%16]. Each step
// rounds as a chain of FMAs over k, as the vector form does.
//
// Per k-step of 4 a wavefront with 2 x 2 blocks issues 16 matrix instructions of 64 cycles on four
// 16-byte LDS reads, so the matrix cores and not LDS set the pace; the 4x4-per-thread vector-FMA
// tile it replaces read two LDS words per FMA pair and ran at 0.40 of the FP64 peak.
#pragma once

#include "dgami_internal.hpp"

namespace dgami {

typedef double ZmmaV4 __attribute__((ext_vector_type(4)));

// THREE: re, im and sum hold re re, im im and (re + im)(re + im).
template <int MI, int NJ, bool THREE = false>
struct ZmmaAcc {
  ZmmaV4 re[MI][NJ], im[MI][NJ], sum[THREE ? MI : 1][THREE ? NJ : 1];
};

template <int MI, int NJ, bool THREE>
__device__ __forceinline__ void zmma_zero(ZmmaAcc<MI, NJ, THREE>& c) {
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      c.re[i][j] = c.im[i][j] = ZmmaV4{0.0, 0.0, 0.0, 0.0};
      if constexpr (THREE) c.sum[i][j] = ZmmaV4{0.0, 0.0, 0.0, 0.0};
    }
}

// Row within a 16-row block of accumulator element r in this lane.
__device__ __forceinline__ int zmma_row(int lane, int r) { return (lane >> 4) + 4 * r; }

template <int MI, int NJ, bool THREE>
__device__ __forceinline__ double2 zmma_value(const ZmmaAcc<MI, NJ, THREE>& c, int i, int j, int r) {
  if constexpr (THREE)
    return make_double2(c.re[i][j][r] - c.im[i][j][r], c.sum[i][j][r] - c.re[i][j][r] - c.im[i][j][r]);
  else
    return make_double2(c.re[i][j][r], c.im[i][j][r]);
}

// c += A B for one k-step of 4: av[i], bv[j] are this lane's operands A[l%16][l/16] and B[l/16][l%16] of
// row block i and column block j.
template <int MI, int NJ, bool THREE>
__device__ __forceinline__ void zmma_step(ZmmaAcc<MI, NJ, THREE>& c, const double2 (&av)[MI], const double2 (&bv)[NJ]) {
  if constexpr (THREE) {
    double as[MI], bs[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) as[i] = av[i].x + av[i].y;
#pragma unroll
    for (int j = 0; j < NJ; ++j) bs[j] = bv[j].x + bv[j].y;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        c.re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].x, bv[j].x, c.re[i][j], 0, 0, 0);
        c.im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].y, bv[j].y, c.im[i][j], 0, 0, 0);
        c.sum[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[i], bs[j], c.sum[i][j], 0, 0, 0);
      }
  } else {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        c.re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].x, bv[j].x, c.re[i][j], 0, 0, 0);
        c.im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].x, bv[j].y, c.im[i][j], 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const double nai = -av[i].y;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        c.re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai, bv[j].y, c.re[i][j], 0, 0, 0);
        c.im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].y, bv[j].x, c.im[i][j], 0, 0, 0);
      }
    }
  }
}

// c += A B for one chunk of TK (a multiple of 4) staged in LDS: sa[row][k], sb[k][col]; the
// wavefront's blocks start at row wm and column wn.
template <int MI, int NJ, int TM, int TN, int TK, bool THREE>
__device__ __forceinline__ void zmma_chunk(ZmmaAcc<MI, NJ, THREE>& c, const double2 (&sa)[TM][TK + 1],
                                           const double2 (&sb)[TK][TN + 1], int wm, int wn, int lane) {
  const int l16 = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int k = 0; k < TK; k += 4) {
    double2 av[MI], bv[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) av[i] = sa[wm + 16 * i + l16][k + kg];
#pragma unroll
    for (int j = 0; j < NJ; ++j) bv[j] = sb[k + kg][wn + 16 * j + l16];
    zmma_step(c, av, bv);
  }
}

}  // namespace dgami
