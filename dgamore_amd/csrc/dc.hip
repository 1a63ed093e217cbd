// Double-counting kernel of the self-energy (nonlocal_sde.py:185-198, with the
// caller's prefactors at :817-820): for every bosonic frequency w one complex
// GEMM with rows ((fe), v'), contraction ((dc), v) and columns ((ab), q):
//   L[w][((dc),v)][(ab,q)]   = (M(u') M(chi0(q,w,v)))[(ab),(dc)],  u'_abij = u_ajib
//   R[w][((dc),v)][((fe),v')] = (1/beta^2) f_dc_dcef(w,v,v') = (2/beta^2) F_magn,loc[e][c][d][f][w][v][v']
//   kernel[w][(ab),(fe)][v'][q] = -(R^T L)[((fe),v')][(ab,q)],  v' cut to the core box.
// With q as the column of the product its result has the kernel's own order (q fastest) and L that of
// chi0; with q as the row both were transposed through memory (64x64, one orbital, 561 q, 61 w, box
// 120: 56 us for the result and 46 us for L beside the 89 us of the product). With one orbital M(u') is a
// number: R takes it and chi0 itself is the operand.
#include "dgami.h"
#include "dgami_internal.hpp"
#include "dgami_launch.hpp"
#include "zgemm.hpp"

namespace dgami {

// L operand: thread per (w, (dc), v, q), all (ab); chi0 is read and L written along q. The elements of u
// are the same for all threads.
template <int NB>
__global__ void __launch_bounds__(256) dc_left_kernel(const double2* __restrict__ chi0, const double2* __restrict__ u,
                                                      double2* __restrict__ L, int nq, int nw, int nvf) {
  constexpr int T = NB * NB;
  const size_t total = static_cast<size_t>(nw) * T * nvf * nq;
  for (size_t idx = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const int q = static_cast<int>(idx % nq);
    const size_t kv = idx / nq;  // (w, (dc), v)
    const int v = static_cast<int>(kv % nvf);
    const int dc = static_cast<int>(kv / nvf % T);
    const int w = static_cast<int>(kv / nvf / T);
    double2 x[T];
#pragma unroll
    for (int ji = 0; ji < T; ++ji) x[ji] = chi0[((static_cast<size_t>(w) * T * T + ji * T + dc) * nvf + v) * nq + q];
    double2* dst = L + kv * T * nq + q;
#pragma unroll 1
    for (int ab = 0; ab < T; ++ab) {  // (unrolled, the elements of u do not fit the scalar registers)
      double2 acc = make_double2(0.0, 0.0);
      // M(u')[(ab),(ji)] = u'_{a b i j} = u_{a j i b} (reference order)
#pragma unroll
      for (int ji = 0; ji < T; ++ji)
        acc = cfma(acc, u[((ab / NB * NB + ji / NB) * NB + ji % NB) * NB + ab % NB], x[ji]);
      dst[static_cast<size_t>(ab) * nq] = acc;
    }
  }
}

// The same for more orbitals than a thread holds: thread per (w, (dc), v, (ab), q).
__global__ void __launch_bounds__(256) dc_left_any_kernel(const double2* __restrict__ chi0,
                                                          const double2* __restrict__ u, double2* __restrict__ L, int nq,
                                                          int nb, int nw, int nvf) {
  const int T = nb * nb;
  const size_t total = static_cast<size_t>(nw) * T * nvf * T * nq;
  for (size_t idx = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * blockDim.x) {
    size_t r = idx;
    const int q = static_cast<int>(r % nq);
    r /= nq;
    const int ab = static_cast<int>(r % T);
    r /= T;
    const int v = static_cast<int>(r % nvf);
    r /= nvf;
    const int dc = static_cast<int>(r % T);
    const int w = static_cast<int>(r / T);
    double2 acc = make_double2(0.0, 0.0);
    for (int ji = 0; ji < T; ++ji)
      acc = cfma(acc, u[((ab / nb * nb + ji / nb) * nb + ji % nb) * nb + ab % nb],
                 chi0[((static_cast<size_t>(w) * T * T + ji * T + dc) * nvf + v) * nq + q]);
    L[idx] = acc;
  }
}

// R operand: thread per (w, (dc), v, (fe), v'); scaled by `scale`, and by u with one orbital.
__global__ void dc_right_kernel(const double2* __restrict__ f, const double2* __restrict__ u, double2* __restrict__ R,
                                int nb, int nw, int nvf, int nvc, int p0, double scale) {
  const int T = nb * nb;
  const size_t total = static_cast<size_t>(nw) * T * nvf * T * nvc;
  const double2 u0 = cscale(nb == 1 ? u[0] : make_double2(1.0, 0.0), scale);
  for (size_t idx = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; idx < total;
       idx += static_cast<size_t>(gridDim.x) * blockDim.x) {
    size_t r = idx;
    const int p = static_cast<int>(r % nvc);
    r /= nvc;
    const int fe = static_cast<int>(r % T);
    r /= T;
    const int v = static_cast<int>(r % nvf);
    r /= nvf;
    const int dc = static_cast<int>(r % T);
    const int w = static_cast<int>(r / T);
    const int d = dc / nb, c = dc % nb, ff = fe / nb, e = fe % nb;
    const size_t src = ((((static_cast<size_t>(e) * nb + c) * nb + d) * nb + ff) * nw + w) * nvf * nvf +
                       static_cast<size_t>(v) * nvf + p0 + p;
    R[idx] = cmul(u0, f[src]);
  }
}

}  // namespace dgami

extern "C" int dgami_dc_kernel(int nq, int nb, int nw, int niv_full, int niv_core, double beta, const dgami_c128* chi0,
                               const dgami_c128* u, const dgami_c128* f_magn_loc, dgami_c128* kernel, void* stream_) {
  using namespace dgami;
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  DGAMI_ARG_CHECK(chi0 && u && f_magn_loc && kernel, "dc_kernel: null pointer");
  DGAMI_ARG_CHECK(nq >= 1 && nb >= 1 && nw >= 1 && niv_core >= 1 && niv_full >= niv_core && beta > 0,
                  "dc_kernel: invalid sizes");
  const int T = nb * nb, nvf = 2 * niv_full, nvc = 2 * niv_core;
  const size_t lsz = nb == 1 ? 0 : static_cast<size_t>(nw) * nq * T * T * nvf;
  const size_t rsz = static_cast<size_t>(nw) * T * nvf * T * nvc;
  double2* ws = static_cast<double2*>(workspace(WS_DC, (lsz + rsz) * sizeof(double2)));
  if (!ws) return -2;
  double2 *L = ws, *R = ws + lsz;
  const double2* x = reinterpret_cast<const double2*>(chi0);
  const double2* du = reinterpret_cast<const double2*>(u);
  auto blocks = [](size_t total) { return ceil_div(total, 256) > 262144u ? 262144u : ceil_div(total, 256); };
  const dim3 gl(blocks(lsz / T));
  switch (nb) {
    case 1: break;
    case 2: hipLaunchKernelGGL(dc_left_kernel<2>, gl, dim3(256), 0, stream, x, du, L, nq, nw, nvf); break;
    case 3: hipLaunchKernelGGL(dc_left_kernel<3>, gl, dim3(256), 0, stream, x, du, L, nq, nw, nvf); break;
    case 4: hipLaunchKernelGGL(dc_left_kernel<4>, gl, dim3(256), 0, stream, x, du, L, nq, nw, nvf); break;
    default:
      hipLaunchKernelGGL(dc_left_any_kernel, dim3(blocks(lsz)), dim3(256), 0, stream, x, du, L, nq, nb, nw, nvf);
      break;
  }
  DGAMI_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(dc_right_kernel, dim3(blocks(rsz)), dim3(256), 0, stream,
                     reinterpret_cast<const double2*>(f_magn_loc), du, R, nb, nw, nvf, nvc, niv_full - niv_core,
                     2.0 / (beta * beta));
  DGAMI_HIP_CHECK(hipGetLastError());
  ZgemmArgs g;
  g.A = R;
  g.B = nb == 1 ? x : L;
  g.C = reinterpret_cast<double2*>(kernel);
  g.M = T * nvc;
  g.K = T * nvf;
  g.N = T * nq;
  g.lda = g.M;
  g.ldb = g.N;
  g.ldc = nq;
  g.cgroup = nq;
  g.sgroup = static_cast<long long>(g.M) * nq;
  g.sa = static_cast<long long>(g.K) * g.M;
  g.sb = static_cast<long long>(g.K) * g.N;
  g.sc = static_cast<long long>(g.M) * g.N;
  g.alpha = make_double2(-1.0, 0.0);
  g.beta = make_double2(0.0, 0.0);
  return launch_zgemm<false, true>(g, nw, stream);
}
