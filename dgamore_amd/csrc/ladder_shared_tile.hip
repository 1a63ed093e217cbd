// Ladder sums through the groups' shared matrix (ladder_shared.hip) for compound sizes up to 256 of one
// and two orbitals (the LU is faster for more of them at these sizes).
//
// Columns are independent, so one workgroup takes a tile of 16 columns of a group through the whole
// solution (products, orthogonalisation, cycles, output) without any other workgroup: one launch, and
// each tile stops when its own columns have converged. The vector an iteration works on stays in LDS;
// only the Krylov basis goes through memory, and the matrix comes from L2, where the tiles of a group on one XCD
// share it. Bound by the reads of the basis (n = 120: matrix cores 28% busy). With a launch per product
// and per pass, as the large sizes have it, 68442 problems of n = 120 took 7.4 ms (now 3.5) and 1872
// problems of n = 216 4.8 ms (now 2.4), most of it gaps between about 250 launches.
#include <algorithm>

#include "dgami.h"
#include "dgami_internal.hpp"
#include "ladder_common.hpp"
#include "ladder_shared.hpp"
#include "zmma.hpp"

namespace dgami {

// Shape of a tile kernel: T = nb^2, NW wavefronts that share the rows of a product (16 MI each), and sweeps of
// JB basis vectors in the orthogonalisation.
template <int T_, int NW_, int MI_>
struct SharedShape {
  static constexpr int T = T_, NC = 16, NW = NW_, TH = 64 * NW_, RG = TH / NC;
  static constexpr int MI = MI_;
  static constexpr int PF = MI == 1 ? 4 : 2;  // k-steps that a product loads ahead
  static constexpr int JB = 4;
  static constexpr int RB = MI == 1 ? 4 : 8;  // rows of a thread at a time
};

struct SharedTileArgs {
  SharedGroups s;
  const double2* A0;  // packed (shared_packed)
  const double2* P;
  int ntile;          // tiles of a group
  double2* vec;       // [workgroups][SH_M + 2][rows][NC]: basis and X
  int* next;          // [NUM_XCD] next tile of the groups of an XCD
};

// A tile's state in LDS. `red` is used between barriers by every reduction.
template <typename H>
struct SharedLds {
  double2 red[H::NW][H::JB + 1][H::NC];
  double2 R[SH_ROT][H::NC];     // triangular factor, column j at j (j + 1) / 2
  double2 h[SH_M + 1][H::NC];   // projections of the current vector; at the end of a cycle the coefficients of X
  double2 rs[SH_M][H::NC];      // rotations
  double2 gv[SH_M + 1][H::NC];  // rotated residual
  double rc[SH_M][H::NC];
  double2 sums[H::T][H::NC];    // sums over v of the vector D(q) is applied to (V_r term)
  int tile;
};

// A tile as its workgroup's threads see it: thread tid owns column tid % NC and the rows
// i = tid / NC + RG k of every pass over a vector, so that the workgroup reads whole runs.
struct SharedTile {
  int c, rg, q, t;  // column within the tile, row group, q-point and right-hand side
  bool in;
  size_t col;       // column of the batch
  const double2* dd;
  const double2* dv;
};

// The n x n matrices of a group in the order the matrix cores read them: for every 16-row block (an
// even number of them) and every k-step of 4 the 64 lanes' elements M[16 rb + l%16][4 ks + l/16] in
// one 1 KiB run, zero beyond n. Read from the row-major matrix a load touched 16 lines of which it
// used half.
__host__ __device__ inline int shared_blocks(int n) { return 2 * ((n + 31) / 32); }
__host__ __device__ inline int shared_steps(int n) { return (n + 3) / 4; }
size_t shared_packed(int n) { return static_cast<size_t>(shared_blocks(n)) * shared_steps(n) * 64; }

// Both matrices packed, z0 = P B (sums of P over the frequencies of every orbital pair), the tile counters
// cleared, and the look for equal rows. grid (2 ceil(packed / 256) + ceil(n / 4) + 1, groups), n uint4 of LDS.
__global__ void __launch_bounds__(256) shared_pack_kernel(SharedGroups s, double2* __restrict__ out, double2* __restrict__ z0,
                                                          int* __restrict__ next) {
  const int n = s.a.n, T = s.a.T, nv = s.a.nv, nk = shared_steps(n);
  const size_t size = static_cast<size_t>(shared_blocks(n)) * nk * 64;
  const unsigned nb = static_cast<unsigned>((size + 255) / 256);
  const size_t mat = blockIdx.y * static_cast<size_t>(n) * n;
  const int lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < NUM_XCD) next[threadIdx.x] = 0;
  if (blockIdx.x == gridDim.x - 1) {
    extern __shared__ uint4 s_hash[];
    const bool equal = shared_equal_rows(s, blockIdx.y, s_hash);
    if (threadIdx.x == 0) s.equal[blockIdx.y] = equal;
    return;
  }
  if (blockIdx.x < 2 * nb) {
    const bool inv = blockIdx.x >= nb;
    const size_t e = (blockIdx.x - (inv ? nb : 0)) * static_cast<size_t>(256) + threadIdx.x;
    if (e >= size) return;
    const int ks = static_cast<int>((e >> 6) % nk), rb = static_cast<int>((e >> 6) / nk);
    const int r = 16 * rb + (lane & 15), k = 4 * ks + (lane >> 4);
    const double2* M = (inv ? s.P : s.A0) + mat;
    out[((inv ? s.groups : 0) + blockIdx.y) * size + e] =
        r < n && k < n ? M[static_cast<size_t>(r) * n + k] : make_double2(0.0, 0.0);
    return;
  }
  const int row = (blockIdx.x - 2 * nb) * 4 + (threadIdx.x >> 6);
  if (row >= n) return;
  for (int t = 0; t < T; ++t) {
    const double2* src = s.P + mat + static_cast<size_t>(row) * n + t * nv;
    double2 acc = make_double2(0.0, 0.0);
    for (int v = lane; v < nv; v += 64) acc = cadd(acc, src[v]);
    for (int o = 32; o > 0; o >>= 1) acc = cadd(acc, make_double2(__shfl_xor(acc.x, o), __shfl_xor(acc.y, o)));
    if (lane == 0) z0[(blockIdx.y * static_cast<size_t>(n) + row) * T + t] = acc;
  }
}

// B <- A B for the tile in LDS: A packed, B [rows][NC] with zero rows up to a multiple of 4. A wavefront
// owns 16 MI rows; A comes from L2 in the matrix cores' layout, PF k-steps ahead, and B from LDS, so no barrier
// holds a wavefront up until the result takes B's place.
template <typename H, bool THREE>
__device__ __forceinline__ void shared_product(const double2* __restrict__ A, double2* B, int n) {
  constexpr int MI = H::MI, PF = H::PF, NC = H::NC;
  const int lane = threadIdx.x & 63, r0 = 16 * MI * (threadIdx.x >> 6), l16 = lane & 15, kg = lane >> 4;
  const int nk = shared_steps(n);
  ZmmaAcc<MI, 1, THREE> acc;
  zmma_zero(acc);
  if (r0 < n) {
    const double2* Ar = A + static_cast<size_t>(r0 / 16) * nk * 64 + lane;
    const double2* Br = B + kg * NC + l16;
    double2 av[PF][MI], bv[PF][1];
    auto load = [&](int s, int ks) {
      ks = min(ks, nk - 1);
#pragma unroll
      for (int i = 0; i < MI; ++i) av[s][i] = Ar[(i * nk + ks) * 64];
      bv[s][0] = Br[ks * 4 * NC];
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) load(s, s);
    int ks = 0;
    for (; ks + PF <= nk; ks += PF) {
#pragma unroll
      for (int s = 0; s < PF; ++s) {
        zmma_step(acc, av[s], bv[s]);
        load(s, ks + PF + s);
      }
    }
#pragma unroll
    for (int s = 0; s < PF - 1; ++s)
      if (ks + s < nk) zmma_step(acc, av[s], bv[s]);
  }
  __syncthreads();
  if (r0 < n) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = r0 + 16 * i + zmma_row(lane, r);
        if (row < n) B[row * NC + l16] = zmma_value(acc, i, 0, r);
      }
  }
  __syncthreads();
}

// Sums over the row groups of K values per thread; every thread gets its column's sums. The barrier
// of the next reduction (or the caller's) separates the reads from the next writes.
template <typename H, int K>
__device__ __forceinline__ void shared_reduce(SharedLds<H>& sh, double2 (&v)[K], int c) {
  static_assert(K <= H::JB + 1, "reduction buffer");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < K; ++j) {
#pragma unroll
    for (int o = H::NC; o < 64; o *= 2) v[j] = cadd(v[j], make_double2(__shfl_xor(v[j].x, o), __shfl_xor(v[j].y, o)));
  }
  __syncthreads();
  if (lane < H::NC) {
#pragma unroll
    for (int j = 0; j < K; ++j) sh.red[wave][j][lane] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < K; ++j) {
    v[j] = sh.red[0][j][c];
#pragma unroll
    for (int k = 1; k < H::NW; ++k) v[j] = cadd(v[j], sh.red[k][j][c]);
  }
}

// u = D(q) v, or (RESIDUAL) u = B - g - D(q) v with g = A0 v. A thread owns the T rows of its column's
// frequencies, which D(q) couples, so u may take the place of v or g. Bound by the loads of D(q).
template <typename H, bool RESIDUAL>
__device__ __forceinline__ void shared_apply(const SharedGroups& s, SharedLds<H>& sh, const SharedTile& x,
                                             const double2* v, const double2* g, double2* u) {
  constexpr int T = H::T, NC = H::NC;
  const int nv = s.a.nv, nq = s.a.nq;
  if (x.dv) {
#pragma unroll 1
    for (int c = 0; c < T; ++c) {
      double2 sv[1] = {make_double2(0.0, 0.0)};
      for (int vi = x.rg; vi < nv; vi += H::RG) sv[0] = cadd(sv[0], v[(c * nv + vi) * NC + x.c]);
      shared_reduce<H, 1>(sh, sv, x.c);
      if (x.rg == 0) sh.sums[c][x.c] = sv[0];
    }
    __syncthreads();
  }
  constexpr int VU = T == 1 ? 4 : 1;
#pragma unroll VU
  for (int vi = x.rg; vi < nv; vi += H::RG) {
    double2 y[T];
#pragma unroll
    for (int c = 0; c < T; ++c) y[c] = v[(c * nv + vi) * NC + x.c];
    const double2* d = x.dd + static_cast<size_t>(vi) * nq;
    const size_t blk = static_cast<size_t>(nv) * nq;
    constexpr int RU = T == 4 ? 4 : 1;
#pragma unroll RU
    for (int r = 0; r < T; ++r) {
      double2 acc = make_double2(0.0, 0.0);
#pragma unroll
      for (int c = 0; c < T; ++c) acc = cfma(acc, d[(r * T + c) * blk], y[c]);
      if (x.dv) {
#pragma unroll 1
        for (int c = 0; c < T; ++c) acc = cfms(acc, x.dv[r * T + c], sh.sums[c][x.c]);
      }
      const int o = (r * nv + vi) * NC + x.c;
      if constexpr (RESIDUAL) acc = csub(make_double2(r == x.t ? 1.0 : 0.0, 0.0), cadd(g[o], acc));
      u[o] = acc;
    }
  }
}

// The column's Hessenberg matrix (1 + P D(q) projected): the rotations of column k, whose projections are in
// sh.h and whose remainder is hn; returns whether the column goes on, and its residual in res. Called by
// row group 0 for its columns (live: the column iterates).
template <typename H>
__device__ __forceinline__ bool shared_rotate(SharedLds<H>& sh, int col, int k, double hn, bool live, double target,
                                              double& res) {
  if (live) {  // row group 0 only
    const int rk = k * (k + 1) / 2;
    double2 hj = sh.h[0][col];
#pragma unroll 1
    for (int j = 0; j < k; ++j) {
      double2 h1 = sh.h[j + 1][col];
      if (j + 1 == k) h1.x += 1.0;
      const double c = sh.rc[j][col];
      const double2 sn = sh.rs[j][col];
      sh.R[rk + j][col] = cfma(cscale(hj, c), sn, h1);
      hj = cfms(cscale(h1, c), cconj(sn), hj);
    }
    if (k == 0) hj.x += 1.0;
    const double ah = hypot(hj.x, hj.y), r = hypot(ah, hn);
    const double c = r > 0.0 ? ah / r : 1.0;
    const double2 ph = ah > 0.0 ? cscale(hj, 1.0 / ah) : make_double2(1.0, 0.0);
    const double2 sn = cscale(ph, r > 0.0 ? hn / r : 0.0);
    sh.rc[k][col] = c;
    sh.rs[k][col] = sn;
    sh.R[rk + k][col] = cscale(ph, r);
    const double2 gk = sh.gv[k][col];
    const double2 gn = cmul(make_double2(-sn.x, sn.y), gk);
    sh.gv[k][col] = cscale(gk, c);
    sh.gv[k + 1][col] = gn;
    res = hypot(gn.x, gn.y);
    // converged, broken down, or not a number: the column waits for the end of the cycle
    live = res > target && hn > 0.0 && k + 1 < SH_M;
  }
  return live;
}

// Orthogonalisation of w against V_0 .. V_k, and V_(k+1). w = P D(q) V_k itself is orthogonalised, not
// V_k + w, so |w - projection|^2 = |w|^2 - sum |h|^2 cancels little, and V and the Hessenberg matrix stay
// consistent. Bound by the two reads of the basis.
template <typename H>
__device__ __forceinline__ bool shared_step(SharedLds<H>& sh, const SharedTile& x, const double2* V, double2* w,
                                            double2* Vn, int n, int stride, int k, bool live, double target,
                                            double& res) {
  constexpr int RG = H::RG, NC = H::NC, SH_JB = H::JB;
  double left = 0.0;
#pragma unroll 1
  for (int j0 = 0; j0 <= k; j0 += SH_JB) {
    double2 h[SH_JB + 1];
#pragma unroll
    for (int j = 0; j <= SH_JB; ++j) h[j] = make_double2(0.0, 0.0);
    const double2* Vj[SH_JB];
#pragma unroll
    for (int j = 0; j < SH_JB; ++j) Vj[j] = V + min(j0 + j, k) * stride;  // beyond k: V_k, not used
#pragma unroll 4
    for (int i = x.rg; i < n; i += RG) {
      const int o = i * NC + x.c;
      const double2 y = w[o];
      double2 p[SH_JB];
#pragma unroll
      for (int j = 0; j < SH_JB; ++j) p[j] = Vj[j][o];
      h[SH_JB].x = fma(y.x, y.x, fma(y.y, y.y, h[SH_JB].x));
#pragma unroll
      for (int j = 0; j < SH_JB; ++j) h[j] = cfma(h[j], cconj(p[j]), y);
    }
    shared_reduce<H, SH_JB + 1>(sh, h, x.c);
    if (j0 == 0) left = h[SH_JB].x;
#pragma unroll
    for (int j = 0; j < SH_JB; ++j) {
      if (j0 + j <= k) {
        left -= h[j].x * h[j].x + h[j].y * h[j].y;
        if (x.rg == 0) sh.h[j0 + j][x.c] = h[j];
      }
    }
  }
  const double hn = sqrt(fmax(left, 0.0));
  const double inv = hn > 1e-150 ? 1.0 / hn : 0.0;
  __syncthreads();  // sh.h
  constexpr int RB = H::RB;
#pragma unroll 1
  for (int i0 = x.rg; i0 < n; i0 += RB * RG) {
    int o[RB];
    double2 y[RB];
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      o[m] = min(i0 + m * RG, n - 1) * NC + x.c;
      y[m] = w[o[m]];
    }
#pragma unroll 2
    for (int j = 0; j <= k; ++j) {
      const double2 hj = sh.h[j][x.c];
      const double2* Vj = V + j * stride;
#pragma unroll
      for (int m = 0; m < RB; ++m) y[m] = cfms(y[m], hj, Vj[o[m]]);
    }
#pragma unroll
    for (int m = 0; m < RB; ++m)
      if (i0 + m * RG < n) {
        y[m] = cscale(y[m], inv);
        Vn[o[m]] = y[m];
        w[o[m]] = y[m];  // D(q) is applied to it there
      }
  }
  return shared_rotate<H>(sh, x.c, k, hn, live, target, res);
}

// The coefficients y of the cycle's vectors, from the column's triangular factor, into sh.h (kd of row
// group 0: the column's own vectors, of kmax in the tile).
template <typename H>
__device__ __forceinline__ void shared_coefficients(SharedLds<H>& sh, const SharedTile& x, int kd, int kmax) {
  if (x.rg == 0) {
#pragma unroll 1
    for (int j = kmax - 1; j >= 0; --j) {
      double2 r = make_double2(0.0, 0.0);
      if (j < kd) {
        r = sh.gv[j][x.c];
#pragma unroll 1
        for (int l = j + 1; l < kd; ++l) r = cfms(r, sh.R[l * (l + 1) / 2 + j][x.c], sh.h[l][x.c]);
        r = cmul(r, cinv(sh.R[j * (j + 1) / 2 + j][x.c]));
      }
      sh.h[j][x.c] = r;
    }
  }
  __syncthreads();
}

// X (+)= sum_j y_j V_j over the kmax vectors of the cycle; returns |X| of the column.
template <typename H>
__device__ __forceinline__ double shared_update(SharedLds<H>& sh, const SharedTile& x, const double2* V, double2* X,
                                                int n, int stride, int kd, int kmax, bool first) {
  constexpr int RG = H::RG, NC = H::NC;
  shared_coefficients<H>(sh, x, kd, kmax);
  double2 nrm[1] = {make_double2(0.0, 0.0)};
  constexpr int RB = H::RB;
#pragma unroll 1
  for (int i0 = x.rg; i0 < n; i0 += RB * RG) {
    int o[RB];
    double2 y[RB];
#pragma unroll
    for (int m = 0; m < RB; ++m) {
      o[m] = min(i0 + m * RG, n - 1) * NC + x.c;
      y[m] = first ? make_double2(0.0, 0.0) : X[o[m]];
    }
#pragma unroll 2
    for (int j = 0; j < kmax; ++j) {
      const double2 hj = sh.h[j][x.c];
      const double2* Vj = V + j * stride;
#pragma unroll
      for (int m = 0; m < RB; ++m) y[m] = cfma(y[m], hj, Vj[o[m]]);
    }
#pragma unroll
    for (int m = 0; m < RB; ++m)
      if (i0 + m * RG < n) {
        nrm[0].x = fma(y[m].x, y[m].x, fma(y[m].y, y[m].y, nrm[0].x));
        X[o[m]] = y[m];
      }
  }
  shared_reduce<H, 1>(sh, nrm, x.c);
  return sqrt(nrm[0].x);
}

// One tile from B to its output; u: its vector in LDS.
template <typename H>
__device__ __forceinline__ void shared_tile(const SharedTileArgs& ta, SharedLds<H>& sh, double2* u, int grp, int tile) {
  constexpr int RG = H::RG, T = H::T, NC = H::NC;
  const SharedGroups& s = ta.s;
  const LadderArgs& a = s.a;
  const int n = a.n, nv = a.nv, nq = a.nq, stride = 4 * shared_steps(n) * NC;
  const int g_abs = s.group0 + grp, w = g_abs % a.nw, chan = g_abs / a.nw;
  SharedTile x;
  x.c = threadIdx.x % NC;
  x.rg = threadIdx.x / NC;
  const int e = tile * NC + x.c, ec = min(e, s.N - 1);
  x.in = e < s.N;
  x.q = ec / T;
  x.t = ec - x.q * T;
  x.col = static_cast<size_t>(grp) * s.N + ec;
  x.dd = s.dd + static_cast<size_t>(w) * T * T * nv * nq + x.q;
  x.dv = s.dv ? s.dv + (static_cast<size_t>(chan) * nq + x.q) * T * T : nullptr;
  const size_t pk = static_cast<size_t>(shared_blocks(n)) * shared_steps(n) * 64;
  const double2* A0 = ta.A0 + grp * pk;
  const double2* P = ta.P + grp * pk;
  double2* V = ta.vec + static_cast<size_t>(blockIdx.x) * (SH_M + 2) * stride;
  double2* X = V + (SH_M + 1) * stride;

  for (int o = n * NC + threadIdx.x; o < stride; o += H::TH) u[o] = make_double2(0.0, 0.0);  // the products' zero rows
  // the state of a column is kept by its thread of row group 0
  int state = x.in && x.rg == 0 ? SH_RUN : SH_DONE;
  double xn = 0.0;
#pragma unroll 1
  for (int cycle = 0; cycle < SH_CYCLES; ++cycle) {
    const double2* b = s.z0 + static_cast<size_t>(grp) * n * T + x.t;
    if (cycle > 0) {
#pragma unroll 4
      for (int i = x.rg; i < n; i += RG) u[i * NC + x.c] = X[i * NC + x.c];
      __syncthreads();
      shared_product<H, false>(A0, u, n);
      shared_apply<H, true>(s, sh, x, X, u, u);
      __syncthreads();
      shared_product<H, true>(P, u, n);
    }
    // V_0 = b / |b|
    double2 nrm[1] = {make_double2(0.0, 0.0)};
#pragma unroll 4
    for (int i = x.rg; i < n; i += RG) {
      const double2 y = cycle > 0 ? u[i * NC + x.c] : b[i * T];
      nrm[0].x = fma(y.x, y.x, fma(y.y, y.y, nrm[0].x));
    }
    shared_reduce<H, 1>(sh, nrm, x.c);
    const double beta0 = sqrt(nrm[0].x);
    const double inv = beta0 > 0.0 ? 1.0 / beta0 : 0.0;
#pragma unroll 4
    for (int i = x.rg; i < n; i += RG) {
      const double2 y = cscale(cycle > 0 ? u[i * NC + x.c] : b[i * T], inv);
      V[i * NC + x.c] = y;
      u[i * NC + x.c] = y;
    }
    if (cycle == 0) xn = beta0;
    if (!(beta0 <= 1e300)) state = SH_FAIL;  // infinite or NaN
    if (cycle == 0 && !(beta0 >= SH_NORM_MIN && beta0 <= SH_NORM_MAX)) state = SH_FAIL;
    if (state == SH_RUN && beta0 <= SH_DONE_TOL * xn) state = SH_DONE;
    if (state == SH_RUN && cycle > 0 && beta0 > SH_STAGNATION * xn) state = SH_FAIL;  // P is no inverse
    const double target = fmax(SH_CYCLE_TOL * beta0, SH_DONE_TOL * xn);
    if (x.rg == 0) sh.gv[0][x.c] = make_double2(beta0, 0.0);
    bool live = state == SH_RUN;
    int kd = 0, k = 0;
    double res = beta0;
    while (__syncthreads_or(live)) {
      shared_apply<H, false>(s, sh, x, u, nullptr, u);
      __syncthreads();
      shared_product<H, true>(P, u, n);
      if (live) kd = k + 1;
      live = shared_step<H>(sh, x, V, u, V + (k + 1) * stride, n, stride, k, live, target, res);
      ++k;
    }
    const bool run = state == SH_RUN;
    const double xnew = shared_update<H>(sh, x, V, X, n, stride, run ? kd : 0, k, cycle == 0);
    if (run) {
      xn = xnew;
      if (!(xn <= 1e300) || !(res <= 1e300))
        state = SH_FAIL;
      else if (cycle > 0 && res <= 2.0 * SH_DONE_TOL * xn && beta0 <= SH_TRUST * xn)
        state = SH_DONE;
      else if (!(res <= SH_STAGNATION * beta0))
        state = SH_FAIL;
    }
    if (!__syncthreads_or(state == SH_RUN)) break;
  }
  if (x.in) {
    if (x.rg == 0) s.state[x.col] = state;
    const size_t ob = (static_cast<size_t>(chan) * a.nw + w) * T * T * nv * nq + x.q;
    for (int i = x.rg; i < n; i += RG) {
      const int ri = i / nv, vi = i - ri * nv;
      a.out[ob + (static_cast<size_t>(ri * T + x.t) * nv + vi) * nq] = cscale(X[i * NC + x.c], a.inv_beta);
    }
  }
}

// Workgroups take tiles from a counter per XCD (the tiles of a group share P and A0 in its L2; workgroup
// b runs on XCD b % NUM_XCD), then from the other XCDs' groups. Every counter only grows, so each
// workgroup leaves after at most NUM_XCD exhausted counters.
template <typename H, int WG_PER_CU>
__global__ void __launch_bounds__(H::TH, WG_PER_CU * H::NW / 4) shared_tile_kernel(SharedTileArgs ta) {
  __shared__ SharedLds<H> sh;
  extern __shared__ double2 s_u[];
  for (int off = 0; off < NUM_XCD; ++off) {
    const int xcd = (blockIdx.x + off) % NUM_XCD;
    const int tiles = (ta.s.groups - xcd + NUM_XCD - 1) / NUM_XCD * ta.ntile;  // of the groups xcd, xcd + NUM_XCD, ...
    for (;;) {
      __syncthreads();
      if (threadIdx.x == 0) sh.tile = atomicAdd(&ta.next[xcd], 1);
      __syncthreads();
      const int id = sh.tile;
      if (id >= tiles) break;
      const int j = id / ta.ntile;
      shared_tile<H>(ta, sh, s_u, xcd + NUM_XCD * j, id - j * ta.ntile);
    }
  }
}

// ---------------------------------------------------------------------------
// Up to n = 128: four wavefronts of 32 rows and two workgroups per CU, which overlap one another's products and
// sweeps, where there are tiles for them; with fewer tiles eight wavefronts of 16 rows, each with half the
// rows to pass over. Up to 256 eight wavefronts of 32 rows.
static bool tile_pairs(const SharedGroups& s) {
  return s.a.n <= 128 && static_cast<size_t>(s.groups) * ceil_div(s.N, 16) > 512;
}

static int tile_workgroups(const SharedGroups& s) {
  const size_t tiles = static_cast<size_t>(s.groups) * ceil_div(s.N, 16);
  return static_cast<int>(std::min<size_t>(s.a.n <= 128 ? 512 : 256, tiles));
}

size_t shared_tile_workspace(const SharedGroups& s) {
  return static_cast<size_t>(tile_workgroups(s)) * (SH_M + 2) * 4 * shared_steps(s.a.n) * 16;
}

template <typename H, int WG_PER_CU>
static int tile_launch(const SharedTileArgs& ta, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(4 * shared_steps(ta.s.a.n)) * H::NC * sizeof(double2);
  auto kern = shared_tile_kernel<H, WG_PER_CU>;
  allow_lds(kern, lds);
  hipLaunchKernelGGL(kern, dim3(tile_workgroups(ta.s)), dim3(H::TH), lds, stream, ta);
  DGAMI_HIP_CHECK(hipGetLastError());
  return 0;
}

template <int T>
static int tile_launch_t(const SharedTileArgs& ta, hipStream_t stream) {
  if (tile_pairs(ta.s)) return tile_launch<SharedShape<T, 4, 2>, 2>(ta, stream);
  if (ta.s.a.n <= 128) return tile_launch<SharedShape<T, 8, 1>, 1>(ta, stream);
  return tile_launch<SharedShape<T, 8, 2>, 1>(ta, stream);
}

int shared_tile_solve(const SharedGroups& s, double2* pack, double2* z0, double2* vec, int* next, hipStream_t stream) {
  const int n = s.a.n;
  const size_t pk = shared_packed(n);
  hipLaunchKernelGGL(shared_pack_kernel, dim3(2 * ceil_div(pk, 256) + ceil_div(n, 4) + 1, s.groups), dim3(256),
                     n * sizeof(uint4), stream, s, pack, z0, next);
  DGAMI_HIP_CHECK(hipGetLastError());
  const SharedTileArgs ta{s, pack, pack + pk * s.groups, static_cast<int>(ceil_div(s.N, 16)), vec, next};
  return s.a.T == 1 ? tile_launch_t<1>(ta, stream) : tile_launch_t<4>(ta, stream);
}

}  // namespace dgami
