// Ladder sums through the (channel, w) groups' shared matrix: ladder_shared.hip (the method, its set-up and
// the form for large compound sizes) and ladder_shared_tile.hip (the form for sizes up to SHARED_TILE_N).
#pragma once

#include "dgami_internal.hpp"
#include "ladder_common.hpp"

namespace dgami {

// The rule: at least SHARED_MIN_NQ q-points share a matrix (its inversion costs three LUs), and there are
// enough problems for the LU to be past its own latency, by how much more an LU computes per problem than a
// product: work = problems x ratio reaches a bound, with ratio = n / (3 T) + 1. The LU's time does not depend on the
// data, this form's does: the matrices of a self-consistency loop are harder than those of its first iteration, 10 ... 18
// iterations per column there, 14 ... 35 at the eighth. The lines lie where the first eight iterations of a loop
// (mixing 0.3) take this form no longer than the LU, in the geometric mean over a strong and a weak interaction,
// within 3%. That leaves the last of them slower near a line (by up to 1.7 times) and faster from about twice the
// bound on; a single first iteration gains 1.2 ... 3 times everywhere above.
// Measured: problems, work: LU / mean of the eight, and LU / the first and the last, strong and weak interaction.
// T = 1, n = 30: 1890, 20790: 0.82; 2790, 30690: 1.07 (1.59 0.96, 1.24 0.82). n = 40: 1440, 20640: 0.81;
// 1890, 27090: 0.97 (1.49 0.81, 1.18 0.73); 3822, 54782: 1.64 (2.49 1.36, 1.99 1.24). n = 64: 990, 22110: 0.99; 1350, 30150:
// 1.28. n = 80: 1188, 32868: 1.06. n = 96: 990, 32670: 0.96. n = 120: 810, 33210: 0.98; 1170, 47970: 1.18 (2.02 0.61, 1.64 0.83);
// 2790, 114390: 1.88. n = 150: 990, 50490: 0.92. n = 200: 630, 42630: 1.01; 1530, 103530: 1.61. n = 240: 810, 65610: 1.21.
// T = 4, n = 32: 3690, 13530: 0.96. n = 48: 1890, 9450: 1.04. n = 64: 1440, 9120: 1.23 (1.61 1.24, 1.34 0.94). n = 96: 1440, 12960:
// 0.97. n = 120: 990, 10890: 1.01; 1440, 15840: 1.11; 2912, 32032: 1.21. n = 160: 1584, 22704: 0.89; 2730, 39130: 1.06.
// n = 216: 540, 10260: 0.81; 1080, 20520: 1.05; 2184, 41496: 1.37 (1.97 1.19, 1.60 0.86). n = 256: 540, 12060: 0.91; 2002, 44711: 1.52.
// Large, complex128: T = 4, n = 320: 1890, 52290: 0.87; n = 400: 1452, 49852: 0.88; 3822, 131222: 1.51 (2.79 0.96, 2.05 1.04);
// n = 720: 630, 38430: 0.97; 1350, 82350: 1.55. T = 9, n = 360: 2912, 41739: 0.80; n = 540: 2366, 49686: 0.90; 5642, 118482:
// 1.30; n = 720: 1638, 45318: 0.92; 2366, 65459: 1.12; 5642, 156095: 1.59 (2.38 1.29, 1.91 1.18); n = 1080: 1274, 52234: 1.30.
// Complex64 and split BF16: T = 4, n = 320: 1890: 1.11, 1.04; n = 400: 630, 21630: 0.83, 0.75; 1452: 1.19, 1.05; T = 9,
// n = 540: 1170, 24570: 0.85, 0.78; n = 720: 728, 20141: 0.91, 0.80; 1638: 1.14, 1.02; 5642: 2.01, 1.66.
constexpr int SHARED_MIN_NQ = 16;
constexpr double SHARED_MIN_WORK_N32 = 30000.0;  // n <= 32, where the LU is one small register tile (T <= 4)
// up to n = 64 (the inverse in the small register tile), 128 and 256, one (T = 1) and two (T = 4) orbitals
constexpr double SHARED_MIN_WORK_1[3] = {27000.0, 35000.0, 60000.0};
constexpr double SHARED_MIN_WORK_4[3] = {9000.0, 13500.0, 30000.0};
// the large form: with a small ratio the passes over the basis and the D(q) blocks, which grow with T, weigh more
constexpr double SHARED_MIN_WORK = 65000.0, SHARED_MIN_WORK_MIXED = 45000.0;
constexpr double SHARED_MIN_RATIO = 18.0, SHARED_MIN_RATIO_MIXED = 24.0;
constexpr int SHARED_TILE_N = 256, SHARED_TILE_T = 4;  // of the form in tiles

constexpr int SH_M = 10;           // Krylov vectors of a cycle
constexpr int SH_ROT = SH_M * (SH_M + 1) / 2;

// A cycle stops a column at a residual of SH_CYCLE_TOL of its start (below that the error of P
// decides); the column is done when its residual is below SH_DONE_TOL of |X|.
constexpr int SH_CYCLES = 5;
constexpr double SH_CYCLE_TOL = 1e-10;
constexpr double SH_DONE_TOL = 2e-16;
// ... provided that the cycle began at a residual below SH_TRUST of |X|: the preceding cycle then was right
// to SH_TRUST, so P is the inverse of A0 to SH_TRUST and this cycle's error is at most that part of its start.
constexpr double SH_TRUST = 1e-7;
// The same with the basis, P and D(q) in complex64 (the mixed forms above SHARED_TILE_N; X, A0 and the residuals
// stay in FP64; the split-BF16 form multiplies P in split BF16, with the same number of cycles in every case
// measured): a cycle can gain five digits, and the residual P (B - A X) is wanted below SH_DONE_TOL_C64 of |X|, four
// digits beyond what the refinement of the mixed LU asks for.
constexpr double SH_CYCLE_TOL_C64 = 1e-5, SH_DONE_TOL_C64 = 1e-14, SH_TRUST_C64 = 1e-9;
// The norms and the orthogonality of a complex64 basis hold to about 2^-23 only, so |w|^2 - sum |h|^2 says nothing
// about a remainder below SH_LOSS_C64 |w|^2 (where D(q) is close to a multiple of A0 it came out as zero, and columns
// ended at 5e-12). The remainder is taken as no smaller; and whether a column is done decides the norm of the
// residual as the stored vectors give it, formed with the update of X, not the Hessenberg matrix's estimate.
constexpr double SH_LOSS_C64 = 2.4e-7;
// A cycle that leaves more than this of its residual is stagnating.
constexpr double SH_STAGNATION = 0.3;
// Columns whose first vector P B lies outside these bounds are left to the LU: its square, or that of a residual
// 2^-53 of it, would leave the range of double (or P and its products that of float), and a column of zeros
// pass for a converged one.
constexpr double SH_NORM_MIN = 1e-130, SH_NORM_MAX = 1e130;
constexpr double SH_NORM_MIN_C64 = 1e-20, SH_NORM_MAX_C64 = 1e20;

enum SharedState { SH_RUN = 0, SH_DONE = 1, SH_FAIL = 2 };

// The groups of a batch and their operands.
struct SharedGroups {
  LadderArgs a;
  int group0, groups;     // groups of this batch
  int N;                  // columns (q, t) of a group
  const double2* A0;      // [groups][n][n] mean matrices
  const double2* P;       // [groups][n][n] their inverses
  const double2* dd;      // D(q): [nw][T*T][nv][nq]
  const double2* dv;      // (V_r(q) - mean V_r) / beta^2: [nchan][nq][T*T], or null
  const double2* z0;      // P B [groups][n][T]
  int* state;             // [groups][N] SharedState
  const int* zero;        // [nw][T][nv] whether chi0^-1 vanishes on the block's diagonal for some q
  int* equal;             // [groups] whether a matrix of the group may have two equal rows
};

// Whether some A(q) of a group may have two equal rows of one orbital pair: such a matrix is singular, but its
// right-hand sides are equal there too, so the iteration would solve it where the LU reports the zero pivot
// (collected problems go to the LU). Rows (c, a) and (c, b) can only be equal if those of the vertex are in every
// column but those of the frequencies a and b; four columns are compared (as hashes in LDS, [n][4]), which
// tells any two rows of an actual vertex apart. Where they and the columns a and b of the pair agree (a vertex
// that is constant there), A(q) has equal rows if chi0^-1 vanishes in both; otherwise it has them if chi0^-1 makes
// up for the difference, which is left to the LU to find out. All 256 threads of a workgroup call it; it runs
// beside the packing (calls of n = 40, 120, 216 and 720 take the same time with and without it).
__device__ inline bool shared_equal_rows(const SharedGroups& s, int grp, uint4* hash) {
  const int n = s.a.n, T = s.a.T, nv = s.a.nv;
  const double2* G = s.a.gamma + static_cast<size_t>(s.group0 + grp) * n * n;
  const int* zero = s.zero + static_cast<size_t>((s.group0 + grp) % s.a.nw) * n;
  unsigned* words = reinterpret_cast<unsigned*>(hash);
  for (int e = threadIdx.x; e < 4 * n; e += 256) {
    const int row = e >> 2, col = row / nv * nv + (e & 3) * nv / 4;
    const double2 x = G[static_cast<size_t>(row) * n + col];
    const unsigned long long re = __double_as_longlong(x.x + 0.0), im = __double_as_longlong(x.y + 0.0);  // -0 = 0
    words[e] = static_cast<unsigned>(re ^ (re >> 32)) * 0x9e3779b1u + static_cast<unsigned>(im ^ (im >> 32)) * 0x85ebca77u;
  }
  __syncthreads();
  int found = 0;
  for (int e = threadIdx.x; e < T * nv * nv; e += 256) {
    const int ra = e / nv, b = e - ra * nv, c = ra / nv, a = ra - c * nv, rb = c * nv + b;
    if (a >= b) continue;
    const uint4 ha = hash[ra], hb = hash[rb];
    auto same = [&](unsigned x, unsigned y, int v) { return x == y || v == a || v == b; };
    if (!(same(ha.x, hb.x, 0) && same(ha.y, hb.y, nv / 4) && same(ha.z, hb.z, nv / 2) && same(ha.w, hb.w, 3 * nv / 4)))
      continue;
    const double2* A = G + static_cast<size_t>(ra) * n + c * nv;
    const double2* B = G + static_cast<size_t>(rb) * n + c * nv;
    const bool constant = A[a].x == B[a].x && A[a].y == B[a].y && A[b].x == B[b].x && A[b].y == B[b].y;
    found |= !constant || (zero[ra] && zero[rb]);
  }
  return __syncthreads_or(found) != 0;
}

// DGAMI_LADDER_SHARED = 0 / 1: never / wherever the form can run (for comparisons and tests).
bool ladder_shared_applies(const LadderArgs& a, int precision);
// slot_offset: of the workspaces (k WS_STREAM_STRIDE for work on extra stream k). SHARED_NO_SPACE: the device
// memory holds not even one group of it, and nothing was launched (the caller takes the LU, which may need less).
constexpr int SHARED_NO_SPACE = -3;
int ladder_solve_shared(const LadderArgs& a, int precision, hipStream_t stream, int slot_offset = 0);

// A batch of n <= SHARED_TILE_N and T <= SHARED_TILE_T, to the output and the columns' state, with z0 = P B. pack: space for two
// packed matrices per group (shared_packed); next: NUM_XCD integers.
size_t shared_packed(int n);
size_t shared_tile_workspace(const SharedGroups& s);
int shared_tile_solve(const SharedGroups& s, double2* pack, double2* z0, double2* vec, int* next, hipStream_t stream);

// Mean matrices of a batch and their inverses (vmean may be null; ladder_shared_inverse.hip). work: groups times
// shared_inverse_workspace(n) values. A matrix that cannot be inverted is NaN in P.
constexpr int SHARED_SMALL_N = 128;
size_t shared_inverse_workspace(int n);
int shared_inverse(const SharedGroups& s, const double2* mean, const double2* vmean, double2* A0, double2* P,
                   double2* work, hipStream_t stream);

}  // namespace dgami
