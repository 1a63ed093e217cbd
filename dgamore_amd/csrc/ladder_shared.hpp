// Ladder sums through the (channel, w) groups' shared matrix: ladder_shared.hip (the method, its set-up and
// the form for large compound sizes) and ladder_shared_tile.hip (the form for sizes up to SHARED_TILE_N).
#pragma once

#include "dgami_internal.hpp"
#include "ladder_common.hpp"

namespace dgami {

// The rule: at least SHARED_MIN_NQ q-points share a matrix (its inversion costs three LUs), and there are
// enough problems for the LU to be past its own latency, by how much more an LU computes per problem than a
// product: problems x ratio >= a bound, with ratio = n / (3 T) + 1. With one or two orbitals up to n = 256 the
// bound is SHARED_MIN_WORK_1 (T = 1) or SHARED_MIN_WORK_4, and SHARED_MIN_WORK_N32 up to n = 32, where the LU is
// one small register tile; beyond, the ratio itself has to reach SHARED_MIN_RATIO (the passes over the basis and the
// D(q) blocks grow with T), with other bounds for the mixed forms, whose LU is faster too. The lines lie where
// this form wins by a third: the iterations of a self-consistency loop grow harder than its first (n = 540, 240 and
// 1080, eight of them, mixing 0.3: 20 -> 37, 5.7 -> 8.4 and 118 -> 212 ms; LU 27, 10.2 and 248), and the LU's time does not.
// Measured, LU / this form in us (beta = 10 ... 40, U = 3 ... 8). T = 1 below: n = 30, 1440 problems 168 / 230; n = 40,
// 990 problems 161 / 185, 1350 230 / 187; n = 96, 392 problems 444 / 563; n = 120, 450 problems 608 / 472; above: n = 40,
// 1890 problems 276 / 184; n = 64, 990 problems 384 / 229; n = 120, 810 problems 765 / 482, 68442 problems 38100 / 3530.
// T = 4 below: n = 32, 1440 problems 203 / 293; n = 48, 1440 problems 323 / 336; above: n = 64, 1440 problems 550 / 379;
// n = 120, 1440 problems 1072 / 764; n = 216, 540 problems 1588 / 1300; n = 256, 540 problems 2101 / 1422. Large,
// complex128, below: T = 9, n = 252, 560 problems 2207 / 2652; n = 360, 2790 problems 18169 / 17032; n = 720, 448
// problems 16025 / 15066; T = 4, n = 400, 540 problems 5488 / 5309; above: 630 problems 5756 / 3839; T = 9, n = 540, 1170
// problems 20020 / 15003; n = 720, 5642 problems 239700 / 82000. Split-BF16 below: T = 9, n = 360, 2790 problems 12119 /
// 8767; n = 540, 2700 problems 26600 / 20050; n = 720, 448 problems 9814 / 8481; T = 4, n = 400, 540 problems 4681 / 3416;
// above: n = 720, 5642 problems 93282 / 39980. Complex64: n = 720, 720 problems 20929 / 13331.
constexpr int SHARED_MIN_NQ = 16;
constexpr double SHARED_MIN_WORK_1 = 20000.0, SHARED_MIN_WORK_4 = 9000.0, SHARED_MIN_WORK_N32 = 30000.0;
constexpr double SHARED_MIN_WORK = 20000.0, SHARED_MIN_WORK_MIXED = 25000.0;
constexpr double SHARED_MIN_RATIO = 18.0, SHARED_MIN_RATIO_MIXED = 24.0;
constexpr int SHARED_TILE_N = 256;

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
};

// DGAMI_LADDER_SHARED = 0 / 1: never / wherever the form can run (for comparisons and tests).
bool ladder_shared_applies(const LadderArgs& a, int precision);
// slot_offset: of the workspaces (k WS_STREAM_STRIDE for work on extra stream k).
int ladder_solve_shared(const LadderArgs& a, int precision, hipStream_t stream, int slot_offset = 0);

// A batch of n <= SHARED_TILE_N, to the output and the columns' state, with z0 = P B. pack: space for two
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
