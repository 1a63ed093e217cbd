// Ladder sums through the (channel, w) groups' shared matrix: ladder_shared.hip (the method, its set-up and
// the form for large compound sizes) and ladder_shared_tile.hip (the form for sizes up to SHARED_TILE_N).
#pragma once

#include "dgami_internal.hpp"
#include "ladder_common.hpp"

namespace dgami {

// Compound sizes above SHARED_MIN_N with at least SHARED_MIN_NQ q-points per group take it.
constexpr int SHARED_MIN_N = 64;
constexpr int SHARED_MIN_NQ = 16;
constexpr int SHARED_TILE_N = 256;

constexpr int SH_M = 10;           // Krylov vectors of a cycle
constexpr int SH_ROT = SH_M * (SH_M + 1) / 2;

// A cycle stops a column at a residual of SH_CYCLE_TOL of its start (below that the error of P
// decides); the column is done when its residual is below SH_DONE_TOL of |X|.
constexpr int SH_CYCLES = 4;
constexpr double SH_CYCLE_TOL = 1e-10;
constexpr double SH_DONE_TOL = 2e-16;
// A cycle that leaves more than this of its residual is stagnating.
constexpr double SH_STAGNATION = 0.3;

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

bool ladder_shared_applies(const LadderArgs& a);
int ladder_solve_shared(const LadderArgs& a, hipStream_t stream);

// The solution of a batch of n <= SHARED_TILE_N, to the output and the columns' state. pack: space for two
// packed matrices per group (shared_packed); next: NUM_XCD integers.
size_t shared_packed(int n);
size_t shared_tile_workspace(const SharedGroups& s);
int shared_tile_solve(const SharedGroups& s, double2* pack, double2* vec, int* next, hipStream_t stream);

}  // namespace dgami
