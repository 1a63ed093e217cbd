// Ladder sums through the (channel, w) groups' shared matrix (ladder_shared.hip).
#pragma once

#include "ladder_common.hpp"

namespace dgami {

// Compound sizes above SHARED_MIN_N with at least SHARED_MIN_NQ q-points per group take it.
constexpr int SHARED_MIN_N = 64;
constexpr int SHARED_MIN_NQ = 16;

bool ladder_shared_applies(const LadderArgs& a);
int ladder_solve_shared(const LadderArgs& a, hipStream_t stream);

}  // namespace dgami
