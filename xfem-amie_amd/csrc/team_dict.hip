// Team CG kernels: FP32 vectors on the value-indexed FIX48 matrix.
#include "team.hpp"

namespace amie {

TeamFn team_fn_dict(int b, int nr, bool bj, int j) { return team_pick<float, Dict>(b, nr, bj, j); }

} // namespace amie
