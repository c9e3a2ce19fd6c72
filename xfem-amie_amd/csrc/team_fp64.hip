// Team CG kernels: FP64 vectors on the scaled FP64 planes.
#include "team.hpp"

namespace amie {

TeamFn team_fn_fp64(int b, int nr, bool bj, int j) { return team_pick<double, Pre64>(b, nr, bj, j); }

} // namespace amie
