// Team CG kernels: FP32 vectors on the FIX48 planes.
#include "team.hpp"

namespace amie {

TeamFn team_fn_fix48(int b, int nr, bool bj, int j) { return team_pick<float, Fix48>(b, nr, bj, j); }

} // namespace amie
