// Pair-symmetric EC flux-differencing kernels on box elements for EulerLaw, rusanov surface flux.
#include "box_fast.hpp"

namespace atm {
Resolved resolve_box_fast_euler_rusanov(int dim, int Nq) { return fast_box_dims<Euler, ATM_FLUX_RUSANOV>(dim, Nq); }
}  // namespace atm
