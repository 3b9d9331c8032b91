// Pair-symmetric EC flux-differencing kernels on box elements for EulerGravityLaw, rusanov surface flux.
#include "box_fast.hpp"

namespace atm {
Resolved resolve_box_fast_euler_gravity_rusanov(int dim, int Nq) { return fast_box_dims<EulerGravity, ATM_FLUX_RUSANOV>(dim, Nq); }
}  // namespace atm
