// Weak-form kernels on box elements for EulerGravityLaw.
#include "box.hpp"

namespace atm {
Resolved resolve_box_weak_euler_gravity(int dim, int mask, int Nq) {
  return weak_box_dims<EulerGravity, ATM_FLUX_RUSANOV, false>(dim, mask, Nq);
}
}  // namespace atm
