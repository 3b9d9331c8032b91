// Weak-form kernels on box elements for LinearEulerGravityLaw.
#include "box.hpp"

namespace atm {
Resolved resolve_box_weak_linear(int dim, int mask, int Nq) {
  return weak_box_dims<LinearEulerGravity, ATM_FLUX_RUSANOV, true>(dim, mask, Nq);
}
}  // namespace atm
