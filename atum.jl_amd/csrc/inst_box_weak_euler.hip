// Weak-form kernels on box elements for EulerLaw.
#include "box.hpp"

namespace atm {
Resolved resolve_box_weak_euler(int dim, int mask, int Nq) {
  return weak_box_dims<Euler, ATM_FLUX_RUSANOV, false>(dim, mask, Nq);
}
}  // namespace atm
