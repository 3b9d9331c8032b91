// Weak-form kernels on box elements for ShallowWaterLaw.
#include "box.hpp"

namespace atm {
Resolved resolve_box_weak_shallow_water(int dim, int mask, int Nq) {
  Resolved r = weak_box_dims<ShallowWater, ATM_FLUX_RUSANOV, false>(dim, mask, Nq);
  // 2-D members of N = 3..7 take one launch per stage whatever their N
  if (r.fn && dim == 2 && Nq >= 4 && Nq <= 8) r.mbfn = launch_weak_box_multi_batch<ShallowWater<2>, ATM_FLUX_RUSANOV>;
  return r;
}
}  // namespace atm
