// Reference-order EC flux-differencing kernels on box elements for EulerGravityLaw, rusanov surface flux.
#include "box_fd.hpp"

namespace atm {
Resolved resolve_box_fd_euler_gravity_rusanov(int dim, int Nq) { return fd_box_dims<EulerGravity, ATM_FLUX_RUSANOV>(dim, Nq); }
}  // namespace atm
