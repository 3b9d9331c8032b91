// Reference-order EC flux-differencing kernels on box elements for EulerGravityLaw, roe surface flux.
#include "box_fd.hpp"

namespace atm {
Resolved resolve_box_fd_euler_gravity_roe(int dim, int Nq) { return fd_box_dims<EulerGravity, ATM_FLUX_ROE>(dim, Nq); }
}  // namespace atm
