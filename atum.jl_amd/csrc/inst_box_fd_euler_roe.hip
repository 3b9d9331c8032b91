// Reference-order EC flux-differencing kernels on box elements for EulerLaw, roe surface flux.
#include "box_fd.hpp"

namespace atm {
Resolved resolve_box_fd_euler_roe(int dim, int Nq) { return fd_box_dims<Euler, ATM_FLUX_ROE>(dim, Nq); }
}  // namespace atm
