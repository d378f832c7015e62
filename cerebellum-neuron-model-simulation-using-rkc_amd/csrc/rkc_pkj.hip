// The resident RKC kernels of the Purkinje model.
#include "rkc_models.hpp"

namespace cbrkc {
const void *rkc_kernel_pkj(int k) { return rkc_kernel_of<PkjModel>(k); }
}  // namespace cbrkc
