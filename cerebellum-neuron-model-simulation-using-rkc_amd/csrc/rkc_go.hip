// The resident RKC kernels of the Golgi model.
#include "rkc_models.hpp"

namespace cbrkc {
const void *rkc_kernel_go(int k) { return rkc_kernel_of<GoModel>(k); }
}  // namespace cbrkc
