// The resident RKC kernels of the granule model.
#include "rkc_models.hpp"

namespace cbrkc {
const void *rkc_kernel_gr(int k) { return rkc_kernel_of<GrModel>(k); }
}  // namespace cbrkc
