// The resident RKC kernels of the olive model.
#include "rkc_models.hpp"

namespace cbrkc {
const void *rkc_kernel_io(int k) { return rkc_kernel_of<IoModel>(k); }
}  // namespace cbrkc
