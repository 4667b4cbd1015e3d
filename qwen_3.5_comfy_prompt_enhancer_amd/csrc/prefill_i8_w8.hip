// The tiled int8-activation kernels for int8 weights (the kernel is in prefill_i8_kernel.h).
#include "prefill_i8_kernel.h"

namespace qlin {

template hipError_t launch_i8_w<WK_W8, false>(const SkArgs&, int, int, int, hipStream_t);

}  // namespace qlin
