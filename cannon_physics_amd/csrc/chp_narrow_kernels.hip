// chp_narrow_kernels.hip -- the narrowphase resolver kernels of one precision (CHP_REAL).
#include "chp_kernels.h"

namespace chp {
CHP_NARROW_KERNELS(template __global__, CHP_REAL)
}  // namespace chp
