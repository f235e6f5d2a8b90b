// LDS path: mixed-radix kernels and launchers for double planes.
#include "kern_mix.h"

namespace curig {
CURIG_MIX_INST(double)
}  // namespace curig
