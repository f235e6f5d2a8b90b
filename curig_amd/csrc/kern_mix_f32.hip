// LDS path: mixed-radix kernels and launchers for float planes.
#include "kern_mix.h"

namespace curig {
CURIG_MIX_INST(float)
}  // namespace curig
