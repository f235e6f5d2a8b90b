// LDS path: whole power-of-two rows, kernels and launchers for float planes.
#include "kern_rowreg.h"

namespace curig {
CURIG_ROWREG_INST(float)
}  // namespace curig
