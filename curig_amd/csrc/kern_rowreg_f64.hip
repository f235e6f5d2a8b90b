// LDS path: whole power-of-two rows, kernels and launchers for double planes.
#include "kern_rowreg.h"

namespace curig {
CURIG_ROWREG_INST(double)
}  // namespace curig
