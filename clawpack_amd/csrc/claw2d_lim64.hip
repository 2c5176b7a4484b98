// The FP64 step kernels with superbee and van Leer and those without transverse waves, in a translation
// unit of their own so that they are compiled beside the others.  claw2d.hip declares them extern and
// launches them.
#define CLAW_KERNEL_UNIT 1
#include "claw2d.hip"

namespace claw {
CLAW_LIMITER_KERNELS(CLAW_LIMITER_DEFINE, double)
CLAW_NO_TRANSVERSE_KERNELS(CLAW_LIMITER_DEFINE, double)
}  // namespace claw
