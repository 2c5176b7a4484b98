// The FP64 unsplit Euler step kernels (plain and periodic boundaries, no capacity function), in a
// translation unit of their own so that they can be built with LLVM's max-ilp machine scheduler
// (clawpack_amd/build.py).  claw2d.hip declares them extern and launches them.
#define CLAW_KERNEL_UNIT 1
#include "claw2d.hip"

namespace claw {
#define CLAW_EULER64_DEFINE(LIM, TWC)                                                        \
  template __global__ void step2_fused<double, EulerP<double>, LIM, false, TWC, false, 0, false>( \
      StepArgs<double, EulerP<double>>);
CLAW_EULER64_KERNELS(CLAW_EULER64_DEFINE)
}  // namespace claw
