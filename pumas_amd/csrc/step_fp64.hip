/* The FP64 stepping kernels. */
#include "k_step.h"

template StepKernel step_kernel<false, false>(int, bool);
