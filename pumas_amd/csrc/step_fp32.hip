/* The FP32-bulk stepping kernels. */
#include "k_step.h"

template StepKernel step_kernel<true, false>(int, bool);
