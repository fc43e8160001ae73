/* The FP64 stepping kernels of launches with a frame recorder. */
#include "k_step.h"

template StepKernel step_kernel<false, true>(int, bool);
