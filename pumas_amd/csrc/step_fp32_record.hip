/* The FP32-bulk stepping kernels of launches with a frame recorder. */
#include "k_step.h"

template StepKernel step_kernel<true, true>(int, bool);
