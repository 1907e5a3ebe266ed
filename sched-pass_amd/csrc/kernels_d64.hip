// kernels_d64.hip -- instantiates the decode kernels for head dim 64 on the
// matrix cores (the list is in kernel_set.h).
#include <hip/hip_runtime.h>

#include "kernel_set.h"

SCHED_PD_MFMA_D64()
