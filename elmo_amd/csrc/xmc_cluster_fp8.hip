// The variants of the one-pass cluster step for e4m3 weights with FP8 logits (true FP8); compiled with the register-pressure trackers of the instruction
// scheduler (elmo_amd/build.py), which halve the spills of these kernels.
#define CLU_VARIANT fp8
#define CLU_WT CLU_E4M3
#define CLU_QX 1
#include <hip/hip_runtime.h>
#include "xmc_cluster.hip"
