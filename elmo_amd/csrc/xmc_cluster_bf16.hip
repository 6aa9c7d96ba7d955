// The variants of the one-pass cluster step for bf16 weights; compiled with the register-pressure trackers of the instruction
// scheduler (elmo_amd/build.py), which halve the spills of these kernels.
#define CLU_VARIANT bf16
#define CLU_WT CLU_BF16
#define CLU_QX 0
#include <hip/hip_runtime.h>
#include "xmc_cluster.hip"
