// NNVT kernels of the two-species network potential in FP64, two workgroups a CU.
#define N2R double
#define N2_THREADS (NNP2_NT / 2)
#define N2_SWEEP_FN nnp2_sweep_fn_half
#define N2_INIT_FN nnp2_init_fn_half
#include "ptmc_nnp2_mc.hpp"
