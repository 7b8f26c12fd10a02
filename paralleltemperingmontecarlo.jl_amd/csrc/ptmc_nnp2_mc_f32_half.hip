// NNVT kernels of the two-species network potential with binary32 positions,
// features and networks (FP64 energy sums), two workgroups a CU.
#define N2R float
#define N2_THREADS (NNP2_NT / 2)
#define N2_SWEEP_FN nnp2_sweep_fn_f32_half
#define N2_INIT_FN nnp2_init_fn_f32_half
#include "ptmc_nnp2_mc.hpp"
