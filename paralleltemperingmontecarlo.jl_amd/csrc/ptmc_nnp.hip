// Neural-network potential kernels (one translation unit; see ptmc_nnp.hpp).
#include "ptmc_nnp.hpp"

namespace ptmc {

using SweepFn = void (*)(SweepArgs);

// np: atoms per slot, NNP_NP (64) or NNP_NP_WIDE (128); nt: threads per
// workgroup, NNP_NT or (always for 128 atoms) twice that
SweepFn nnp_sweep_fn(int np, int nt)
{
    if (np > NNP_NP) return &nnp_sweep_kernel<false, NNP_NP_WIDE, 2 * NNP_NT>;
    return nt > NNP_NT ? &nnp_sweep_kernel<false, NNP_NP, 2 * NNP_NT> : &nnp_sweep_kernel<false, NNP_NP, NNP_NT>;
}
SweepFn nnp_sweep_da_fn() { return &nnp_sweep_kernel<true, NNP_NP, NNP_NT>; }
SweepFn nnp_init_fn(int np, int nt)
{
    if (np > NNP_NP) return &nnp_init_kernel<NNP_NP_WIDE, 2 * NNP_NT>;
    return nt > NNP_NT ? &nnp_init_kernel<NNP_NP, 2 * NNP_NT> : &nnp_init_kernel<NNP_NP, NNP_NT>;
}
SweepFn nnp_cycle_fn() { return &nnp_cycle_kernel; }

}  // namespace ptmc
