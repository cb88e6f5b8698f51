// Fused Gaussian random walk (GaussianRandomWalk.kernel,
// src/flowMC/resource/kernel/Gaussian_random_walk.py:25-61): the chain kernels
// of fmc_chain_kernel.h instantiated for that step kind, in a translation unit
// of their own.
#include "fmc_chain_kernel.h"

namespace fmc {

int launch_grw(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg, const Layout& L) {
  return launch_chain_impl<KK_GRW>(st, t, io, cfg, L);
}

}  // namespace fmc
