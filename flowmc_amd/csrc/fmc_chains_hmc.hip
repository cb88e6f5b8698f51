// Fused HMC with a unit or diagonal condition matrix (HMC.kernel,
// src/flowMC/resource/kernel/HMC.py:98-151): the chain kernels
// of fmc_chain_kernel.h instantiated for that step kind, in a translation unit
// of their own.
#include "fmc_chain_kernel.h"

namespace fmc {

int launch_hmc(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg, const Layout& L) {
  if (io.chol) return launch_hmc_dense(st, t, io, cfg, L);
  return launch_chain_impl<KK_HMC>(st, t, io, cfg, L);
}

}  // namespace fmc
