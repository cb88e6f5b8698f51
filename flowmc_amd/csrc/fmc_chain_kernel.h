// The fused chain kernel (one kernel per lane layout NV, step kind and target
// kind) and its host-side launch helpers: target-descriptor check, lane
// layout heuristic and launch. Shared by fmc_chains_mala.hip, fmc_chains_grw.hip,
// fmc_chains_hmc.hip (a unit or diagonal metric) and fmc_hmc_dense.hip (HMC with a dense
// condition matrix).
#pragma once

#include <type_traits>

#include "fmc_chain_steps.h"

namespace fmc {

// KK_HMC runs the unit and diagonal condition matrices; a dense condition
// matrix has a kernel of its own (KK_HMC_DENSE, built in fmc_hmc_dense.hip):
// its momentum product would otherwise raise every HMC kernel's register
// allocation (and lower its occupancy).
enum KernelKind { KK_MALA = 0, KK_HMC = 1, KK_GRW = 2, KK_HMC_DENSE = 3 };

// Bound by instruction issue: the state stays in registers, and rows leave at
// 5.2 TB/s at most. What a step costs is its VALU instructions (a MALA step of
// the 128-D Rosenbrock 350, of the 8-mode 64-D mixture 469) and, with few
// chains, the wait of a lone wavefront between them. us, the same calls with
// one kernel for all targets, parameters read from memory and runtime lane
// counts -> now: 1000 MALA steps of 1000 5-D dense-Gaussian chains 3133 -> 714;
// 64 of 16384 128-D Rosenbrock chains 237 -> 164; 100 tempered steps of 20480
// 64-D mixture rows 660 -> 370; 128 HMC steps of 2301 27-D Rosenbrock chains
// 9.6 -> 4.5 a step.
//
// One kernel per (lane layout NV, step kind, target kind TK, lanes per chain
// LPC): the target's value and gradient are inlined without a run-time
// dispatch, and with LPC > 0 (the default layouts, workgroups of at most 256
// threads) the group sums and broadcasts are straight-line DPP code and
// parameters are always staged in rows. LPC_RUN takes the lane count at run time
// and any workgroup up to 1024 threads (HMC keeps position, momentum, gradient,
// metric and the leapfrog copies in registers: bounded at 512 threads, which gives
// it 256 VGPRs instead of 128, where NV >= 2 spilled); four and more chunks a lane
// in workgroups of at most 256 threads have a kernel of their own (LPC_RUN256),
// which does not spill: 16 MALA steps of 2000
// 1500-D Rosenbrock chains 425 -> 182 us, of 5000 600-D diagonal Gaussian ones
// 204 -> 112.
//
// PAR: where the parameters are (a kernel for each: two or three copies of the
// step loop in one kernel shared its registers, and the largest layouts spilled
// more: MALA of a 600-D diagonal Gaussian took 1.5 times as long).
//
// RING: wavefront 0 advances the workgroup's 64 / lpc chains and the others
// draw its random numbers, a block of steps ahead, into LDS (use_ring has
// the rule).
enum { LPC_RUN = 0, LPC_RUN256 = -1 };
template <int NV, int KIND, int TK, int LPC, bool RING, int PAR>
__global__ void __launch_bounds__(LPC != LPC_RUN ? 256 : (KIND == KK_HMC || KIND == KK_HMC_DENSE) ? 512 : 1024)
chain_kernel(fmc_target tg, ChainIO io, StepCfg cfg, int lpc_rt, int dp, NoiseRing nr) {
  const int lpc = LPC > 0 ? LPC : lpc_rt;
  const TargetDev t{tg.kind, tg.n_dim, tg.n_modes, (gparam_t)tg.params, dp};
  if (PAR == PAR_ROWS) stage_target<TK>(t);
  if (PAR == PAR_RAW) stage_raw(t, (int)target_param_count(TK, t.d, t.K));
  const int lane = threadIdx.x & 63;
  const int r = lane & (lpc - 1);
  const int gbase = lane - r;
  int64_t c = (int64_t)blockIdx.x * (blockDim.x / lpc) + threadIdx.x / lpc;
  if constexpr (RING) {
    const int64_t c0 = (int64_t)blockIdx.x * (64 / lpc);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nblk = (nr.n_steps + ring_T<NV> - 1) / ring_T<NV>;
    constexpr uint32_t SN = KIND == KK_MALA ? RNG_MALA_NOISE : RNG_GRW_NOISE;
    constexpr uint32_t SU = KIND == KK_MALA ? RNG_MALA_UNIFORM : RNG_GRW_UNIFORM;
    if (wave > 0) {
      for (int b = 0; b < nblk; ++b) {
        fill_ring<NV>(io, nr, cfg, t.d, lpc, c0, b, wave - 1, (int)(blockDim.x >> 6) - 1, SN, SU);
        __syncthreads();  // block b full, block b - 1 consumed
      }
      return;
    }
    __syncthreads();
    c = c0 + lane / lpc;
  }
  if (c >= io.C) return;  // whole group leaves together
  using RG = std::conditional_t<LPC <= 0, RunLanes,
                                std::conditional_t<TK == FMC_TARGET_GAUSS_DENSE && LPC == 1 && NV <= 2, DenseRegs<NV>, NoRegs>>;
  if constexpr (KIND == KK_MALA)
    mala_group<NV, TK, PAR, RING, RG>(t, io, cfg, nr, c, r, lpc, gbase);
  else if constexpr (KIND == KK_GRW)
    grw_group<NV, TK, PAR, RING, RG>(t, io, cfg, nr, c, r, lpc, gbase);
  else if constexpr (KIND == KK_HMC_DENSE)
    hmc_group<NV, MK_DENSE, TK, PAR, RG>(t, io, cfg, c, r, lpc, gbase);
  else if (io.metric)
    hmc_group<NV, MK_DIAG, TK, PAR, RG>(t, io, cfg, c, r, lpc, gbase);
  else
    hmc_group<NV, MK_UNIT, TK, PAR, RG>(t, io, cfg, c, r, lpc, gbase);
}

// ----------------------------------------------------------- host side ----
static inline int check_target(const fmc_target* t) {
  FMC_ARG(t != nullptr, "target is NULL");
  FMC_ARG(t->n_dim >= 1, "target n_dim must be >= 1 (got %d)", t->n_dim);
  FMC_ARG(t->kind >= FMC_TARGET_GAUSS_DIAG && t->kind <= FMC_TARGET_DUAL_MOON, "unknown target kind %d",
          t->kind);
  if (t->kind == FMC_TARGET_GMM_DIAG) FMC_ARG(t->n_modes >= 1, "GMM target needs n_modes >= 1");
  if (t->kind == FMC_TARGET_DUAL_MOON) FMC_ARG(t->n_dim >= 2, "dual-moon target needs n_dim >= 2");
  int64_t need = target_param_count(t->kind, t->n_dim, t->n_modes);
  FMC_ARG(t->n_params >= need, "target kind %d with d=%d needs %lld params, got %lld", t->kind, t->n_dim,
          (long long)need, (long long)t->n_params);
  FMC_ARG(need == 0 || t->params != nullptr, "target params pointer is NULL");
  return FMC_OK;
}

struct Layout {
  int lpc, nv, block;
};

static inline bool is_pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }

// Heuristic lane layout: aim for ~4 dims per lane for long vectors (one float4
// chunk, so the fused step's register footprint stays small), but keep whole
// chains in one lane when d is tiny. Rosenbrock takes two chunks per lane: its
// three neighbour reads per chunk and the group sum amortise over twice the
// elements (d = 128: 16 x 2 beats 32 x 1 by 6 % for MALA and 7 % for GRW),
// while the mixture's per-mode loop is 8 % slower at two chunks per lane.
static inline Layout choose_layout(int d, int kind, const fmc_launch_cfg* cfg) {
  Layout L{0, 0, 256};
  if (cfg && cfg->lanes_per_chain > 0 && cfg->vec_per_lane > 0) {
    L.lpc = cfg->lanes_per_chain;
    L.nv = cfg->vec_per_lane;
  } else {
    int chunks = (d + 3) / 4;
    if (kind == FMC_TARGET_GAUSS_DENSE) {
      // O(d^2) gather: keep the chain in few lanes.
      L.lpc = 1;
      while (L.lpc * 8 < chunks) L.lpc *= 2;
      L.nv = (chunks + L.lpc - 1) / L.lpc;
    } else {
      const int per_lane = (kind == FMC_TARGET_ROSENBROCK) ? 2 : 1;
      L.lpc = 1;
      while (L.lpc * per_lane < chunks && L.lpc < 64) L.lpc *= 2;
      L.nv = (chunks + L.lpc - 1) / L.lpc;
    }
    if (L.nv > 2) L.nv = (L.nv <= 4) ? 4 : 8;
  }
  if (cfg && cfg->block_size > 0) L.block = cfg->block_size;
  return L;
}

static inline int check_layout(const Layout& L, int d) {
  FMC_ARG(is_pow2(L.lpc) && L.lpc <= 64, "lanes_per_chain must be a power of two <= 64 (got %d)", L.lpc);
  FMC_ARG(L.nv == 1 || L.nv == 2 || L.nv == 4 || L.nv == 8, "vec_per_lane must be 1, 2, 4 or 8 (got %d)",
          L.nv);
  FMC_ARG(4LL * L.nv * L.lpc >= d, "layout lanes_per_chain=%d vec_per_lane=%d holds %d dims < d=%d", L.lpc,
          L.nv, 4 * L.nv * L.lpc, d);
  FMC_ARG(L.block >= 64 && L.block <= 1024 && L.block % 64 == 0, "block_size must be a multiple of 64 in [64,1024]");
  return FMC_OK;
}

static inline bool raw_fits(const fmc_target* t) {
  return target_param_count(t->kind, t->n_dim, t->n_modes) * 4 <= 48 * 1024;
}
// How a layout stages the parameters: the stride of rows padded to the lanes'
// dims where they fit the 64 KB of LDS that need no attribute, STAGE_RAW where
// only the unpadded block fits 48 KB (the rows are up to twice as long: d = 65
// takes 128 dims a row), else STAGE_NONE. 32 MALA steps of 4096 chains, us,
// padded / unpadded / from memory: dense d = 100 1652 / 4883 / 9359, mixture d =
// 65 with 60 modes 542 / 715 / 1012, with 93 modes - / 1088 / 1563.
static inline int staged_stride(const fmc_target* t, const Layout& L) {
  const int dp = 4 * L.nv * L.lpc;
  const int64_t n = target_staged_count(t->kind, t->n_dim, t->n_modes, dp);
  if (n == 0) return STAGE_NONE;
  if (((n + 3) & ~3LL) * 4 <= 64 * 1024) return dp;
  return raw_fits(t) ? STAGE_RAW : STAGE_NONE;
}
// Where rows that are partly padding lose to the unpadded block: an explicit
// layout of mostly idle lanes, or more workgroups than the rows leave room for on
// the CUs (16 random-walk steps of 10,000 chains of a 300-D 8-mode mixture, 512
// dims a row: 329 / 285 us; of 1000 chains 70 / 82). Never for a few hundred
// floats (9 / 15 us a launch of a 100-D diagonal Gaussian over 256 dims) or, in
// the explicit layout, few wavefronts (64-D 8-mode mixture over 256 dims, random
// walks of 7 chains 35 / 58, of 1000 72 / 59).
static inline bool idle_lanes(const fmc_target* t, const Layout& L, int dp, int64_t n) {
  return t->kind != FMC_TARGET_GAUSS_DENSE && dp > 2 * t->n_dim + 8 && n * L.lpc > 64 * 256 &&
         target_staged_count(t->kind, t->n_dim, t->n_modes, dp) > 1024;
}
static inline bool rows_cost_more(const fmc_target* t, const Layout& L, int dp, int64_t n) {
  if (t->kind == FMC_TARGET_GAUSS_DENSE || 4 * dp <= 5 * t->n_dim) return false;
  if (idle_lanes(t, L, dp, n)) return true;
  const int64_t bytes = 4 * target_staged_count(t->kind, t->n_dim, t->n_modes, dp), per = L.block / L.lpc;
  return bytes > 4096 && (n + per - 1) / per > 256 * (160 * 1024 / bytes);
}
static inline int staged_floats(const fmc_target* t, int dp) {
  if (dp == STAGE_NONE) return 0;
  return (int)(((dp > 0 ? target_staged_count(t->kind, t->n_dim, t->n_modes, dp)
                        : target_param_count(t->kind, t->n_dim, t->n_modes)) + 3) & ~3LL);
}

// Whether a workgroup is one chain wavefront and three that draw its random
// numbers, or four that draw their own. A lone wavefront on a SIMD issues an instruction every
// ~6.5 clocks (4 with company), and the Philox draws are half of a small
// target's step: while the chains fill at most one wavefront a SIMD (1024), the
// idle issue slots take them over. us a step, without / with the ring: MALA
// dense Gaussian d = 5, C = 1000 (16 wavefronts) 1.29 / 0.76, d = 12, C = 1000
// 3.16 / 2.32; funnel d = 7, C = 1343 0.90 / 0.54; Rosenbrock d = 128, C = 500
// (125) 1.22 / 0.81, C = 4096 (1024) 1.32 / 1.15; mixture d = 64, C = 500 2.07 /
// 1.85. Above, the SIMDs are full and the ring only adds LDS traffic: funnel
// d = 100, C = 4000 (2000) 1.01 / 1.24, Rosenbrock d = 128, C = 16384 (4096)
// 2.80 / 4.18. More than three filling wavefronts give nothing (0.93 -> 0.92).
// The launch stays within the 64 KB of LDS that need no attribute: a mixture's
// staged parameters can leave no room for the ring.
constexpr int RING_MAX_WAVES = 1024;
constexpr size_t RING_MAX_LDS = 64 * 1024;

template <int NV>
static size_t ring_bytes(int lpc) { return 4 * 2 * (size_t)ring_T<NV> * (NV * 256 + 64 / lpc); }

template <int NV>
static bool use_ring(const ChainIO& io, const StepCfg& cfg, const Layout& L, int staged) {
  return !io.noise && !io.log_u && L.block == 256 && cfg.n_steps >= 8 &&
         (io.C * L.lpc + 63) / 64 <= RING_MAX_WAVES && 4 * (size_t)staged + ring_bytes<NV>(L.lpc) <= RING_MAX_LDS;
}

template <int NV, int KIND, int TK, int LPC, int PAR>
static void launch_chain_par(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg,
                             const Layout& L, int dp) {
  const int nf = staged_floats(t, dp);
  const NoiseRing nr{nf, cfg.n_steps};
  if constexpr (LPC > 0 && (KIND == KK_MALA || KIND == KK_GRW)) {
    if (use_ring<NV>(io, cfg, L, nf)) {
      const int per_block = 64 / LPC;
      hipLaunchKernelGGL((chain_kernel<NV, KIND, TK, LPC, true, PAR>),
                         dim3((unsigned)((io.C + per_block - 1) / per_block)), dim3(256),
                         4 * (size_t)nf + ring_bytes<NV>(LPC), st, *t, io, cfg, L.lpc, dp, nr);
      return;
    }
  }
  const int per_block = L.block / L.lpc;
  hipLaunchKernelGGL((chain_kernel<NV, KIND, TK, LPC, false, PAR>), dim3((unsigned)((io.C + per_block - 1) / per_block)),
                     dim3((unsigned)L.block), 4 * (size_t)nf, st, *t, io, cfg, L.lpc, dp, nr);
}

// (LPC > 0: parameters are staged in rows, if the target has any)
template <int NV, int KIND, int TK, int LPC>
static void launch_chain_lpc(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg,
                             const Layout& L, int dp) {
  if constexpr (TK == FMC_TARGET_ROSENBROCK || TK == FMC_TARGET_FUNNEL) {
    launch_chain_par<NV, KIND, TK, LPC, PAR_MEM>(st, t, io, cfg, L, dp);
  } else if constexpr (LPC > 0) {
    launch_chain_par<NV, KIND, TK, LPC, PAR_ROWS>(st, t, io, cfg, L, dp);
  } else {
    // (the rows' loads move out of the step loop, and the 1024-thread kernels
    // that hold most else have no registers for them: MALA of a 600-D diagonal
    // Gaussian, four chunks, 201 us, unpadded 117; random-walk steps of a 1500-D
    // one, eight, 149 / 95)
    constexpr bool ROWS = LPC == LPC_RUN256 || TK == FMC_TARGET_GAUSS_DENSE || KIND == KK_HMC || KIND == KK_HMC_DENSE ||
                          NV < 4 || (NV == 4) == (KIND == KK_GRW);
    if (dp > 0 && (!ROWS || rows_cost_more(t, L, dp, io.C))) dp = raw_fits(t) ? STAGE_RAW : ROWS ? dp : STAGE_NONE;
    if constexpr (ROWS) {
      if (dp > 0) {
        launch_chain_par<NV, KIND, TK, LPC, PAR_ROWS>(st, t, io, cfg, L, dp);
        return;
      }
    }
    if (dp == STAGE_RAW)
      launch_chain_par<NV, KIND, TK, LPC, PAR_RAW>(st, t, io, cfg, L, dp);
    else
      launch_chain_par<NV, KIND, TK, LPC, PAR_MEM>(st, t, io, cfg, L, dp);
  }
}

// Four and eight chunks a lane: workgroups of at most 256 threads without spills
// where that pays, MALA and, at eight, random-walk steps (random-walk steps of
// 5000 600-D diagonal Gaussian chains, four chunks, 75 -> 82 us; HMC and a dense
// precision need the second wavefront on a SIMD more: HMC of 2000 1500-D Rosenbrock
// chains 107 -> 158 us).
template <int NV, int KIND, int TK>
static void launch_chain_wide(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg,
                              const Layout& L, int dp) {
  if constexpr ((KIND == KK_MALA || (KIND == KK_GRW && NV == 8)) && TK != FMC_TARGET_GAUSS_DENSE) {
    if (L.block <= 256) {
      launch_chain_lpc<NV, KIND, TK, LPC_RUN256>(st, t, io, cfg, L, dp);
      return;
    }
  }
  launch_chain_lpc<NV, KIND, TK, LPC_RUN>(st, t, io, cfg, L, dp);
}

// The kernels specialised on their lane count: the layouts choose_layout gives
// to up to 256 dims (512 for Rosenbrock, 32 for a dense Gaussian).
template <int KIND, int TK>
static void launch_chain_kind(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg,
                              const Layout& L) {
  const int dp = staged_stride(t, L);
  if constexpr (KIND != KK_HMC_DENSE) {
    // (an explicit layout of mostly idle lanes stages its parameters unpadded)
    const bool staged = TK == FMC_TARGET_ROSENBROCK || TK == FMC_TARGET_FUNNEL || (dp > 0 && !idle_lanes(t, L, dp, io.C));
    if (staged && L.block <= 256) {
#define FMC_LPC(NV_, LPC_)                                                      \
  case LPC_:                                                                    \
    launch_chain_lpc<NV_, KIND, TK, LPC_>(st, t, io, cfg, L, dp);               \
    return;
      constexpr int NVD = TK == FMC_TARGET_ROSENBROCK ? 2 : 1;  // chunks a lane holds by default
      if constexpr (TK == FMC_TARGET_GAUSS_DENSE) {
        if (L.lpc == 1) {
          switch (L.nv) {
            case 1: launch_chain_lpc<1, KIND, TK, 1>(st, t, io, cfg, L, dp); return;
            case 2:
              if (t->n_dim <= 4) break;  // (registers: no chunk of padding only)
              launch_chain_lpc<2, KIND, TK, 1>(st, t, io, cfg, L, dp);
              return;
            case 4: launch_chain_lpc<4, KIND, TK, 1>(st, t, io, cfg, L, dp); return;
            default: break;
          }
        }
      } else {
        if (TK == FMC_TARGET_ROSENBROCK && L.nv == 1 && L.lpc == 1) {
          launch_chain_lpc<1, KIND, TK, 1>(st, t, io, cfg, L, dp);
          return;
        }
        if (L.nv == NVD) {
          switch (L.lpc) {
            FMC_LPC(NVD, 1)
            FMC_LPC(NVD, 2)
            FMC_LPC(NVD, 4)
            FMC_LPC(NVD, 8)
            FMC_LPC(NVD, 16)
            FMC_LPC(NVD, 32)
            FMC_LPC(NVD, 64)
            default: break;
          }
        }
      }
#undef FMC_LPC
    }
  }
  switch (L.nv) {
    case 1: launch_chain_lpc<1, KIND, TK, LPC_RUN>(st, t, io, cfg, L, dp); break;
    case 2: launch_chain_lpc<2, KIND, TK, LPC_RUN>(st, t, io, cfg, L, dp); break;
    case 4: launch_chain_wide<4, KIND, TK>(st, t, io, cfg, L, dp); break;
    default: launch_chain_wide<8, KIND, TK>(st, t, io, cfg, L, dp); break;
  }
}

template <int KIND>
static int launch_chain_impl(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg,
                             const Layout& L) {
  FMC_ARG((KIND != KK_HMC && KIND != KK_HMC_DENSE) || L.block <= 512,
          "fused HMC launches take at most 512 threads per workgroup (got %d)", L.block);
  FMC_ARG((io.C * L.lpc + 63) / 64 <= 0x7fffffffLL, "too many chains for one launch");
  switch (t->kind) {  // check_target has accepted the kind
    case FMC_TARGET_GAUSS_DIAG: launch_chain_kind<KIND, FMC_TARGET_GAUSS_DIAG>(st, t, io, cfg, L); break;
    case FMC_TARGET_GAUSS_DENSE: launch_chain_kind<KIND, FMC_TARGET_GAUSS_DENSE>(st, t, io, cfg, L); break;
    case FMC_TARGET_ROSENBROCK: launch_chain_kind<KIND, FMC_TARGET_ROSENBROCK>(st, t, io, cfg, L); break;
    case FMC_TARGET_FUNNEL: launch_chain_kind<KIND, FMC_TARGET_FUNNEL>(st, t, io, cfg, L); break;
    case FMC_TARGET_GMM_DIAG: launch_chain_kind<KIND, FMC_TARGET_GMM_DIAG>(st, t, io, cfg, L); break;
    default: launch_chain_kind<KIND, FMC_TARGET_DUAL_MOON>(st, t, io, cfg, L); break;
  }
  return check_launch(KIND == KK_MALA ? "mala chain kernel" : KIND == KK_GRW ? "grw chain kernel" : "hmc chain kernel");
}

// One translation unit per step kind (they build in parallel).
int launch_mala(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg, const Layout& L);
int launch_grw(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg, const Layout& L);
int launch_hmc(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg, const Layout& L);
// Fused HMC with a dense condition matrix (defined in fmc_hmc_dense.hip).
int launch_hmc_dense(hipStream_t st, const fmc_target* t, const ChainIO& io, const StepCfg& cfg, const Layout& L);

}  // namespace fmc
