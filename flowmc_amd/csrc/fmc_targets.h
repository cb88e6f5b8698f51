// Built-in log-densities: value and hand-written gradient, evaluated by the
// lanes of one chain group.
//
// Lane layout: a chain is held by `lpc` consecutive lanes (lane r = 0..lpc-1
// of the group whose first lane is `gbase`); lane r holds NV float4 chunks,
// element e of chunk v being dimension  j = (v*lpc + r)*4 + e  (j >= d is
// padding and must hold 0, and its gradient is 0). Every function returns the full log-density in
// every lane of the group and writes the lane's gradient chunks.
//
// Sums of products are written as the FMAs they run as, so that every kernel
// that inlines a target (fused, batched, per-step evaluation) rounds alike,
// with one exception: the funnel's evaluation at the entry of a MALA or
// random-walk launch (ENTRY) adds two squares in the other order.
//
// These replace jax.value_and_grad(logpdf) of the user target at
// src/flowMC/resource/kernel/MALA.py:59 and jax.grad(potential) at
// src/flowMC/resource/kernel/HMC.py:75-77 for the targets listed in
// include/flowmc.h.
#pragma once

#include <type_traits>

#include "fmc_common.h"

namespace fmc {

// Parameters in global memory (an explicit address space: a generic pointer
// would make every access a FLAT one), or staged in LDS by stage_target.
typedef const __attribute__((address_space(1))) float* gparam_t;
extern __shared__ float fmc_chain_lds[];

struct TargetDev {
  int kind;
  int d;
  int K;           // modes (GMM)
  gparam_t p;      // parameter block
  int dp;          // row stride of the padded staged copy (the dims the lanes of a group hold), or STAGE_*
};

__device__ __forceinline__ int dim_of(int v, int e, int r, int lpc) { return (v * lpc + r) * 4 + e; }

// Where a kernel reads the parameters: memory, LDS rows padded to the lanes'
// dims, or an unpadded LDS copy, for parameters that fit the LDS only so.
enum { PAR_MEM = 0, PAR_ROWS = 1, PAR_RAW = 2 };
constexpr int STAGE_NONE = 0, STAGE_RAW = -1;

// Parameter i of the block (not of padded rows)
template <int PAR>
__device__ __forceinline__ float param(const TargetDev& t, int64_t i) {
  return PAR == PAR_RAW ? fmc_chain_lds[i] : t.p[i];
}

// Four consecutive parameters of a staged row (LDS; zero past the dims)
__device__ __forceinline__ float4 staged4(int off) { return *reinterpret_cast<const float4*>(fmc_chain_lds + off); }

template <int NV, int PAR>
__device__ __forceinline__ float tgt_gauss_diag(const TargetDev& t, const float4 (&x)[NV],
                                                float4 (&g)[NV], int r, int lpc) {
  float acc = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    float4 m4, p4;
    if (PAR == PAR_ROWS) {
      m4 = staged4(dim_of(v, 0, r, lpc));
      p4 = staged4(t.dp + dim_of(v, 0, r, lpc));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int j = dim_of(v, e, r, lpc);
      float gj = 0.f;
      if (PAR == PAR_ROWS || j < t.d) {
        float y = f4c(x[v], e) - (PAR == PAR_ROWS ? f4c(m4, e) : param<PAR>(t, j));
        float pr = PAR == PAR_ROWS ? f4c(p4, e) : param<PAR>(t, t.d + j);
        gj = -pr * y;
        acc = fmaf(0.5f * gj, y, acc);
      }
      f4(g[v], e) = gj;
    }
  }
  return group_sum(acc, lpc);
}

// Staged: mean, then the precision transposed row by row (row j2 holds P[j][j2]
// for all j, zero-padded to the dims of the lane group), so that a lane reads
// its dims of one column as float4 without an index test. With one lane a
// chain every lane reads the same address (an LDS broadcast); up to 8 dims are
// held in registers over the steps (DenseRegs: an LDS read a column was 5 round
// trips a step at d = 5).
template <int NV>
struct DenseRegs {
  float4 m[NV], P[4 * NV][NV];
  __device__ __forceinline__ explicit DenseRegs(const TargetDev& t) {
#pragma unroll
    for (int v = 0; v < NV; ++v) m[v] = staged4(4 * v);
#pragma unroll
    for (int j = 0; j < 4 * NV; ++j)
#pragma unroll
      for (int v = 0; v < NV; ++v) P[j][v] = j < t.d ? staged4(t.dp * (j + 1) + 4 * v) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
};
struct NoRegs {
  __device__ __forceinline__ explicit NoRegs(const TargetDev&) {}
};
// ... and a lane count that is known at run time only
struct RunLanes {
  __device__ __forceinline__ explicit RunLanes(const TargetDev&) {}
};

template <int NV, int PAR, class RG>
__device__ __forceinline__ float tgt_gauss_dense(const TargetDev& t, const RG& rg, const float4 (&x)[NV],
                                                 float4 (&g)[NV], int r, int lpc, int gbase) {
  constexpr bool REG = std::is_same<RG, DenseRegs<NV>>::value;
  const int d = t.d;
  float4 y[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    float4 m4;
    if constexpr (REG) m4 = rg.m[v];
    else if (PAR == PAR_ROWS) m4 = staged4(dim_of(v, 0, r, lpc));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int j = dim_of(v, e, r, lpc);
      if (PAR == PAR_ROWS)
        f4(y[v], e) = f4c(x[v], e) - f4c(m4, e);
      else
        f4(y[v], e) = (j < d) ? f4c(x[v], e) - param<PAR>(t, j) : 0.f;
      f4(g[v], e) = 0.f;
    }
  }
  // g_i = -sum_j P_ij y_j; y_j gathered from the lane that owns it.
  for (int s = 0; s < (REG ? 1 : lpc); ++s) {
#pragma unroll
    for (int v2 = 0; v2 < NV; ++v2)
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        const int j2 = REG ? 4 * v2 + e2 : dim_of(v2, e2, s, lpc);
        // (in registers by two columns: a zero column costs less than its test)
        float ys = 0.f;  // (from memory the shuffle ahead of the test: HMC, d = 200, 13.2 / 12.6 ms)
        if (PAR == PAR_MEM) ys = __shfl(f4c(y[v2], e2), gbase + s, 64);
        if ((REG ? j2 & ~1 : j2) < d) {
          if (PAR != PAR_MEM) ys = (REG || lpc == 1) ? f4c(y[v2], e2) : __shfl(f4c(y[v2], e2), gbase + s, 64);
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            float4 p4;
            if constexpr (REG) p4 = rg.P[4 * v2 + e2][v];
            else if (PAR == PAR_ROWS) p4 = staged4(t.dp * (j2 + 1) + dim_of(v, 0, r, lpc));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              int j = dim_of(v, e, r, lpc);
              if (PAR == PAR_ROWS)
                f4(g[v], e) = fmaf(-f4c(p4, e), ys, f4c(g[v], e));
              else if (j < d)
                f4(g[v], e) = fmaf(-param<PAR>(t, d + (int64_t)j * d + j2), ys, f4c(g[v], e));
            }
          }
        }
      }
  }
  float acc = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // (a padding row's zeros make a NaN of an infinite y; parameters in
      // registers have padding in their last chunk only)
      if (PAR == PAR_ROWS && (!REG || (v == NV - 1 && e > 0)) && dim_of(v, e, r, lpc) >= d) f4(g[v], e) = 0.f;
      acc = fmaf(0.5f * f4c(y[v], e), f4c(g[v], e), acc);
    }
  return group_sum(acc, lpc);
}

// x of the next / previous lane of the wavefront, on the VALU (row shifts
// stay inside a group of at most 16 lanes; wave shifts above); the lanes at a
// group's ends take their neighbour elsewhere.
__device__ __forceinline__ float lane_next(float v, int lpc) {
  return lpc <= 16 ? dpp_all<0x101>(v) : dpp_all<0x130>(v);  // row_shl:1 / wave_shl:1
}
__device__ __forceinline__ float lane_prev(float v, int lpc) {
  return lpc <= 16 ? dpp_all<0x111>(v) : dpp_all<0x138>(v);  // row_shr:1 / wave_shr:1
}
// in the group's first lane: the value of its last lane
__device__ __forceinline__ float group_last_to_first(float v, int lpc) {
  if (lpc == 1) return v;
  if (lpc == 2) return dpp_all<DPP_XOR1>(v);
  if (lpc == 4) return dpp_all<0x1B>(v);  // quad_perm [3,2,1,0]
  if (lpc == 8) return dpp_all<DPP_HALF_MIRROR>(v);
  if (lpc == 64) return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
  const float m = dpp_all<DPP_MIRROR>(v);
  if (lpc == 16) return m;
  float lo, hi;
  swap16(m, lo, hi);
  return hi;  // lane 0 of a 32-lane half: lane 0 of its second row, which mirrored lane 31
}

// log p = -scale * sum_{i<d-1} [100 (x_{i+1} - x_i^2)^2 + (1 - x_i)^2]
// RUN: a run-time lane count reads its neighbours by shuffles (a branch on it
// for each read made HMC of d = 700 up to 1.2 times slower)
template <int NV, bool RUN>
__device__ __forceinline__ float tgt_rosenbrock(const TargetDev& t, const float4 (&x)[NV],
                                                float4 (&g)[NV], int r, int lpc, int gbase) {
  const float scale = t.p[0];
  const int d = t.d;
  float acc = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    // x_{j+1} for element 3 and x_{j-1} for element 0 live in neighbouring lanes.
    float nx_same = RUN ? __shfl(x[v].x, gbase + ((r + 1) & (lpc - 1)), 64) : lane_next(x[v].x, lpc);
    float nx_next = group_bcast0(x[(v + 1 < NV) ? v + 1 : v].x, lpc);
    float pw_same = RUN ? __shfl(x[v].w, gbase + ((r - 1) & (lpc - 1)), 64) : lane_prev(x[v].w, lpc);
    const float last = x[(v > 0) ? v - 1 : 0].w;
    float pw_prev = RUN ? __shfl(last, gbase + lpc - 1, 64) : group_last_to_first(last, lpc);
    float nxt3 = (r < lpc - 1) ? nx_same : nx_next;
    float prv0 = (r > 0) ? pw_same : pw_prev;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int j = dim_of(v, e, r, lpc);
      float xi = f4c(x[v], e);
      float xn = (e < 3) ? f4c(x[v], e + 1) : nxt3;
      float xp = (e > 0) ? f4c(x[v], e - 1) : prv0;
      float gi = 0.f;
      if (j < d - 1) {
        const float tt = fmaf(-xi, xi, xn);
        const float om = 1.f - xi;
        acc += fmaf(om, om, 100.f * tt * tt);
        gi = fmaf(-400.f * xi, tt, -2.f * om);
      }
      if (j > 0 && j < d) gi = fmaf(200.f, fmaf(-xp, xp, xi), gi);
      f4(g[v], e) = -scale * gi;
    }
  }
  return -scale * group_sum(acc, lpc);
}

// Neal's funnel: x_0 = v ~ N(0, 3^2), x_i | v ~ N(0, e^v) (unnormalised).
// Padding elements (j >= d) hold 0 on entry, so they add nothing to the sum
// and get a zero gradient without a per-element index test; only element 0
// of the group's first lane (v itself) is special. exp(-v) is capped at
// FLT_MAX so that 0 * exp(-v) stays 0 on padding when e^-v overflows.
// ENTRY (the evaluation at the entry of a MALA / random-walk launch): the
// first two squares are added the other way round, as in every release so far.
template <int NV, bool ENTRY>
__device__ __forceinline__ float tgt_funnel(const TargetDev& t, const float4 (&x)[NV],
                                            float4 (&g)[NV], int r, int lpc, int gbase) {
  const int d = t.d;
  const float v0 = group_bcast0(x[0].x, lpc);
  const float x00 = (r == 0) ? 0.f : x[0].x;
  float s = ENTRY ? fmaf(x00, x00, x[0].y * x[0].y) : fmaf(x[0].y, x[0].y, x00 * x00);
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = (v == 0) ? 2 : 0; e < 4; ++e) s = fmaf(f4c(x[v], e), f4c(x[v], e), s);
  s = group_sum(s, lpc);
  const float em = fminf(expf(-v0), 3.402823466e38f);
  const float nm1 = (float)(d - 1);
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) f4(g[v], e) = -f4c(x[v], e) * em;
  const float g0 = fmaf(0.5f * em, s, fmaf(v0, -1.f / 9.f, -0.5f * nm1));
  if (r == 0) g[0].x = g0;
  return fmaf(-0.5f * em, s, fmaf(v0 * v0, -1.f / 18.f, -(0.5f * nm1 * v0)));
}

// Diagonal Gaussian mixture: log p = logsumexp_k [ c_k - 1/2 sum_j ((x_j - mu_kj) / s_kj)^2 ]
// with c_k = log w_k - sum_j log s_kj. Online softmax over modes, without a
// branch on the lanes: with e = exp(-|q - m|) a new largest mode scales what
// was summed by e and adds itself once, another adds itself e times (the same
// FMAs, their operands selected). Where e underflows to 0 for every chain of
// the wavefront (modes a few sigma apart in many dims), the mode replaces the
// sums or leaves them alone: no exponential, and its gradient is only formed
// if it is some chain's largest so far (d = 64, 8 modes, 16 lanes a chain: 624
// -> 469 VALU instructions a MALA step). Two modes' forms are summed
// together: their loads and lane sums overlap (20480 tempered rows, 100 steps:
// 442 -> 420 us, 500 chains 2.1 -> 1.84 us a step; four together take the
// registers of the fifth wavefront on a SIMD, 487 us).
template <int NV, int PAR>
__device__ __forceinline__ float tgt_gmm_diag(const TargetDev& t, const float4 (&x)[NV],
                                              float4 (&g)[NV], int r, int lpc) {
  const int d = t.d, K = t.K;
  const int o_is = K * t.dp, o_c = 2 * K * t.dp;  // staged: mu [K][dp], 1 / s [K][dp], c [K]
  float m = -INFINITY, sw = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) g[v] = make_float4(0.f, 0.f, 0.f, 0.f);
  // U modes' quadratic forms at once: their loads and sums over the lanes overlap
  constexpr int U = PAR != PAR_MEM && NV <= 2 ? 2 : 1;
  if constexpr (U == 1) {
    // many chunks a lane, or parameters in memory: one mode at a time, its
    // gradient the only copy of it (the form above took twice the registers and
    // spilled: MALA of a 1100-D mixture 2.0 times as long), a branch on the chain
    for (int k = 0; k < K; ++k) {
      float4 gk[NV];
      float q = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = dim_of(v, e, r, lpc);
          float gj = 0.f;
          if (PAR == PAR_ROWS || j < d) {
            const float is = PAR == PAR_ROWS ? fmc_chain_lds[o_is + k * t.dp + j] : param<PAR>(t, (int64_t)(K + k) * d + j);
            const float mu = PAR == PAR_ROWS ? fmc_chain_lds[k * t.dp + j] : param<PAR>(t, (int64_t)k * d + j);
            const float z = (f4c(x[v], e) - mu) * is;
            q = fmaf(z, z, q);
            gj = -z * is;
          }
          f4(gk[v], e) = gj;
        }
      q = fmaf(-0.5f, group_sum(q, lpc), PAR == PAR_ROWS ? fmc_chain_lds[o_c + k] : param<PAR>(t, 2 * (int64_t)K * d + k));
      if (q > m) {  // (q is bitwise equal across the group)
        const float sc = expf(m - q);
        sw = fmaf(sw, sc, 1.f);
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) f4(g[v], e) = fmaf(f4c(g[v], e), sc, f4c(gk[v], e));
        m = q;
      } else {
        const float w = expf(q - m);
        sw += w;
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
          for (int e = 0; e < 4; ++e) f4(g[v], e) = fmaf(w, f4c(gk[v], e), f4c(g[v], e));
      }
    }
  } else {
    for (int k0 = 0; k0 < K; k0 += U) {
      float4 z[U][NV], i4[U][NV];
      float qs[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u < K ? k0 + u : k0;
        float q = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          float4 m4;
          if (PAR == PAR_ROWS) {
            m4 = staged4(k * t.dp + dim_of(v, 0, r, lpc));
            i4[u][v] = staged4(o_is + k * t.dp + dim_of(v, 0, r, lpc));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int j = dim_of(v, e, r, lpc);
              f4(m4, e) = j < d ? param<PAR>(t, (int64_t)k * d + j) : 0.f;
              f4(i4[u][v], e) = j < d ? param<PAR>(t, (int64_t)(K + k) * d + j) : 0.f;
            }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f4(z[u][v], e) = (f4c(x[v], e) - f4c(m4, e)) * f4c(i4[u][v], e);
            q = fmaf(f4c(z[u][v], e), f4c(z[u][v], e), q);
          }
        }
        qs[u] = q;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u < K ? k0 + u : k0;
        qs[u] = fmaf(-0.5f, group_sum(qs[u], lpc), PAR == PAR_ROWS ? fmc_chain_lds[o_c + k] : param<PAR>(t, 2 * (int64_t)K * d + k));
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + u >= K) break;
        const float q = qs[u];
        const bool top = q > m;
        const float a = fabsf(q - m);
        // (expf gives 0 below -103.97; not for a NaN)
        if (__builtin_amdgcn_ballot_w64(!(a > 104.f)) == 0) {
          if (__builtin_amdgcn_ballot_w64(top) != 0) {
            sw = top ? 1.f : sw;
#pragma unroll
            for (int v = 0; v < NV; ++v)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                f4(g[v], e) = top ? -f4c(z[u][v], e) * f4c(i4[u][v], e) : f4c(g[v], e);
            m = top ? q : m;
          }
        } else {
          const float w = expf(-a);
          sw = fmaf(top ? sw : 1.f, w, top ? 1.f : sw);
#pragma unroll
          for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float gk = -f4c(z[u][v], e) * f4c(i4[u][v], e);
              f4(g[v], e) = fmaf(top ? f4c(g[v], e) : gk, w, top ? gk : f4c(g[v], e));
            }
          m = top ? q : m;
        }
      }
    }
  }
  float inv = 1.f / sw;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) f4(g[v], e) *= inv;
  return m + logf(sw);
}

// Dual moon (docs/tutorials/dualmoon.ipynb, test/integration/test_MALA.py:11-20):
// log p = -50 (|x - center| - 2)^2 + LSE_a(-(x0 + a)^2 / (2*0.8^2)) + LSE_a(-(x1 + a)^2 / (2*0.6^2)),
// a in {-3, +3}. Requires d >= 2.
template <int NV, int PAR>
__device__ __forceinline__ float tgt_dual_moon(const TargetDev& t, const float4 (&x)[NV],
                                               float4 (&g)[NV], int r, int lpc, int gbase) {
  const int d = t.d;
  float4 ctr[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (PAR == PAR_ROWS) {
      ctr[v] = staged4(dim_of(v, 0, r, lpc));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) f4(ctr[v], e) = dim_of(v, e, r, lpc) < d ? param<PAR>(t, dim_of(v, e, r, lpc)) : 0.f;
    }
  }
  float n2 = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int j = dim_of(v, e, r, lpc);
      if (j < d) {
        float y = f4c(x[v], e) - f4c(ctr[v], e);
        n2 = fmaf(y, y, n2);
      }
    }
  n2 = group_sum(n2, lpc);
  float n = sqrtf(n2);
  float x0 = group_bcast0(x[0].x, lpc);
  float x1 = group_bcast0(x[0].y, lpc);
  // logsumexp pieces
  float a0 = -0.5f * ((x0 - 3.f) / 0.8f) * ((x0 - 3.f) / 0.8f);
  float b0 = -0.5f * ((x0 + 3.f) / 0.8f) * ((x0 + 3.f) / 0.8f);
  float m0 = fmaxf(a0, b0);
  float ea0 = expf(a0 - m0), eb0 = expf(b0 - m0);
  float l0 = m0 + logf(ea0 + eb0);
  float a1 = -0.5f * ((x1 - 3.f) / 0.6f) * ((x1 - 3.f) / 0.6f);
  float b1 = -0.5f * ((x1 + 3.f) / 0.6f) * ((x1 + 3.f) / 0.6f);
  float m1 = fmaxf(a1, b1);
  float ea1 = expf(a1 - m1), eb1 = expf(b1 - m1);
  float l1 = m1 + logf(ea1 + eb1);
  float t1 = (n - 2.f) / 0.1f;
  float radial = -100.f * (n - 2.f) / n;  // d/dx_j of -50 (n-2)^2 is radial * y_j
  float g0 = (ea0 * (-(x0 - 3.f)) + eb0 * (-(x0 + 3.f))) / ((ea0 + eb0) * 0.64f);
  float g1 = (ea1 * (-(x1 - 3.f)) + eb1 * (-(x1 + 3.f))) / ((ea1 + eb1) * 0.36f);
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int j = dim_of(v, e, r, lpc);
      float gj = 0.f;
      if (j < d) {
        gj = radial * (f4c(x[v], e) - f4c(ctr[v], e));
        if (j == 0) gj += g0;
        if (j == 1) gj += g1;
      }
      f4(g[v], e) = gj;
    }
  return -(0.5f * t1 * t1 - l0 - l1);
}

// TK >= 0: the kind is fixed at compile time (one target per kernel);
// TK = -1: dispatch on t.kind at run time. PAR: where the parameters are
// (stage_target, stage_raw).
// RG: parameters held in registers (DenseRegs), or NoRegs; RunLanes where lpc
// is no compile-time constant.
template <int NV, int TK, int PAR, bool ENTRY, class RG>
__device__ __forceinline__ float target_vg(const TargetDev& t, const RG& rg, const float4 (&x)[NV],
                                           float4 (&g)[NV], int r, int lpc, int gbase) {
  switch (TK >= 0 ? TK : t.kind) {
    case FMC_TARGET_GAUSS_DIAG:
      return tgt_gauss_diag<NV, PAR>(t, x, g, r, lpc);
    case FMC_TARGET_GAUSS_DENSE:
      return tgt_gauss_dense<NV, PAR>(t, rg, x, g, r, lpc, gbase);
    case FMC_TARGET_ROSENBROCK:
      return tgt_rosenbrock<NV, std::is_same<RG, RunLanes>::value>(t, x, g, r, lpc, gbase);
    case FMC_TARGET_FUNNEL:
      return tgt_funnel<NV, ENTRY>(t, x, g, r, lpc, gbase);
    case FMC_TARGET_GMM_DIAG:
      return tgt_gmm_diag<NV, PAR>(t, x, g, r, lpc);
    case FMC_TARGET_DUAL_MOON:
    default:
      return tgt_dual_moon<NV, PAR>(t, x, g, r, lpc, gbase);
  }
}

// Floats of the staged parameters of a kind for lane groups holding dp dims.
inline int64_t target_staged_count(int kind, int d, int K, int dp) {
  switch (kind) {
    case FMC_TARGET_GAUSS_DIAG: return 2LL * dp;
    case FMC_TARGET_GAUSS_DENSE: return (int64_t)dp * (d + 1);
    case FMC_TARGET_GMM_DIAG: return 2LL * K * dp + K;
    case FMC_TARGET_DUAL_MOON: return dp;
    default: return 0;  // Rosenbrock's scale is one scalar load, the funnel has none
  }
}

// Copies the parameters of kind TK to LDS rows of dp dims (the whole workgroup).
template <int TK>
__device__ __forceinline__ void stage_target(const TargetDev& t) {
  const int d = t.d, dp = t.dp;
  const int rows = TK == FMC_TARGET_GAUSS_DIAG ? 2 : TK == FMC_TARGET_GAUSS_DENSE ? d + 1
                   : TK == FMC_TARGET_GMM_DIAG ? 2 * t.K : TK == FMC_TARGET_DUAL_MOON ? 1 : 0;
  const int sh = __builtin_ctz(dp);  // (a power of two)
  for (int i = threadIdx.x; i < rows * dp; i += blockDim.x) {
    const int w = i >> sh, j = i & (dp - 1);
    float v = 0.f;
    if (j < d) v = (TK == FMC_TARGET_GAUSS_DENSE && w > 0) ? t.p[d + (int64_t)j * d + (w - 1)] : t.p[(int64_t)w * d + j];
    fmc_chain_lds[i] = v;
  }
  if (TK == FMC_TARGET_GMM_DIAG)
    for (int k = threadIdx.x; k < t.K; k += blockDim.x) fmc_chain_lds[rows * dp + k] = t.p[2 * (int64_t)t.K * d + k];
  __syncthreads();
}

// Copies the n parameters to LDS as they are (the whole workgroup).
__device__ __forceinline__ void stage_raw(const TargetDev& t, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) fmc_chain_lds[i] = t.p[i];
  __syncthreads();
}

// Number of floats of the parameter block of each kind (host check).
__host__ __device__ inline int64_t target_param_count(int kind, int d, int K) {
  switch (kind) {
    case FMC_TARGET_GAUSS_DIAG: return 2LL * d;
    case FMC_TARGET_GAUSS_DENSE: return (int64_t)d + (int64_t)d * d;
    case FMC_TARGET_ROSENBROCK: return 1;
    case FMC_TARGET_FUNNEL: return 0;
    case FMC_TARGET_GMM_DIAG: return 2LL * K * d + K;
    case FMC_TARGET_DUAL_MOON: return d;
    default: return -1;
  }
}

}  // namespace fmc
