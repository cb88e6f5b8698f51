// Fused chain steps shared by the chain kernels (fmc_chains.hip) and the
// batched uneven-dimension HMC kernel (fmc_hmc_batched.hip): buffer I/O of a
// chain group, Philox draws, and the MALA / GRW / HMC step loops of one chain
// held by `lpc` lanes of a wavefront (lpc a power of two <= 64, groups
// aligned inside the wave); each lane keeps NV float4 chunks of position /
// gradient in registers for the whole launch.
#pragma once

#include "fmc_common.h"
#include "fmc_targets.h"

namespace fmc {

struct ChainIO {
  float* x;
  float* logp;
  const float* metric;
  const float* noise;
  const float* log_u;
  float* out_pos;
  float* out_logp;
  float* out_acc;
  int64_t C;
  int64_t buf_len;
  int64_t cursor;
  uint32_t key0, key1;
  const float* temps;  // tempered rows: row c targets log p / temps[c % n_temps] (NULL: untempered)
  int n_temps;
  // HMC with a dense condition matrix M: chol = the lower-triangular
  // Cholesky factor of inv(M) ([d, d] row-major), and metric = the kinetic
  // weights colsum(M) (NULL: diagonal or unit metric)
  const float* chol = nullptr;
};

struct StepCfg {
  int n_steps;
  int step0;
  float dt;
  int n_leapfrog;
  int thinning;
};

template <int NV>
__device__ __forceinline__ void load_row(const float* __restrict__ src, int d, int r, int lpc,
                                         float4 (&x)[NV]) {
  const bool vec = (d & 3) == 0;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    int j0 = (v * lpc + r) * 4;
    if (vec) {
      x[v] = (j0 < d) ? *reinterpret_cast<const float4*>(src + j0) : make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) f4(x[v], e) = (j0 + e < d) ? src[j0 + e] : 0.f;
    }
  }
}

// A float4 at any 4-byte aligned address (global accesses need no more)
struct __attribute__((packed, aligned(4))) float4_a4 {
  float x, y, z, w;
};

template <int NV>
__device__ __forceinline__ void store_row(float* __restrict__ dst, int d, int r, int lpc,
                                          const float4 (&x)[NV]) {
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int j0 = (v * lpc + r) * 4;
    if (j0 + 3 < d) {
      *reinterpret_cast<float4_a4*>(dst + j0) = float4_a4{x[v].x, x[v].y, x[v].z, x[v].w};
    } else if (j0 < d) {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (j0 + e < d) dst[j0 + e] = f4c(x[v], e);
    }
  }
}

// Where a step's random numbers come from: memory (injected), the Philox
// stream, or LDS blocks that other wavefronts of the workgroup fill from the
// same stream (NoiseRing).
struct NoiseRing {
  int base;     // float offset of the ring in LDS: [2][T][NV][64] float4, then [2][T][64 / lpc] log u
  int n_steps;
};

// Steps a ring block holds
template <int NV>
constexpr int ring_T = NV == 1 ? 16 : NV == 2 ? 8 : 4;

template <int NV>
__device__ __forceinline__ int ring_lu(const NoiseRing& nr) { return nr.base + 2 * ring_T<NV> * NV * 256; }

// Standard normals of (chain, step) for this lane's chunks; padding zeroed.
template <int NV, bool RING>
__device__ __forceinline__ void draw_normals(const ChainIO& io, const NoiseRing& nr, int d, int r, int lpc, int64_t c,
                                             int s, int t_glob, uint32_t sid, float4 (&xi)[NV]) {
  if (RING) {
    const int slot = s & (2 * ring_T<NV> - 1);
#pragma unroll
    for (int v = 0; v < NV; ++v)
      xi[v] = *reinterpret_cast<const float4*>(fmc_chain_lds + nr.base + ((slot * NV + v) * 64 + (threadIdx.x & 63)) * 4);
  } else if (io.noise) {
    load_row<NV>(io.noise + ((int64_t)s * io.C + c) * d, d, r, lpc, xi);
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      int chunk = v * lpc + r;
      xi[v] = philox_normal4(io.key0, io.key1, (uint32_t)chunk, (uint32_t)c, (uint32_t)t_glob, sid);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (chunk * 4 + e >= d) f4(xi[v], e) = 0.f;
    }
  }
}

// log u of (chain, step). A group's lanes would all compute the same Philox
// block: each computes another step's instead, once every lpc steps (keep),
// and hands it over in its turn.
template <int NV, bool RING>
__device__ __forceinline__ float draw_log_u(const ChainIO& io, const NoiseRing& nr, int r, int lpc, int gbase, int64_t c,
                                            int s, int t_glob, uint32_t sid, float& keep) {
  if (RING) return fmc_chain_lds[ring_lu<NV>(nr) + (s & (2 * ring_T<NV> - 1)) * (64 / lpc) + (threadIdx.x & 63) / lpc];
  if (io.log_u) return io.log_u[(int64_t)s * io.C + c];
  const int k = s & (lpc - 1);
  if (k == 0) keep = philox_log_uniform(io.key0, io.key1, (uint32_t)c, (uint32_t)(t_glob + r), sid);
  return lpc == 1 ? keep : __shfl(keep, gbase + k, 64);
}

// Fills ring block `blk` (steps blk T .. ) for the chain wavefront of this
// workgroup: wavefront w of nw takes every nw-th (step, chunk) item, a log u
// item being 64 (step, chain) pairs. c0: the workgroup's first chain.
template <int NV>
__device__ __forceinline__ void fill_ring(const ChainIO& io, const NoiseRing& nr, const StepCfg& cfg, int d, int lpc,
                                          int64_t c0, int blk, int w, int nw, uint32_t sid, uint32_t sid_u) {
  constexpr int T = ring_T<NV>;
  const int lane = threadIdx.x & 63, r = lane & (lpc - 1), cpw = 64 / lpc;
  const int s0 = blk * T, half = (blk & 1) * T;
  const int ns = nr.n_steps - s0 < T ? nr.n_steps - s0 : T;  // steps of the block
  const int n_norm = ns * NV, n_u = (ns * cpw + 63) / 64;
  const uint32_t c = (uint32_t)(c0 + lane / lpc);
  for (int i = w; i < n_norm + n_u; i += nw) {
    if (i < n_norm) {
      const int st = i / NV, v = i - st * NV, chunk = v * lpc + r;
      float4 z = philox_normal4(io.key0, io.key1, (uint32_t)chunk, c, (uint32_t)(cfg.step0 + s0 + st), sid);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (chunk * 4 + e >= d) f4(z, e) = 0.f;
      *reinterpret_cast<float4*>(fmc_chain_lds + nr.base + (((half + st) * NV + v) * 64 + lane) * 4) = z;
    } else {
      const int k = (i - n_norm) * 64 + lane, st = k / cpw, cl = k - st * cpw;
      if (st < ns)
        fmc_chain_lds[ring_lu<NV>(nr) + (half + st) * cpw + cl] =
            philox_log_uniform(io.key0, io.key1, (uint32_t)(c0 + cl), (uint32_t)(cfg.step0 + s0 + st), sid_u);
    }
  }
}
// A ring block ends: its filler and its reader change places.
template <int NV, bool RING>
__device__ __forceinline__ void ring_step(const NoiseRing& nr, int s) {
  if (RING && ((s + 1) & (ring_T<NV> - 1)) == 0 && s + 1 < nr.n_steps) __syncthreads();
}

// The thinned buffer rows of one chain: global step t with t % thinning == 0
// lands on row cursor + t / thinning (pointers and the next such step carried
// along: no division or product a step).
struct RowWriter {
  float *pos = nullptr, *lp = nullptr, *acc = nullptr;
  int next, thinning;
  bool has_pos, has_lp, has_acc;  // the same for every lane: tested without the lanes' pointers
  __device__ __forceinline__ RowWriter(const ChainIO& io, const StepCfg& cfg, int d, int64_t c) {
    thinning = cfg.thinning;
    const int k = (cfg.step0 + thinning - 1) / thinning;
    next = k * thinning;
    const int64_t row = c * io.buf_len + io.cursor + k;
    has_pos = io.out_pos != nullptr;
    has_lp = io.out_logp != nullptr;
    has_acc = io.out_acc != nullptr;
    if (has_pos) pos = io.out_pos + row * d;
    if (has_lp) lp = io.out_logp + row;
    if (has_acc) acc = io.out_acc + row;
  }
  template <int NV>
  __device__ __forceinline__ void write(int t_glob, int d, int r, int lpc, const float4 (&x)[NV], float lpv, bool a) {
    if (t_glob != next) return;
    next += thinning;
    if (has_pos) {
      store_row<NV>(pos, d, r, lpc, x);
      pos += d;
    }
    if (has_lp) {
      if (r == 0) *lp = lpv;
      ++lp;
    }
    if (has_acc) {
      if (r == 0) *acc = a ? 1.f : 0.f;
      ++acc;
    }
  }
};

// Tempered rows (parallel tempering): row c of a tempered launch targets
// log p(x) / T with T = temps[c % n_temps] — TemperedPDF.tempered_log_pdf
// (src/flowMC/resource/logPDF.py:104-106) with a zero log prior. The value and
// the gradient of the target are scaled by beta = 1/T after each evaluation.
__device__ __forceinline__ float row_beta(const ChainIO& io, int64_t c) {
  return io.temps ? 1.f / io.temps[c % io.n_temps] : 1.f;
}

template <int NV>
__device__ __forceinline__ float temper(const ChainIO& io, float beta, float lp, float4 (&g)[NV]) {
  if (io.temps == nullptr) return lp;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e) f4(g[v], e) *= beta;
  return beta * lp;
}

// ------------------------------------------------------------------ MALA ---
// One chain group runs cfg.n_steps MALA steps (src/flowMC/resource/kernel/
// MALA.py:26-89). The gradient at the current point is carried from the
// previous step instead of being re-evaluated: MALA.py:59 recomputes it at the
// same point, which for a deterministic target is the same value.
template <int NV, int TK, int PAR, bool RING, class RG>
__device__ __forceinline__ void mala_group(const TargetDev& t, const ChainIO& io, const StepCfg& cfg,
                                           const NoiseRing& nr, int64_t c, int r, int lpc, int gbase) {
  const int d = t.d;
  const RG rg(t);
  float4 x[NV], g[NV];
  load_row<NV>(io.x + c * d, d, r, lpc, x);
  const float beta = row_beta(io, c);
  float lp = temper<NV>(io, beta, target_vg<NV, TK, PAR, true>(t, rg, x, g, r, lpc, gbase), g);
  const float dt = cfg.dt;
  const float h = 0.5f * dt * dt;
  const float inv2dt2 = 1.f / (2.f * dt * dt);
  RowWriter rows(io, cfg, d, c);
  float lu_keep = 0.f;
  for (int s = 0; s < cfg.n_steps; ++s) {
    const int tg = cfg.step0 + s;
    float4 xi[NV], prop[NV], g1[NV];
    draw_normals<NV, RING>(io, nr, d, r, lpc, c, s, tg, RNG_MALA_NOISE, xi);
    const float lu = draw_log_u<NV, RING>(io, nr, r, lpc, gbase, c, s, tg, RNG_MALA_UNIFORM, lu_keep);
    float s1 = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float n = dt * f4c(xi[v], e);
        f4(prop[v], e) = fmaf(dt, f4c(xi[v], e), fmaf(h, f4c(g[v], e), f4c(x[v], e)));
        s1 = fmaf(n, n, s1);
      }
    float lp1 = temper<NV>(io, beta, target_vg<NV, TK, PAR, false>(t, rg, prop, g1, r, lpc, gbase), g1);
    float s2 = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float q = fmaf(-h, f4c(g1[v], e), f4c(x[v], e) - f4c(prop[v], e));
        s2 = fmaf(q, q, s2);
      }
    // padding lanes contribute exactly 0 to s1 and s2
    float ds = group_sum(s1 - s2, lpc);
    const float ratio = fmaf(ds, inv2dt2, lp1 - lp);
    bool acc = lu < ratio;
    if (acc) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        x[v] = prop[v];
        g[v] = g1[v];
      }
      lp = lp1;
    }
    rows.write<NV>(tg, d, r, lpc, x, lp, acc);
    ring_step<NV, RING>(nr, s);
  }
  store_row<NV>(io.x + c * d, d, r, lpc, x);
  if (r == 0 && io.logp) io.logp[c] = lp;
}

// ------------------------------------------------------------------- GRW ---
// GaussianRandomWalk.kernel (src/flowMC/resource/kernel/Gaussian_random_walk.py:
// 25-61) scanned by TakeSerialSteps: x' = x + step * xi, accept iff
// log u < logp(x') - logp(x). The log-density of the entry state is evaluated
// once (take_steps.py:177) and carried; the target's gradient output is dead
// and removed by the compiler.
template <int NV, int TK, int PAR, bool RING, class RG>
__device__ __forceinline__ void grw_group(const TargetDev& t, const ChainIO& io, const StepCfg& cfg,
                                          const NoiseRing& nr, int64_t c, int r, int lpc, int gbase) {
  const int d = t.d;
  const RG rg(t);
  float4 x[NV], g[NV];
  load_row<NV>(io.x + c * d, d, r, lpc, x);
  const float beta = row_beta(io, c);
  float lp = temper<NV>(io, beta, target_vg<NV, TK, PAR, true>(t, rg, x, g, r, lpc, gbase), g);
  const float dt = cfg.dt;
  RowWriter rows(io, cfg, d, c);
  float lu_keep = 0.f;
  for (int s = 0; s < cfg.n_steps; ++s) {
    const int tg = cfg.step0 + s;
    float4 xi[NV], prop[NV];
    draw_normals<NV, RING>(io, nr, d, r, lpc, c, s, tg, RNG_GRW_NOISE, xi);
    const float lu = draw_log_u<NV, RING>(io, nr, r, lpc, gbase, c, s, tg, RNG_GRW_UNIFORM, lu_keep);
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) f4(prop[v], e) = fmaf(dt, f4c(xi[v], e), f4c(x[v], e));
    const float lp1 = temper<NV>(io, beta, target_vg<NV, TK, PAR, false>(t, rg, prop, g, r, lpc, gbase), g);
    const bool acc = lu < lp1 - lp;
    if (acc) {
#pragma unroll
      for (int v = 0; v < NV; ++v) x[v] = prop[v];
      lp = lp1;
    }
    rows.write<NV>(tg, d, r, lpc, x, lp, acc);
    ring_step<NV, RING>(nr, s);
  }
  store_row<NV>(io.x + c * d, d, r, lpc, x);
  if (r == 0 && io.logp) io.logp[c] = lp;
}

// ------------------------------------------------------------------- HMC ---
// HMC.kernel (src/flowMC/resource/kernel/HMC.py:98-151) with the leapfrog
// coefficient table of HMC.py:47-50: row 0 = (0, 1/2), rows 1..L = (1, 1),
// row L+1 = (1, 1/2): L+1 drifts x += eps*c0*w*p and L+2 kicks
// p += eps*c1*grad logp(x). H0 - H1 is accumulated in FP64.
//
// Metric kinds MK (the condition matrix M):
//   MK_UNIT  identity (io.metric == nullptr): padding elements of p, x and
//            the gradient are 0 throughout, so this form needs no
//            per-element index test and no metric multiply;
//   MK_DIAG  diagonal: p = xi / sqrt(m), kinetic 1/2 sum m p^2, drift m p;
//   MK_DENSE dense: p = xi @ chol(inv(M))^T (HMC.py:133-136), and the
//            reference's broadcast kinetic 1/2 sum(p^2 * M) =
//            1/2 sum_j w_j p_j^2 with w = colsum(M) (HMC.py:118-121), whose
//            p-gradient w p is the drift; io.chol holds the factor, io.metric w.
enum { MK_UNIT = 0, MK_DIAG = 1, MK_DENSE = 2 };

// p = L xi for the chain held by this lane group (L lower-triangular [d, d]
// row-major): every lane needs all of its chain's xi, gathered chunk by
// chunk from the group's lanes with shuffles; padding elements of p are 0.
template <int NV>
__device__ __forceinline__ void dense_momentum(const float* __restrict__ Lc, int d, int r, int lpc, int gbase,
                                               const float4 (&xi)[NV], float4 (&p)[NV]) {
#pragma unroll
  for (int v = 0; v < NV; ++v) p[v] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int src = 0; src < lpc; ++src) {
#pragma unroll
    for (int vs = 0; vs < NV; ++vs) {
      const int k0 = (vs * lpc + src) * 4;  // the same for every lane of the wave
      float xs[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) xs[e] = __shfl(f4c(xi[vs], e), gbase + src, 64);
      if (k0 >= d) continue;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = dim_of(v, e, r, lpc);
          if (j < d && k0 <= j) {
            const float* row = Lc + (int64_t)j * d + k0;
            float acc = f4c(p[v], e);
#pragma unroll
            for (int ee = 0; ee < 4; ++ee)
              if (k0 + ee <= j) acc += row[ee] * xs[ee];
            f4(p[v], e) = acc;
          }
        }
    }
  }
}

template <int NV, int MK, int TK, int PAR, class RG>
__device__ __forceinline__ void hmc_group(const TargetDev& t, const ChainIO& io, const StepCfg& cfg, int64_t c,
                          int r, int lpc, int gbase) {
  constexpr bool UNIT_M = MK == MK_UNIT;
  const int d = t.d;
  const RG rg(t);
  float4 x[NV], g[NV], m[NV];
  load_row<NV>(io.x + c * d, d, r, lpc, x);
  if (!UNIT_M) {
    load_row<NV>(io.metric, d, r, lpc, m);
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v) m[v] = make_float4(1.f, 1.f, 1.f, 1.f);
  }
  const float beta = row_beta(io, c);
  float lp = temper<NV>(io, beta, target_vg<NV, TK, PAR, false>(t, rg, x, g, r, lpc, gbase), g);
  const float eps = cfg.dt;
  const int L = cfg.n_leapfrog;
  RowWriter rows(io, cfg, d, c);
  float lu_keep = 0.f;
  for (int s = 0; s < cfg.n_steps; ++s) {
    const int tg = cfg.step0 + s;
    float4 p[NV], xl[NV], gl[NV];
    draw_normals<NV, false>(io, NoiseRing{0, 0}, d, r, lpc, c, s, tg, RNG_HMC_MOMENTUM, p);
    const float lu = draw_log_u<NV, false>(io, NoiseRing{0, 0}, r, lpc, gbase, c, s, tg, RNG_HMC_UNIFORM, lu_keep);
    if (MK == MK_DENSE) {
      float4 xi[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) xi[v] = p[v];
      dense_momentum<NV>(io.chol, d, r, lpc, gbase, xi, p);
    }
    double k0 = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (UNIT_M) {
          // sum of squares; the 1/2 is applied after the group sum (a power
          // of two: the same bits as summing 0.5 p^2)
          const double pj = (double)f4c(p[v], e);
          k0 = fma(pj, pj, k0);
        } else {
          int j = dim_of(v, e, r, lpc);
          float mj = f4c(m[v], e);
          float pj = (j < d) ? (MK == MK_DENSE ? f4c(p[v], e) : f4c(p[v], e) / sqrtf(mj)) : 0.f;
          f4(p[v], e) = pj;
          k0 += 0.5 * (double)mj * (double)pj * (double)pj;
        }
      }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      xl[v] = x[v];
      gl[v] = g[v];
    }
    k0 = group_sum(k0, lpc);
    if (UNIT_M) k0 *= 0.5;
    // row 0: drift coefficient 0, kick 1/2
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) f4(p[v], e) = fmaf(eps * 0.5f, f4c(gl[v], e), f4c(p[v], e));
    float lpl = lp;
    for (int i = 1; i <= L + 1; ++i) {
      const float kick = (i <= L) ? 1.f : 0.5f;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) f4(xl[v], e) = fmaf(eps, UNIT_M ? f4c(p[v], e) : f4c(m[v], e) * f4c(p[v], e), f4c(xl[v], e));
      lpl = temper<NV>(io, beta, target_vg<NV, TK, PAR, false>(t, rg, xl, gl, r, lpc, gbase), gl);
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) f4(p[v], e) = fmaf(eps * kick, f4c(gl[v], e), f4c(p[v], e));
    }
    double k1 = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (UNIT_M) {
          const double pj = (double)f4c(p[v], e);
          k1 = fma(pj, pj, k1);
        } else {
          int j = dim_of(v, e, r, lpc);
          if (j < d) k1 += 0.5 * (double)f4c(m[v], e) * (double)f4c(p[v], e) * (double)f4c(p[v], e);
        }
      }
    k1 = group_sum(k1, lpc);
    if (UNIT_M) k1 *= 0.5;
    double h0 = -(double)lp + k0;
    double h1 = -(double)lpl + k1;
    double log_acc = h0 - h1;
    bool acc = (double)lu < log_acc;
    if (acc) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        x[v] = xl[v];
        g[v] = gl[v];
      }
      lp = lpl;
    }
    rows.write<NV>(tg, d, r, lpc, x, lp, acc);
  }
  store_row<NV>(io.x + c * d, d, r, lpc, x);
  if (r == 0 && io.logp) io.logp[c] = lp;
}

}  // namespace fmc
