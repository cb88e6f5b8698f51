// MaskedCouplingRQSpline flow passes over many samples: 64-sample tiles, one
// activation region, weights streamed without a break (rqSpline.py:450-504).
// fmc_flow_pass.hip holds the general pass and the rule that chooses.
#include "fmc_flow_common.h"
#include "fmc_flow_wide.h"

namespace fmc {

constexpr int WD_MB = WIDE_MT / 32;  // 32-sample blocks of the tile
struct WdRing {
  bf16x8_t r[WD_P][2];
};
// A panel's (up to) two 32-row blocks: byte offsets of their fragment images
// in the packed buffer, and their k-steps
struct WdPanel {
  uint32_t b[2];
  int KB;
};
// Fragments come by buffer loads: the block and k-step as a scalar offset, the
// lane's place as the vector offset (no address arithmetic on the lanes). The
// ring reads up to WD_P - 1 k-steps past a panel and uses none of them: what
// follows a panel in the packed buffer is another image, after the last w3r
// panel the transposed one (flow_wide checks it; a bounds check of the load
// would not count the scalar offset).
struct WdSrc {
  __amdgpu_buffer_rsrc_t rs;
  int voff;
  __device__ __forceinline__ bf16x8_t load(uint32_t off) const {
    return __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, (int)off, 0));
  }
};
constexpr uint32_t WD_STEP = 64 * 16;  // bytes of one k-step's fragments

template <int CB>
__device__ __forceinline__ void wd_fill(WdRing& ring, const WdPanel& p, const WdSrc& src) {
#pragma unroll
  for (int i = 0; i < WD_P; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) ring.r[i][j] = src.load(p.b[j] + i * WD_STEP);
}

// acc += the panel's 32 CB weight rows x the tile's 64 samples, in ascending
// k-steps. The ring holds the panel's first k-steps on entry; a step loads
// what the ring needs WD_P steps on, at the end of the panel the first k-steps
// of `next`, so that the stream does not stop between panels, barriers and
// splines. The steps are kept apart (sched_barrier): left to itself the
// compiler moves a group's loads behind its last MFMA, where the next group
// waits for them at once. The LDS rows of a step are read one step ahead.
template <int CB, int CBN, class LA>
__device__ __forceinline__ void wd_run(WdRing& ring, const WdPanel& p, const WdPanel& next, const WdSrc& src,
                                       LA&& load_a, f32x16_t (&acc)[CB][WD_MB]) {
  __builtin_amdgcn_s_setprio(1);
  bf16x8_t x[2][WD_MB];
#pragma unroll
  for (int r = 0; r < WD_MB; ++r) x[0][r] = load_a(r, 0);
  auto step = [&](int i, int k, uint32_t n0, uint32_t n1, bool more) {
    if (more) {
#pragma unroll
      for (int r = 0; r < WD_MB; ++r) x[(i + 1) & 1][r] = load_a(r, k + 1);
    }
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int r = 0; r < WD_MB; ++r) acc[j][r] = PBF16::mma(ring.r[i][j], x[i & 1][r], acc[j][r]);
    ring.r[i][0] = src.load(n0 + i * WD_STEP);
    if (CB == 2 || CBN == 2) ring.r[i][1] = src.load(n1 + i * WD_STEP);
    __builtin_amdgcn_sched_barrier(0);
  };
  int kb = 0;
  auto group = [&] {
    const bool last = kb + WD_P >= p.KB;
    const uint32_t n0 = last ? next.b[0] : p.b[0] + (kb + WD_P) * WD_STEP;
    const uint32_t n1 = last ? next.b[1] : p.b[1] + (kb + WD_P) * WD_STEP;
#pragma unroll
    for (int i = 0; i < WD_P; ++i) step(i, kb + i, n0, n1, i + 1 < WD_P || !last);
    kb += WD_P;
  };
  if (WD_P <= p.KB) {  // the first group apart: it takes the biases as the MFMAs' third operand
    group();
    while (kb + WD_P <= p.KB) group();
  }
  if (kb < p.KB) {
#pragma unroll
    for (int i = 0; i < WD_P; ++i) {
      if (kb + i < p.KB) {
        step(i, kb + i, next.b[0], next.b[1], kb + i + 1 < p.KB);
      } else {
        ring.r[i][0] = src.load(next.b[0] + i * WD_STEP);
        if (CB == 2 || CBN == 2) ring.r[i][1] = src.load(next.b[1] + i * WD_STEP);
      }
    }
  }
  __builtin_amdgcn_s_setprio(0);
}

// One affine layer of a direction: forward (v + shift) e^scale, else v e^-scale - shift
struct WdAff {
  float e, sh;
  __device__ __forceinline__ float operator()(bool fwd, float v) const { return fwd ? (v + sh) * e : fmaf(v, e, -sh); }
};

// Bound by the weights' way from L2 to the CUs and, next, by VALU issue (spline
// and tanh, 56 % of the time, beside 35 % for the MFMAs): every workgroup reads
// all weights of a layer (668 KB at d = 64, [256, 256]), so a tile of twice the
// samples halves that stream, and two workgroups a CU (256 registers a lane)
// run it. 10 layers, d = 64, [256, 256], 8 bins, 409600 samples with their
// log-density: 4.60 -> 3.48 ms (84 -> 43 GB of weights); log_prob of 300000 at
// d = 32, [128, 128], 10 bins 1.25 -> 1.05 ms. Measured and left: a ring of
// eight k-steps (3.63 ms; the loads' rate, not their latency, is what binds),
// three workgroups a CU (168 registers spill: 5.0 ms), tiles of 96 (7.0 ms) or
// 128 samples (4.5 ms; one workgroup a CU). What else left the general pass:
// the affine passes over the tile (a dim's affine goes where its spline reads
// or writes it), the conditioner-input copy (hidden layer 0 reads the tile),
// one of the two activation regions (written after a barrier), three of four
// draws of each Philox block, a thread's serial sum over the base terms.
// Every sum keeps the general pass's order, so the results are the same bits.
template <int KT, int NH, int CBH>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
flow_wide_kernel(FlowDev f, PassArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const FlowDims& dm = f.dm;
  const WideSmem sm(dm);
  float* xs = reinterpret_cast<float*>(smem + sm.xs);
  float* ldw = reinterpret_cast<float*>(smem + sm.ldw);
  __bf16* hb = reinterpret_cast<__bf16*>(smem + sm.h);
  float* bb = reinterpret_cast<float*>(smem + sm.b);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = dm.d, ldx = sm.ldx, lh = sm.lh, hf = lane >> 5;
  const int64_t m0 = (int64_t)blockIdx.x * WIDE_MT;
  const float* th = f.theta;
  const bool fwd = a.dir == 0;

  // the affine between the splines of steps s - 1 and s (identity at the open end)
  auto layer_of = [&](int s) { return fwd ? s : dm.L - 1 - s; };
  auto affine = [&](int s) {
    const int at = a.dir == 2 ? s - 1 : s;
    if (at < 0 || at >= dm.L) return WdAff{1.f, 0.f};
    const int l = layer_of(at);
    const float sc = th[dm.th_scale(l)];
    return WdAff{expf(fwd ? sc : -sc), th[dm.th_shift(l)]};
  };

  // hidden layer i of layer l: this wavefront's blocks (a wavefront without any: valid ones)
  auto hidden_panel = [&](int l, int i) {
    const int NBt = dm.hp(i) / 32, c0 = wave < NBt ? wave : 0, c1 = c0 + 4 < NBt ? c0 + 4 : c0;
    const int KB = dm.wh_k(l, i) / 16;
    const uint32_t o = (uint32_t)(dm.pk_layer(l) + dm.pk_wh(l, i)) * 2;
    return WdPanel{{o + c0 * KB * WD_STEP, o + c1 * KB * WD_STEP}, KB};
  };
  // output rows of dim pair q of layer l
  auto pair_panel = [&](int l, int q) {
    const int KB = dm.hlp() / 16;
    const uint32_t o = (uint32_t)(dm.pk_layer(l) + dm.pk_w3r(l)) * 2 + 2 * q * KB * WD_STEP;
    return WdPanel{{o, o + KB * WD_STEP}, KB};
  };
  const WdSrc src{__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(f.packed), 0, (int)(dm.pk_total() * 2), 0x00027000),
                  lane * 16};
  WdRing ring;
  wd_fill<2>(ring, hidden_panel(layer_of(0), 0), src);

  // ---- the tile: standardised input or base draws; the first step's
  // conditioning dims go through the first affine here, the others when their
  // spline reads them
  const WdAff A0 = affine(0);
  const int cpar = (layer_of(0) + 1) & 1;
  auto put = [&](int m, int j, float v) { xs[m * ldx + j] = (j & 1) == cpar ? A0(fwd, v) : v; };
  if ((a.flags & FL_SAMPLE) && a.x_in == nullptr) {  // one Philox block for four dims
    for (TileWalk tw(tid, (d + 3) / 4); tw.m < WIDE_MT; tw.next()) {
      const int64_t row = m0 + tw.m;
      const float4 z = philox_normal4(a.key0, a.key1, (uint32_t)tw.j, (uint32_t)(a.sample0 + row), 0u, RNG_FLOW_BASE);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 4 * tw.j + e;
        if (j >= d) break;
        float v = 0.f;
        if (row < a.n) v = th[dm.th_base_mean() + j] + sqrtf(th[dm.th_base_cov() + (int64_t)j * d + j]) * f4c(z, e);
        put(tw.m, j, v);
      }
    }
  } else {
    for (TileWalk tw(tid, d); tw.m < WIDE_MT; tw.next()) {
      const int64_t row = m0 + tw.m;
      const int j = tw.j;
      float v = 0.f;
      if (row < a.n) {
        v = a.x_in[row * d + j];
        if (fwd && (a.flags & FL_STD))
          v = (v - th[dm.th_data_mean() + j]) / sqrtf(th[dm.th_data_cov() + (int64_t)j * d + j]);
        else if (!fwd && (a.flags & FL_SAMPLE))
          v = th[dm.th_base_mean() + j] + sqrtf(th[dm.th_base_cov() + (int64_t)j * d + j]) * v;
      }
      put(tw.m, j, v);
    }
  }
  __syncthreads();

  // log N(row; base_mean, diag(base_cov)) without its sign: sum_j (x_j - mean_j)^2
  // / var_j and sum_j log var_j in ascending j for thread `tid`'s row. The terms
  // are computed by all threads, a block of dims at a time, in the activation
  // region; A: an affine the dims of parity `par` still have to go through.
  auto base_sums = [&](const WdAff& A, int par, float& q, float& lg) {
    float* t = reinterpret_cast<float*>(hb);
    const int jc = sm.base_cols(d), ldt = jc | 1;
    q = lg = 0.f;
    for (int j0 = 0; j0 < d; j0 += jc) {
      const int nj = d - j0 < jc ? d - j0 : jc;
      for (TileWalk tw(tid, nj); tw.m <= WIDE_MT; tw.next()) {
        const int j = j0 + tw.j;
        const float var = th[dm.th_base_cov() + (int64_t)j * d + j];
        if (tw.m < WIDE_MT) {
          float v = xs[tw.m * ldx + j];
          if ((j & 1) == par) v = A(fwd, v);
          const float u = v - th[dm.th_base_mean() + j];
          t[tw.m * ldt + tw.j] = u * u / var;
        } else {
          t[tw.m * ldt + tw.j] = logf(var);
        }
      }
      __syncthreads();
      if (tid < WIDE_MT)
        for (int jj = 0; jj < nj; ++jj) {
          q += t[tid * ldt + jj];
          lg += t[WIDE_MT * ldt + jj];
        }
      __syncthreads();
    }
  };
  // exact inverse with FL_BASE: the flow log-density of the output, log N(z) -
  // sum of the inverse log-dets; starts from -log N(z). Thread m < 64 carries row m's.
  float half_log_2pi_d;  // (a product of its own, not the half of an FMA, as in the general pass)
  {
#pragma clang fp contract(off)
    half_log_2pi_d = 0.91893853320467274f * (float)d;
  }
  const bool inv_logq = a.dir == 2 && (a.flags & FL_BASE);
  float ldr = 0.f;
  if (inv_logq) {
    float q, lg;
    base_sums(WdAff{1.f, 0.f}, 2, q, lg);
    ldr = 0.5f * q + 0.5f * lg + half_log_2pi_d;
  }

  WdAff As = A0;
  for (int step = 0; step < dm.L; ++step) {
    const int l = layer_of(step);
    const WdAff An = affine(step + 1);
    const float sc = th[dm.th_scale(l)];
    const float* bl = f.pbias + dm.pb_layer(l);
    const int npair = dm.n_pairs(l), dtl = dm.dt(l), dc = dm.dc(l);
    const WdPanel after = hidden_panel(step + 1 < dm.L ? layer_of(step + 1) : l, 0);
    // the layer's biases (read from memory, a panel waited for them: 4 + 2 round
    // trips a layer); hidden layer 0 starts before the barrier that shows them
    for (int i = tid; i < (int)dm.pb_size(l); i += 256) bb[i] = bl[i];
    if (a.dir != 2) ldr = fmaf(fwd ? sc : -sc, (float)d, ldr);

    // ---- hidden layers
#pragma unroll
    for (int i = 0; i < NH; ++i) {
      const int NBt = dm.hp(i) / 32;
      const WdPanel nxt = i + 1 < NH ? hidden_panel(l, i + 1) : wave < npair ? pair_panel(l, wave) : after;
      f32x16_t acc[CBH][WD_MB];
      if (wave < NBt) {
#pragma unroll
        for (int j = 0; j < CBH; ++j) bias_tr<WD_MB>(acc[j], (i == 0 ? bl : bb) + dm.pb_b(i), wave + 4 * j < NBt ? wave + 4 * j : wave, lane);
        if (i == 0) {
          // the conditioning dims, straight from the tile
          const float* xr = xs + (lane & 31) * ldx + ((l + 1) & 1);
          wd_run<CBH, 2>(ring, hidden_panel(l, 0), nxt, src,
                      [&](int r, int kb) {
                        bf16x8_t v;
                        const float* x = xr + r * 32 * ldx;
                        const int k0 = 16 * kb + 8 * hf;
                        if (16 * kb + 16 <= dc) {
#pragma unroll
                          for (int e = 0; e < 8; ++e) v[e] = (__bf16)x[2 * (k0 + e)];
                        } else {  // past the last conditioning dim: that dim's value, replaced by 0
#pragma unroll
                          for (int e = 0; e < 8; ++e) {
                            const int k = k0 + e, kk = k < dc ? k : (dc > 0 ? dc - 1 : 0);
                            const float u = x[2 * kk];
                            v[e] = (__bf16)(k < dc ? u : 0.f);
                          }
                        }
                        return v;
                      },
                      acc);
        } else {
          wd_run<CBH, 2>(ring, hidden_panel(l, i), nxt, src, [&](int r, int kb) { return PBF16::load_a(hb, lh, 32 * r, kb, lane); },
                      acc);
        }
      } else {
        wd_fill<2>(ring, nxt, src);
      }
      if (i > 0) __syncthreads();  // the region's readers are done
      if (wave < NBt) {
#pragma unroll
        for (int j = 0; j < CBH; ++j)
          if (wave + 4 * j < NBt) hidden_epilogue_tr<PBF16, WD_MB>(hb, lh, nullptr, wave + 4 * j, acc[j], lane);
      }
      __syncthreads();
    }
    // ---- spline parameters of two dims at a time and their spline
    float ldacc[WD_MB] = {};
    const float* b3r = bb + dm.pb_b3r(l);
    for (int q = wave; q < npair; q += 4) {
      const int k = 2 * q + hf;
      f32x16_t acc[2][WD_MB];
      const float4* bp = reinterpret_cast<const float4*>(b3r + q * 64 + (k < dtl ? hf * 32 : 0));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float4 b4 = bp[u];
#pragma unroll
        for (int r = 0; r < WD_MB; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[u >> 2][r][4 * (u & 3) + e] = f4c(b4, e);
      }
      wd_run<2, 2>(ring, pair_panel(l, q), q + 4 < npair ? pair_panel(l, q + 4) : after, src,
                [&](int r, int kb) { return PBF16::load_a(hb, lh, 32 * r, kb, lane); }, acc);
      if (k < dtl) {
        const int j = dm.trans(l, k);
#pragma unroll
        for (int r = 0; r < WD_MB; ++r) {
          float pp[32];
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            pp[v] = acc[0][r][v];
            pp[16 + v] = acc[1][r][v];
          }
          float* x = xs + (r * 32 + (lane & 31)) * ldx + j;
          const float xv = As(fwd, *x);
          float yv, ldv;
          if (fwd)
            rs_fwd<KT, true>(pp, dm.K, f, xv, yv, ldv);
          else
            rs_inv<KT, true>(pp, dm.K, f, xv, yv, ldv);
          *x = An(fwd, yv);
          ldacc[r] += ldv;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < WD_MB; ++r) {
      const float o = __shfl_xor(ldacc[r], 32, 64);
      if (lane < 32) ldw[wave * WIDE_MT + r * 32 + lane] = ldacc[r] + o;
    }
    __syncthreads();
    if (tid < WIDE_MT)
      ldr += (ldw[tid] + ldw[WIDE_MT + tid]) + (ldw[2 * WIDE_MT + tid] + ldw[3 * WIDE_MT + tid]);
    if (a.dir == 2) ldr = fmaf(-sc, (float)d, ldr);
    As = An;
  }
  // the last step's conditioning dims still have the closing affine to go through
  const int opar = (layer_of(dm.L - 1) + 1) & 1;
  if (fwd && (a.flags & FL_BASE)) {
    float q, lg;
    base_sums(As, opar, q, lg);
    ldr += -0.5f * q - 0.5f * lg - half_log_2pi_d;
  }
  if (inv_logq) ldr = -ldr;
  if (a.logdet && tid < WIDE_MT && m0 + tid < a.n) a.logdet[m0 + tid] = ldr;
  if (a.x_out) {
    for (TileWalk tw(tid, d); tw.m < WIDE_MT; tw.next()) {
      const int64_t row = m0 + tw.m;
      const int j = tw.j;
      if (row >= a.n) continue;
      float v = xs[tw.m * ldx + j];
      if ((j & 1) == opar) v = As(fwd, v);
      if (!fwd && (a.flags & FL_STD))
        v = v * sqrtf(th[dm.th_data_cov() + (int64_t)j * d + j]) + th[dm.th_data_mean() + j];
      a.x_out[row * d + j] = v;
    }
  }
}

template <int KT, int NH>
static void launch_wide_nh(dim3 g, size_t shm, hipStream_t st, const FlowDev& fd, const PassArgs& a) {
  if (fd.dm.hmaxp() <= 128) {
    set_lds(flow_wide_kernel<KT, NH, 1>, shm);
    hipLaunchKernelGGL((flow_wide_kernel<KT, NH, 1>), g, dim3(256), shm, st, fd, a);
  } else {
    set_lds(flow_wide_kernel<KT, NH, 2>, shm);
    hipLaunchKernelGGL((flow_wide_kernel<KT, NH, 2>), g, dim3(256), shm, st, fd, a);
  }
}

template <int KT>
static void launch_wide_kt(dim3 g, size_t shm, hipStream_t st, const FlowDev& fd, const PassArgs& a) {
  switch (fd.dm.nh) {
    case 1: launch_wide_nh<KT, 1>(g, shm, st, fd, a); break;
    case 2: launch_wide_nh<KT, 2>(g, shm, st, fd, a); break;
    case 3: launch_wide_nh<KT, 3>(g, shm, st, fd, a); break;
    default: launch_wide_nh<KT, 4>(g, shm, st, fd, a); break;
  }
}

void launch_flow_wide(hipStream_t st, const FlowDev& fd, const PassArgs& a) {
  const size_t shm = (size_t)WideSmem(fd.dm).total;
  const dim3 g((unsigned)((a.n + WIDE_MT - 1) / WIDE_MT));
  const int kt = spline_kt(fd.dm.K);
  if (kt == 8)
    launch_wide_kt<8>(g, shm, st, fd, a);
  else if (kt == 10)
    launch_wide_kt<10>(g, shm, st, fd, a);
  else
    launch_wide_kt<0>(g, shm, st, fd, a);
}

}  // namespace fmc
