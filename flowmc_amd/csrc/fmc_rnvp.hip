// RealNVP flow kernels for gfx950 (src/flowMC/resource/model/nf_model/
// realNVP.py). Per layer a masked coupling layer whose scale and shift MLPs
// ([d, hidden, d], ReLU; common.py:68-112, 171-208) read the conditioning
// dims and drive the transformed dims:
//   s = tanh(MLP_s(c)) dt,  t = MLP_t(c) dt,  y = (x + t) e^s,  log-det = sum s.
// The model is FP32 end to end. The passes run on the FP32 matrix cores
// (v_mfma_f32_16x16x4: the FP32 vector rate without packed forms is half of
// it): 409,600 samples at d = 32, 8 layers, hidden 256 drawn in 1.10 ms, 98
// TFLOP/s, where FMA register tiles over LDS took 4.05 ms; 10,000 in 67 us
// (213 us). Training (forward with saved inputs, adjoint) uses FP32 FMA
// register tiles (4 outputs x 4 samples per thread) over LDS-resident
// activations, with weights read as aligned float4 rows of an L2-resident
// packed copy; products with few outputs split their reduction over the lanes
// of a wavefront and combine them with xor shuffles. Its workgroups of 256
// threads own RN_TS = 16 samples; the adjoint runs one layer per launch and
// writes per-tile weight-gradient partials, which a second kernel sums over
// tiles in a fixed order and scatters into the gradient vector.
#include "fmc_common.h"

namespace fmc {

constexpr int RN_TS = 16;       // samples per workgroup
constexpr int RN_THREADS = 256;
constexpr int RN_Q = RN_TS / 4;  // float4 sample groups

struct RnvpDev {
  int d, L, h;
  float dt;
  const float* theta;
  const float* packed;
  const int32_t* layout;
};

// ---- flat parameter layout (theta): per layer, for p = scale, shift:
//   W1 [h][d], b1 [h], W2 [d][h], b2 [d]; then data_mean [d], data_cov [d][d],
//   base_mean [d], base_cov [d][d].
__host__ __device__ inline int64_t rn_mlp_size(int d, int h) { return 2LL * h * d + h + d; }
__host__ __device__ inline int64_t rn_layer_size(int d, int h) { return 2 * rn_mlp_size(d, h); }
__host__ __device__ inline int64_t rn_mlp(int d, int h, int l, int p) {
  return l * rn_layer_size(d, h) + p * rn_mlp_size(d, h);
}
__host__ __device__ inline int64_t rn_stats(int d, int h, int L) { return L * rn_layer_size(d, h); }
__host__ __device__ inline int64_t rn_theta_size(int d, int h, int L) {
  return rn_stats(d, h, L) + 2LL * d + 2LL * d * d;
}
// ---- packed copy, per (layer, p), with d4 / h4 = d / h rounded up to 4 and
// zero padding: W1T [d4][h4] (W1T[k][j] = W1[j][cond_k]), W1c [h4][d4] (its
// transpose), W2T [h4][d4] (W2T[j][i] = W2[trans_i][j]), W2c [d4][h4] (its
// transpose), b1 [h4], b2c [d4] (b2c[i] = b2[trans_i]). Every row starts on a
// 16-byte boundary.
__host__ __device__ inline int rn_r4(int v) { return (v + 3) & ~3; }
__host__ __device__ inline int64_t rn_pk_mlp(int d, int h) {
  return 4LL * rn_r4(d) * rn_r4(h) + rn_r4(h) + rn_r4(d);
}
__host__ __device__ inline int64_t rn_pk(int d, int h, int l, int p) { return (2LL * l + p) * rn_pk_mlp(d, h); }
struct RnPk {
  const float *W1T, *W1c, *W2T, *W2c, *b1, *b2c;
  __device__ RnPk(const float* base, int d4, int h4) {
    const int64_t s = (int64_t)d4 * h4;
    W1T = base;
    W1c = base + s;
    W2T = base + 2 * s;
    W2c = base + 3 * s;
    b1 = base + 4 * s;
    b2c = b1 + h4;
  }
};
// ---- MFMA fragment images, per (layer, p), after the images above. Blocks of
// 16 conditioning dims (kg < KC), 16 transformed dims (r < R) and 16 hidden
// features (hb < HB); one 16 x 16 weight block is 64 lanes x float4, lane l
// (c = l % 16, q = l / 16) holding four k-steps of v_mfma_f32_16x16x4:
//   W1f [hb][kg]: W1[16 hb + c][cond(16 kg + 4q + e)]
//   W2f [hb][r]:  W2[trans(16 r + c)][16 hb + 4q + e]
// (k = 4q + e is also the row a lane's accumulator e holds, so the output
// block of the first product is the second product's operand as it lies),
// then b1 [16 HB], b2 [16 R], and the index words {n_cond, n_trans, 0, 0,
// cond [16 KC], trans [16 R]} (padding entries 0). A slot has a fixed size:
// KC + R <= ceil(d / 16) + 1 whatever the mask.
__host__ __device__ inline int rn_b16(int v) { return (v + 15) >> 4; }
__host__ __device__ inline int64_t rn_fr_slot(int d, int h) {
  const int kr = rn_b16(d) + 1, hb = rn_b16(h);
  return 256LL * hb * kr + 16LL * hb + 16LL * rn_b16(d) + 4 + 16LL * kr;
}
__host__ __device__ inline int64_t rn_fr_base(int d, int h, int L) { return (2LL * L * rn_pk_mlp(d, h) + 15) & ~15LL; }
__host__ __device__ inline int64_t rn_packed_size(int d, int h, int L) {
  return rn_fr_base(d, h, L) + 2LL * L * ((rn_fr_slot(d, h) + 15) & ~15LL);
}
struct RnFr {
  int KC, R, HB;
  const float *W1f, *W2f, *b1, *b2;
  const int32_t *nct, *cond, *trans;  // {n_cond, n_trans}, index lists
  __device__ RnFr(const float* packed, int d, int h, int L, int l, int p, int dc, int dtr) {
    KC = rn_b16(dc);
    R = rn_b16(dtr);
    HB = rn_b16(h);
    W1f = packed + rn_fr_base(d, h, L) + (2LL * l + p) * ((rn_fr_slot(d, h) + 15) & ~15LL);
    W2f = W1f + 256LL * HB * KC;
    b1 = W2f + 256LL * HB * R;
    b2 = b1 + 16 * HB;
    nct = reinterpret_cast<const int32_t*>(b2 + 16 * R);
    cond = nct + 4;
    trans = cond + 16 * KC;
  }
};
// ---- layout: per layer [n_cond, n_trans, cond[d], trans[d]]
__host__ __device__ inline const int32_t* rn_lay(const RnvpDev& f, int l) { return f.layout + (int64_t)l * (2 + 2 * f.d); }

__host__ __device__ inline int rn_rup16(int v) { return (v + 15) & ~15; }

struct RnSmem {
  int xs, gb, cT, hT, ghT, sT, tT, gcT, ldr, glp, total;
  int ldx, d4, h4;
  __host__ __device__ RnSmem(int d, int h, bool bwd) {
    ldx = d + 1;
    d4 = (d + 3) & ~3;
    h4 = (h + 3) & ~3;
    int o = 0;
    xs = o;
    o += rn_rup16(RN_TS * ldx * 4);
    gb = o;
    o += bwd ? rn_rup16(RN_TS * ldx * 4) : 0;
    cT = o;  // [d4][TS] conditioning inputs, sample-contiguous
    o += d4 * RN_TS * 4;
    hT = o;  // [h4][TS] hidden activations
    o += h4 * RN_TS * 4;
    ghT = o;  // [h4][TS] hidden pre-activation gradients (adjoint)
    o += bwd ? h4 * RN_TS * 4 : 0;
    sT = o;  // [d4][TS] scale pre-activations / tanh / their gradients
    o += d4 * RN_TS * 4;
    tT = o;  // [d4][TS] shift outputs / their gradients
    o += d4 * RN_TS * 4;
    gcT = o;  // [d4][TS] conditioning-input gradients of one MLP (adjoint)
    o += bwd ? d4 * RN_TS * 4 : 0;
    ldr = o;
    o += RN_TS * 4;
    glp = o;
    o += RN_TS * 4;
    total = o;
  }
};

#define RN_FMA16(acc, w, c)                    \
  do {                                         \
    acc[0][0] = fmaf(w.x, c.x, acc[0][0]);     \
    acc[0][1] = fmaf(w.x, c.y, acc[0][1]);     \
    acc[0][2] = fmaf(w.x, c.z, acc[0][2]);     \
    acc[0][3] = fmaf(w.x, c.w, acc[0][3]);     \
    acc[1][0] = fmaf(w.y, c.x, acc[1][0]);     \
    acc[1][1] = fmaf(w.y, c.y, acc[1][1]);     \
    acc[1][2] = fmaf(w.y, c.z, acc[1][2]);     \
    acc[1][3] = fmaf(w.y, c.w, acc[1][3]);     \
    acc[2][0] = fmaf(w.z, c.x, acc[2][0]);     \
    acc[2][1] = fmaf(w.z, c.y, acc[2][1]);     \
    acc[2][2] = fmaf(w.z, c.z, acc[2][2]);     \
    acc[2][3] = fmaf(w.z, c.w, acc[2][3]);     \
    acc[3][0] = fmaf(w.w, c.x, acc[3][0]);     \
    acc[3][1] = fmaf(w.w, c.y, acc[3][1]);     \
    acc[3][2] = fmaf(w.w, c.z, acc[3][2]);     \
    acc[3][3] = fmaf(w.w, c.w, acc[3][3]);     \
  } while (0)

// Wide product, h4 output rows: out[r][m] = sum_k W[k][r] in[k][m] (W rows of
// length h4), one 4-row x 4-sample tile per thread. MODE 0: out = relu(bias +
// .); MODE 1: out = . where hmask > 0, else 0 (ReLU derivative). Padding rows
// come out zero (zero weights and bias).
template <int MODE>
__device__ __forceinline__ void rn_wide(const float* __restrict__ W, const float* __restrict__ bias, int K, int h4,
                                        const float* inT, float* outT, const float* hmask) {
  const int tr = h4 >> 2;
  for (int o = threadIdx.x; o < tr * RN_Q; o += RN_THREADS) {
    const int jq = o % tr, q = o / tr;
    float acc[4][4];
    const float4 b = (MODE == 0) ? *reinterpret_cast<const float4*>(bias + 4 * jq) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      acc[0][v] = b.x;
      acc[1][v] = b.y;
      acc[2][v] = b.z;
      acc[3][v] = b.w;
    }
    for (int k = 0; k < K; ++k) {
      const float4 w = *reinterpret_cast<const float4*>(W + (int64_t)k * h4 + 4 * jq);
      const float4 c = *reinterpret_cast<const float4*>(inT + k * RN_TS + 4 * q);
      RN_FMA16(acc, w, c);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float4 r = make_float4(acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
      const int row = 4 * jq + u;
      if (MODE == 0) {
        r.x = fmaxf(r.x, 0.f);
        r.y = fmaxf(r.y, 0.f);
        r.z = fmaxf(r.z, 0.f);
        r.w = fmaxf(r.w, 0.f);
      } else {
        const float4 hv = *reinterpret_cast<const float4*>(hmask + row * RN_TS + 4 * q);
        r.x = hv.x > 0.f ? r.x : 0.f;
        r.y = hv.y > 0.f ? r.y : 0.f;
        r.z = hv.z > 0.f ? r.z : 0.f;
        r.w = hv.w > 0.f ? r.w : 0.f;
      }
      *reinterpret_cast<float4*>(outT + row * RN_TS + 4 * q) = r;
    }
  }
}

// Narrow product, n output rows (written up to n rounded to 4; the padding
// rows come out zero): out[r][m] = bias[r] + sum_{j < K} W[j][r] in[j][m] (W
// rows of length ldw). The reduction over j is split over S lanes of one
// wavefront (S a power of two, tiles * S <= 256) and combined with xor
// shuffles in a fixed order.
__device__ __forceinline__ void rn_narrow(const float* __restrict__ W, int ldw, const float* __restrict__ bias, int K,
                                          int n, const float* inT, float* outT) {
  const int tr = (n + 3) >> 2;
  const int tiles = tr * RN_Q;
  int S = 1;
  while (S < 64 && tiles * S * 2 <= RN_THREADS) S <<= 1;
  for (int o = threadIdx.x; o < tiles * S; o += RN_THREADS) {
    const int tile = o / S, s = o - tile * S;
    const int iq = tile % tr, q = tile / tr;
    float acc[4][4] = {};
    for (int j = s; j < K; j += S) {
      const float4 w = *reinterpret_cast<const float4*>(W + (int64_t)j * ldw + 4 * iq);
      const float4 c = *reinterpret_cast<const float4*>(inT + j * RN_TS + 4 * q);
      RN_FMA16(acc, w, c);
    }
    for (int off = S >> 1; off > 0; off >>= 1)
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[u][v] += __shfl_xor(acc[u][v], off, 64);
    if (s == 0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = 4 * iq + u;
        const float b = bias ? bias[row] : 0.f;
        *reinterpret_cast<float4*>(outT + row * RN_TS + 4 * q) =
            make_float4(acc[u][0] + b, acc[u][1] + b, acc[u][2] + b, acc[u][3] + b);
      }
    }
  }
}

// Conditioning inputs of layer l into cT (rows >= dc zero, up to d4).
__device__ __forceinline__ void rn_load_cond(const float* xs, int ldx, const int32_t* cond, int dc, int d4, float* cT) {
  for (int o = threadIdx.x; o < d4 * RN_TS; o += RN_THREADS) {
    const int k = o / RN_TS, m = o - k * RN_TS;
    cT[o] = (k < dc) ? xs[m * ldx + cond[k]] : 0.f;
  }
}

// ------------------------------------------------------------- packing ---
__global__ void __launch_bounds__(256) rnvp_pack_kernel(RnvpDev f, float* packed) {
  const int d = f.d, h = f.h, d4 = rn_r4(d), h4 = rn_r4(h);
  const int lp = blockIdx.y, l = lp >> 1, p = lp & 1;
  const int32_t* lay = rn_lay(f, l);
  const int dc = lay[0], dtr = lay[1];
  const int32_t* cond = lay + 2;
  const int32_t* trans = lay + 2 + d;
  const float* W1 = f.theta + rn_mlp(d, h, l, p);
  const float* b1 = W1 + (int64_t)h * d;
  const float* W2 = b1 + h;
  const float* b2 = W2 + (int64_t)d * h;
  float* dst = packed + rn_pk(d, h, l, p);
  const int64_t sq = (int64_t)d4 * h4, n = rn_pk_mlp(d, h);
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    float v = 0.f;
    const int region = (e < 4 * sq) ? (int)(e / sq) : 4;
    const int64_t r = e - (int64_t)region * sq;
    if (region == 0) {  // W1T[k][j]
      const int k = (int)(r / h4), j = (int)(r - (int64_t)k * h4);
      if (k < dc && j < h) v = W1[(int64_t)j * d + cond[k]];
    } else if (region == 1) {  // W1c[j][k]
      const int j = (int)(r / d4), k = (int)(r - (int64_t)j * d4);
      if (k < dc && j < h) v = W1[(int64_t)j * d + cond[k]];
    } else if (region == 2) {  // W2T[j][i]
      const int j = (int)(r / d4), i = (int)(r - (int64_t)j * d4);
      if (i < dtr && j < h) v = W2[(int64_t)trans[i] * h + j];
    } else if (region == 3) {  // W2c[i][j]
      const int i = (int)(r / h4), j = (int)(r - (int64_t)i * h4);
      if (i < dtr && j < h) v = W2[(int64_t)trans[i] * h + j];
    } else if (r < h4) {  // b1
      if (r < h) v = b1[r];
    } else {  // b2c
      const int i = (int)(r - h4);
      if (i < dtr) v = b2[trans[i]];
    }
    dst[e] = v;
  }
}

// The fragment images of one (layer, p) slot (RnFr): one thread per word.
__global__ void __launch_bounds__(256) rnvp_pack_frag_kernel(RnvpDev f, float* packed) {
  const int d = f.d, h = f.h;
  const int lp = blockIdx.y, l = lp >> 1, p = lp & 1;
  const int32_t* lay = rn_lay(f, l);
  const int dc = lay[0], dtr = lay[1];
  const int32_t* cond = lay + 2;
  const int32_t* trans = lay + 2 + d;
  const RnFr fr(packed, d, h, f.L, l, p, dc, dtr);
  const float* W1 = f.theta + rn_mlp(d, h, l, p);
  const float* b1 = W1 + (int64_t)h * d;
  const float* W2 = b1 + h;
  const float* b2 = W2 + (int64_t)d * h;
  float* dst = const_cast<float*>(fr.W1f);
  const int64_t n1 = 256LL * fr.HB * fr.KC, n2 = n1 + 256LL * fr.HB * fr.R, n3 = n2 + 16 * fr.HB, n4 = n3 + 16 * fr.R;
  const int64_t n5 = n4 + 4, n6 = n5 + 16 * fr.KC, n = n6 + 16 * fr.R;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
    float v = 0.f;
    if (e < n2) {
      const bool first = e < n1;
      const int64_t r = first ? e : e - n1;
      const int nb = first ? fr.KC : fr.R;
      const int hb = (int)(r / (256 * nb)), w = (int)(r - (int64_t)hb * 256 * nb);
      const int b = w >> 8, lane = (w >> 2) & 63, el = w & 3, c = lane & 15, k = 4 * (lane >> 4) + el;
      if (first) {
        const int j = 16 * hb + c, i = 16 * b + k;
        if (j < h && i < dc) v = W1[(int64_t)j * d + cond[i]];
      } else {
        const int i = 16 * b + c, j = 16 * hb + k;
        if (j < h && i < dtr) v = W2[(int64_t)trans[i] * h + j];
      }
    } else if (e < n3) {
      if (e - n2 < h) v = b1[e - n2];
    } else if (e < n4) {
      if (e - n3 < dtr) v = b2[trans[e - n3]];
    } else {
      int w = 0;
      if (e < n5)
        w = e == n4 ? dc : (e == n4 + 1 ? dtr : 0);
      else if (e < n6)
        w = e - n5 < dc ? cond[e - n5] : 0;
      else
        w = e - n6 < dtr ? trans[e - n6] : 0;
      v = __int_as_float(w);
    }
    dst[e] = v;
  }
}

// -------------------------------------------------------------- passes ---
struct RnPassArgs {
  int dir;    // 0 forward (realNVP.py:163-180), 1 inverse (:182-198)
  int flags;  // 1 standardize, 2 base log-prob, 4 sample base noise
  const float* x_in;
  int64_t n;
  uint32_t key0, key1;
  int64_t sample0;
  float* x_out;
  float* logdet;
  float* saved;
  const float* g_logp;
  float* gy_out;
};

enum { RN_STD = 1, RN_BASE = 2, RN_SAMPLE = 4 };

template <class K>
static int rn_set_lds(K kernel, size_t shm) {
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
  if (e != hipSuccess) {
    set_error(FMC_ERR_HIP, "hipFuncSetAttribute(%zu bytes of LDS): %s", shm, hipGetErrorString(e));
    return FMC_ERR_HIP;
  }
  return FMC_OK;
}

// The forward pass of a training step (saved layer inputs), on FMA register
// tiles: the adjoint recomputes the hidden layers with the same sums, and a
// ReLU mask that rounds differently in the two changes a weight gradient by a
// whole sample's share.
__global__ void __launch_bounds__(RN_THREADS) rnvp_train_pass_kernel(RnvpDev f, RnPassArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int d = f.d, h = f.h;
  const RnSmem sm(d, h, false);
  float* xs = reinterpret_cast<float*>(smem + sm.xs);
  float* cT = reinterpret_cast<float*>(smem + sm.cT);
  float* hT = reinterpret_cast<float*>(smem + sm.hT);
  float* sT = reinterpret_cast<float*>(smem + sm.sT);
  float* tT = reinterpret_cast<float*>(smem + sm.tT);
  float* ldr = reinterpret_cast<float*>(smem + sm.ldr);
  const int tid = threadIdx.x, ldx = sm.ldx;
  const int64_t m0 = (int64_t)blockIdx.x * RN_TS;
  const float* th = f.theta;
  const int64_t st = rn_stats(d, h, f.L);
  const float* dmean = th + st;
  const float* dcov = dmean + d;

  for (int o = tid; o < RN_TS * d; o += RN_THREADS) {
    const int m = o / d, j = o - m * d;
    const int64_t row = m0 + m;
    float v = 0.f;
    if (row < a.n) {
      v = a.x_in[row * d + j];
      if (a.flags & RN_STD) v = (v - dmean[j]) / sqrtf(dcov[(int64_t)j * d + j]);
    }
    xs[m * ldx + j] = v;
  }
  for (int m = tid; m < RN_TS; m += RN_THREADS) ldr[m] = 0.f;
  __syncthreads();

  for (int l = 0; l < f.L; ++l) {
    for (int o = tid; o < RN_TS * d; o += RN_THREADS) {
      const int m = o / d, j = o - m * d;
      if (m0 + m < a.n) a.saved[((int64_t)l * a.n + m0 + m) * d + j] = xs[m * ldx + j];
    }
    const int32_t* lay = rn_lay(f, l);
    const int dc = lay[0], dtr = lay[1];
    const int32_t* cond = lay + 2;
    const int32_t* trans = lay + 2 + d;
    rn_load_cond(xs, ldx, cond, dc, sm.d4, cT);
    __syncthreads();
    for (int p = 0; p < 2; ++p) {
      const RnPk pk(f.packed + rn_pk(d, h, l, p), sm.d4, sm.h4);
      rn_wide<0>(pk.W1T, pk.b1, dc, sm.h4, cT, hT, nullptr);
      __syncthreads();
      rn_narrow(pk.W2T, sm.d4, pk.b2c, h, dtr, hT, p == 0 ? sT : tT);
      __syncthreads();
    }
    // coupling on the transformed dims; sT keeps s for the log-det sum
    for (int o = tid; o < dtr * RN_TS; o += RN_THREADS) {
      const int i = o / RN_TS, m = o - i * RN_TS;
      const int j = trans[i];
      const float s = tanhf(sT[o]) * f.dt;
      const float t = tT[o] * f.dt;
      const float x = xs[m * ldx + j];
      xs[m * ldx + j] = (x + t) * expf(s);
      sT[o] = s;
    }
    __syncthreads();
    for (int m = tid; m < RN_TS; m += RN_THREADS) {
      float s = 0.f;
      for (int i = 0; i < dtr; ++i) s += sT[i * RN_TS + m];
      ldr[m] += s;
    }
    __syncthreads();
  }
  // ---- outputs
  for (int m = tid; m < RN_TS; m += RN_THREADS) {
    const int64_t row = m0 + m;
    if (row >= a.n) continue;
    float ld = ldr[m];
    if (a.flags & RN_BASE) {
      // log N(y; 0, I) (realNVP.py:211-213: the standard normal, not base_dist)
      float q = 0.f;
      for (int j = 0; j < d; ++j) {
        const float y = xs[m * ldx + j];
        q += y * y;
        if (a.gy_out) a.gy_out[row * d + j] = -a.g_logp[row] * y;
      }
      ld += -0.5f * q - 0.91893853320467274f * (float)d;
    }
    if (a.logdet) a.logdet[row] = ld;
  }
  if (a.x_out) {
    for (int o = tid; o < RN_TS * d; o += RN_THREADS) {
      const int m = o / d, j = o - m * d;
      const int64_t row = m0 + m;
      if (row >= a.n) continue;
      a.x_out[row * d + j] = xs[m * ldx + j];
    }
  }
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t rn_mfma(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t rn_ld4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }

// One hidden block's weight fragments (a lane's share), requested one block
// ahead of their use. Block indices past the end repeat the last block, so
// every block issues the same loads and the waits cover them exactly.
template <int NB>
struct RnFrag {
  f32x4_t w1[NB], w2[NB], b;
  __device__ __forceinline__ void load(const RnFr& f, int hb, int r0, int lane) {
    const int kc = f.KC > 0 ? f.KC : 1;  // (without conditioning dims any block of the slot serves)
#pragma unroll
    for (int k = 0; k < NB; ++k) w1[k] = rn_ld4(f.W1f + ((int64_t)hb * kc + (k < kc ? k : kc - 1)) * 256 + 4 * lane);
#pragma unroll
    for (int r = 0; r < NB; ++r)
      w2[r] = rn_ld4(f.W2f + ((int64_t)hb * f.R + (r0 + r < f.R ? r0 + r : f.R - 1)) * 256 + 4 * lane);
    b = rn_ld4(f.b1 + 16 * hb + 4 * (lane >> 4));
  }
};

// out[r][m] += W2 relu(W1 c + b1) over the hidden blocks hb0, hb0 + hs, ..,
// for the row blocks r0 .. r0 + NB - 1. The hidden block (16 features x 16
// samples) never leaves the registers: a lane's four accumulators are the
// second product's four k-steps.
template <int NB, int MB>
__device__ __forceinline__ void rn_mlp(const RnFr& f, int r0, int hb0, int hs, int dc, const f32x4_t (&c)[NB][MB],
                                       const float* xs, int ldx, f32x4_t (&out)[NB][MB], int lane) {
  if (hb0 >= f.HB) return;
  RnFrag<NB> cur, nxt;
  cur.load(f, hb0, r0, lane);
  for (int hb = hb0; hb < f.HB; hb += hs) {
    nxt.load(f, hb + hs < f.HB ? hb + hs : hb, r0, lane);
    f32x4_t a[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) a[m] = cur.b;
#pragma unroll
    for (int k = 0; k < NB; ++k)
      if (k < f.KC) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int m = 0; m < MB; ++m) a[m] = rn_mfma(cur.w1[k][e], c[k][m][e], a[m]);
      }
    for (int k = NB; k < f.KC; ++k) {  // more conditioning dims than the registers hold
      const f32x4_t w = rn_ld4(f.W1f + ((int64_t)hb * f.KC + k) * 256 + 4 * lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * k + 4 * (lane >> 4) + e;
        const int j = f.cond[i];
#pragma unroll
        for (int m = 0; m < MB; ++m)
          a[m] = rn_mfma(w[e], i < dc ? xs[(16 * m + (lane & 15)) * ldx + j] : 0.f, a[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) a[m][e] = __builtin_amdgcn_fmed3f(a[m][e], 0.f, INFINITY);
#pragma unroll
    for (int r = 0; r < NB; ++r)
      if (r0 + r < f.R) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int m = 0; m < MB; ++m) out[r][m] = rn_mfma(cur.w2[r][e], a[m][e], out[r][m]);
      }
    cur = nxt;
  }
}

// All layers of a pass for 16 MB samples on the FP32 matrix cores, which bound
// it at large n (65 % of a large FP32 product's rate at 409,600 samples, the
// rest tails, tanh / exp and weight reads); small batches are bound by the
// serial chain of hidden blocks and layers.
// SPLIT = false: every wavefront owns 16 MB samples and runs alone (no
// barrier); SPLIT = true: the eight wavefronts of a workgroup share one
// 16-sample tile, each taking one MLP (wave & 1) and every fourth hidden
// block, their partial outputs summed in LDS in a fixed order. NB: blocks of
// 16 conditioning / transformed dims held in registers; masks that leave more
// on one side take the loops over the rest.
template <int NB, int MB, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? 512 : 256) __attribute__((amdgpu_waves_per_eu(NB <= 1 ? 4 : 2)))
rnvp_pass_kernel(RnvpDev f, RnPassArgs a) {
  static_assert(!SPLIT || MB == 1, "a shared tile holds 16 samples");
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int S = 16 * MB, NT = SPLIT ? 512 : 64;
  const int d = f.d, h = f.h, ldx = d + 1;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, q = lane >> 4, t = SPLIT ? (int)threadIdx.x : lane;
  const int xsz = rn_rup16(S * ldx * 4) / 4;
  float* xs = reinterpret_cast<float*>(smem) + (SPLIT ? 0 : wave * xsz);
  float* red = reinterpret_cast<float*>(smem) + xsz;  // SPLIT: [8 waves][NB][64] float4, then [8][16] log-dets
  float* ldp = red + 8 * NB * 256;
  const int64_t m0 = ((int64_t)blockIdx.x * (SPLIT ? 1 : 4) + (SPLIT ? 0 : wave)) * S;
  if (m0 >= a.n) return;  // (a whole wavefront; a whole workgroup when the tile is shared)
  auto sync = [] {
    if constexpr (SPLIT) {
      __syncthreads();
    } else {  // LDS of this wavefront only: order its accesses
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };
  const float* th = f.theta;
  const int64_t st = rn_stats(d, h, f.L);
  const float* dmean = th + st;
  const float* dcov = dmean + d;
  const float* bmean = dcov + (int64_t)d * d;
  const float* bcov = bmean + d;

  if ((a.flags & RN_SAMPLE) && a.x_in == nullptr) {  // base noise: one Philox block per four dims
    const int ch = (d + 3) >> 2;
    for (int o = t; o < S * ch; o += NT) {
      const int m = o / ch, k = o - m * ch;
      const float4 z = philox_normal4(a.key0, a.key1, (uint32_t)k, (uint32_t)(a.sample0 + m0 + m), 0u, RNG_FLOW_BASE);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 4 * k + e;
        if (j < d) xs[m * ldx + j] = m0 + m < a.n ? bmean[j] + sqrtf(bcov[(int64_t)j * d + j]) * f4c(z, e) : 0.f;
      }
    }
  } else {
    for (int o = t; o < S * d; o += NT) {
      const int m = o / d, j = o - m * d;
      float v = 0.f;
      if (m0 + m < a.n) {
        v = a.x_in[m0 * d + o];
        if (a.dir == 0 && (a.flags & RN_STD))
          v = (v - dmean[j]) / sqrtf(dcov[(int64_t)j * d + j]);
        else if (a.dir != 0 && (a.flags & RN_SAMPLE))
          v = bmean[j] + sqrtf(bcov[(int64_t)j * d + j]) * v;
      }
      xs[m * ldx + j] = v;
    }
  }
  sync();

  float ldacc[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) ldacc[m] = 0.f;
  for (int step = 0; step < f.L; ++step) {
    const int l = (a.dir == 0) ? step : f.L - 1 - step;
    const int32_t* lay = rn_lay(f, l);
    const int dc = lay[0], dtr = lay[1];
    const RnFr fs(f.packed, d, h, f.L, l, 0, dc, dtr), ft(f.packed, d, h, f.L, l, 1, dc, dtr);
    f32x4_t c[NB][MB];  // conditioning inputs as MFMA operands
#pragma unroll
    for (int k = 0; k < NB; ++k)
      if (k < fs.KC) {
        const int4 ci = *reinterpret_cast<const int4*>(fs.cond + 16 * k + 4 * q);
        const int i0 = 16 * k + 4 * q;
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          const float* xr = xs + (16 * m + col) * ldx;
          c[k][m] = f32x4_t{i0 < dc ? xr[ci.x] : 0.f, i0 + 1 < dc ? xr[ci.y] : 0.f, i0 + 2 < dc ? xr[ci.z] : 0.f,
                            i0 + 3 < dc ? xr[ci.w] : 0.f};
        }
      }
    for (int r0 = 0; r0 < fs.R; r0 += NB) {
      f32x4_t os[NB][MB], ot[NB][MB];
#pragma unroll
      for (int r = 0; r < NB; ++r)
#pragma unroll
        for (int m = 0; m < MB; ++m) os[r][m] = ot[r][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (SPLIT) {
        rn_mlp<NB, MB>((wave & 1) ? ft : fs, r0, wave >> 1, 4, dc, c, xs, ldx, os, lane);
#pragma unroll
        for (int r = 0; r < NB; ++r) *reinterpret_cast<f32x4_t*>(red + ((wave * NB + r) * 64 + lane) * 4) = os[r][0];
        __syncthreads();
      } else {
        rn_mlp<NB, MB>(fs, r0, 0, 1, dc, c, xs, ldx, os, lane);
        rn_mlp<NB, MB>(ft, r0, 0, 1, dc, c, xs, ldx, ot, lane);
      }
      // coupling on the transformed dims: a lane holds the scale and shift of
      // dims 16 r + 4 q + e of its sample (SPLIT: row block r by wave r)
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        if (r0 + r >= fs.R || (SPLIT && wave != r)) continue;
        if constexpr (SPLIT) {
#pragma unroll
          for (int w = 0; w < 8; w += 2) {
            const f32x4_t u = rn_ld4(red + ((w * NB + r) * 64 + lane) * 4);
            const f32x4_t v = rn_ld4(red + (((w + 1) * NB + r) * 64 + lane) * 4);
            os[r][0] = w == 0 ? u : os[r][0] + u;
            ot[r][0] = w == 0 ? v : ot[r][0] + v;
          }
        }
        const int k0 = 16 * (r0 + r) + 4 * q;
        const f32x4_t bs = rn_ld4(fs.b2 + k0), bt = rn_ld4(ft.b2 + k0);
        const int4 ti = *reinterpret_cast<const int4*>(fs.trans + k0);
        const int tj[4] = {ti.x, ti.y, ti.z, ti.w};
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (k0 + e < dtr) {
              float* xp = xs + (16 * m + col) * ldx + tj[e];
              const float s = tanhf(os[r][m][e] + bs[e]) * f.dt;
              const float tt = (ot[r][m][e] + bt[e]) * f.dt;
              *xp = (a.dir == 0) ? (*xp + tt) * expf(s) : *xp * expf(-s) - tt;
              ldacc[m] += s;
            }
      }
      sync();
    }
  }
  // ---- log-det of each sample: the four lanes that share it (SPLIT: and the
  // waves), in a fixed order
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    ldacc[m] += __shfl_xor(ldacc[m], 16, 64);
    ldacc[m] += __shfl_xor(ldacc[m], 32, 64);
  }
  if constexpr (SPLIT) {
    if (lane < 16) ldp[wave * 16 + lane] = ldacc[0];
    __syncthreads();
    ldacc[0] = 0.f;
#pragma unroll
    for (int w = 0; w < NB; ++w) ldacc[0] += ldp[w * 16 + col];
  }
  // ---- outputs
  if (q == 0 && (!SPLIT || wave == 0)) {
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int64_t row = m0 + 16 * m + col;
      if (row >= a.n) continue;
      float ld = (a.dir == 0) ? ldacc[m] : -ldacc[m];
      if (a.dir == 0 && (a.flags & RN_BASE)) {
        // log N(y; 0, I) (realNVP.py:211-213: the standard normal, not base_dist)
        float s2 = 0.f;
        for (int j = 0; j < d; ++j) {
          const float y = xs[(16 * m + col) * ldx + j];
          s2 += y * y;
        }
        ld += -0.5f * s2 - 0.91893853320467274f * (float)d;
      }
      if (a.logdet) a.logdet[row] = ld;
    }
  }
  if (a.x_out || a.gy_out) {
    for (int o = t; o < S * d; o += NT) {
      const int m = o / d, j = o - m * d;
      if (m0 + m >= a.n) continue;
      float v = xs[m * ldx + j];
      if (a.gy_out) a.gy_out[m0 * d + o] = -a.g_logp[m0 + m] * v;
      if (a.x_out) {
        if (a.dir != 0 && (a.flags & RN_STD)) v = v * sqrtf(dcov[(int64_t)j * d + j]) + dmean[j];
        a.x_out[m0 * d + o] = v;
      }
    }
  }
}

template <int NB, int MB, bool SPLIT>
static int rn_launch_pass(hipStream_t st, const RnvpDev& f, const RnPassArgs& a) {
  const int xsz = rn_rup16(16 * MB * (f.d + 1) * 4);
  const size_t shm = SPLIT ? (size_t)xsz + 8 * NB * 1024 + 512 : 4 * (size_t)xsz;
  if (const int rc = rn_set_lds(rnvp_pass_kernel<NB, MB, SPLIT>, shm)) return rc;
  const int64_t per = SPLIT ? 16 : 64 * MB, grid = (a.n + per - 1) / per;
  FMC_ARG(grid <= 0x7fffffffLL, "too many samples for one launch");
  hipLaunchKernelGGL((rnvp_pass_kernel<NB, MB, SPLIT>), dim3((unsigned)grid), dim3(SPLIT ? 512 : 256), shm, st, f, a);
  return check_launch("realnvp pass");
}

// Which pass runs a batch of n samples (measured, sampling, us; d = 32, 8
// layers, hidden 256 | d = 64, 10 layers, hidden 128 | d = 5, 4 layers, hidden 64):
//   n         shared tile (8 waves)   16 samples a wave   32 samples a wave
//   1000        29 |   39 |  14          82 |   95 |  19      129 |  157 |  26
//   10000       67 |   92 |  22          86 |  101 |  18      131 |  159 |  25
//   20000      108 |  147 |  32         123 |  151 |  24      135 |  164 |  25
//   50000      262 |  350 |  75         219 |  291 |  36      211 |  261 |  36
//   409600    1825 | 2495 | 534        1177 | 1627 | 186     1101 | 1433 | 171
// A shared tile spreads the serial hidden blocks of a layer over eight waves,
// which pays until a wave for every 16 samples fills the chip's SIMDs, and
// less so the fewer hidden blocks there are to spread; 32 samples a wave halve
// the weight reads once the grid is several waves a SIMD deep. Wide states,
// whose four tiles would not leave room for two workgroups a CU, share one.
static int rn_pass_variant(int64_t n, int d, int h) {
  const int64_t tiles = (n + 15) / 16, split_to = 100 * rn_b16(h);
  if (4 * rn_rup16(16 * (d + 1) * 4) > 64 * 1024 || tiles <= (split_to < 1280 ? split_to : 1280)) return 0;
  return tiles <= 2048 ? 1 : 2;
}

template <int NB>
static int rn_pass_nb(hipStream_t st, const RnvpDev& f, const RnPassArgs& a, int var) {
  switch (var) {
    case 0: return rn_launch_pass<NB, 1, true>(st, f, a);
    case 1: return rn_launch_pass<NB, 1, false>(st, f, a);
    default: return rn_launch_pass<NB, 2, false>(st, f, a);
  }
}

// ------------------------------------------------------------- adjoint ---
// One layer in the forward direction: recompute s, t; the coupling's
// reverse sweep; per MLP the hidden gradient (W2^T g), its ReLU mask, the
// tile's weight-gradient partials, and W1^T g into the conditioning dims.
// partial layout per tile (one layer): for p = scale, shift:
//   dW1 [h][d] (column k = k-th conditioning dim), db1 [h],
//   dW2 [d][h] (row i = i-th transformed dim), db2 [d].
struct RnBwdArgs {
  int layer;
  const float* x_in;  // [n, d] layer input
  int64_t n;
  const float* g_logp;
  const float* gy;  // [n, d] dL/d(layer output)
  float* gx;        // [n, d] dL/d(layer input)
  float* part;      // [n_tiles, layer_size]
};

// out[a][b] = sum_m A[a][m] B[b][m] over the tile's 32 samples, 4x4 register
// tiles; A has na rows (storage padded to na4), B nb rows (padded to nb4).
__device__ __forceinline__ void rn_outer(const float* A, int na, const float* B, int nb, float* out, int ldo) {
  const int na4 = (na + 3) >> 2, nb4 = (nb + 3) >> 2;
  for (int o = threadIdx.x; o < na4 * nb4; o += RN_THREADS) {
    const int ta = o / nb4, tb = o - ta * nb4;
    float acc[4][4] = {};
#pragma unroll 1
    for (int q = 0; q < RN_Q; ++q) {
      float4 av[4], bv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        av[u] = *reinterpret_cast<const float4*>(A + (4 * ta + u) * RN_TS + 4 * q);
        bv[u] = *reinterpret_cast<const float4*>(B + (4 * tb + u) * RN_TS + 4 * q);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[u][v] += av[u].x * bv[v].x + av[u].y * bv[v].y + av[u].z * bv[v].z + av[u].w * bv[v].w;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int ia = 4 * ta + u, ib = 4 * tb + v;
        if (ia < na && ib < nb) out[(int64_t)ia * ldo + ib] = acc[u][v];
      }
  }
}

__device__ __forceinline__ void rn_rowsum(const float* A, int na, float* out) {
  for (int i = threadIdx.x; i < na; i += RN_THREADS) {
    float s = 0.f;
    for (int m = 0; m < RN_TS; ++m) s += A[i * RN_TS + m];
    out[i] = s;
  }
}

__global__ void __launch_bounds__(RN_THREADS) rnvp_bwd_kernel(RnvpDev f, RnBwdArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int d = f.d, h = f.h, l = a.layer;
  const RnSmem sm(d, h, true);
  float* xs = reinterpret_cast<float*>(smem + sm.xs);
  float* gb = reinterpret_cast<float*>(smem + sm.gb);
  float* cT = reinterpret_cast<float*>(smem + sm.cT);
  float* hT = reinterpret_cast<float*>(smem + sm.hT);
  float* ghT = reinterpret_cast<float*>(smem + sm.ghT);
  float* sT = reinterpret_cast<float*>(smem + sm.sT);
  float* tT = reinterpret_cast<float*>(smem + sm.tT);
  float* gcT = reinterpret_cast<float*>(smem + sm.gcT);
  float* glp = reinterpret_cast<float*>(smem + sm.glp);
  const int tid = threadIdx.x, ldx = sm.ldx;
  const int64_t m0 = (int64_t)blockIdx.x * RN_TS;
  const int32_t* lay = rn_lay(f, l);
  const int dc = lay[0], dtr = lay[1];
  const int32_t* cond = lay + 2;
  const int32_t* trans = lay + 2 + d;

  for (int o = tid; o < RN_TS * d; o += RN_THREADS) {
    const int m = o / d, j = o - m * d;
    const int64_t row = m0 + m;
    const bool ok = row < a.n;
    xs[m * ldx + j] = ok ? a.x_in[row * d + j] : 0.f;
    gb[m * ldx + j] = ok ? a.gy[row * d + j] : 0.f;
  }
  for (int m = tid; m < RN_TS; m += RN_THREADS) glp[m] = (m0 + m < a.n) ? a.g_logp[m0 + m] : 0.f;
  __syncthreads();
  rn_load_cond(xs, ldx, cond, dc, sm.d4, cT);
  __syncthreads();
  // ---- recompute scale / shift pre-activations
  for (int p = 0; p < 2; ++p) {
    const RnPk pk(f.packed + rn_pk(d, h, l, p), sm.d4, sm.h4);
    rn_wide<0>(pk.W1T, pk.b1, dc, sm.h4, cT, hT, nullptr);
    __syncthreads();
    rn_narrow(pk.W2T, sm.d4, pk.b2c, h, dtr, hT, p == 0 ? sT : tT);
    __syncthreads();
  }
  // ---- coupling reverse sweep: y = (x + t) e^s, log-det += s
  //   g_x = g e^s (transformed dim), g_t = g e^s, g_s = g y + g_logp;
  //   g_spre = g_s dt (1 - tanh^2), g_tpre = g_t dt (in place of sT / tT;
  //   their padding rows stay zero)
  for (int o = tid; o < dtr * RN_TS; o += RN_THREADS) {
    const int i = o / RN_TS, m = o - i * RN_TS;
    const int j = trans[i];
    const float tn = tanhf(sT[o]);
    const float s = tn * f.dt;
    const float t = tT[o] * f.dt;
    const float e = expf(s);
    const float x = xs[m * ldx + j];
    const float y = (x + t) * e;
    const float g = gb[m * ldx + j];
    const float ge = g * e;
    gb[m * ldx + j] = ge;
    sT[o] = (g * y + glp[m]) * f.dt * (1.f - tn * tn);
    tT[o] = ge * f.dt;
  }
  __syncthreads();
  float* part = a.part + (int64_t)blockIdx.x * rn_layer_size(d, h);
  for (int p = 0; p < 2; ++p) {
    const RnPk pk(f.packed + rn_pk(d, h, l, p), sm.d4, sm.h4);
    const float* goT = (p == 0) ? sT : tT;
    float* pp = part + p * rn_mlp_size(d, h);
    rn_wide<0>(pk.W1T, pk.b1, dc, sm.h4, cT, hT, nullptr);
    __syncthreads();
    // g_H[j][m] = sum_i W2[trans_i][j] g_out[i][m], masked by ReLU' (H > 0)
    rn_wide<1>(pk.W2c, nullptr, dtr, sm.h4, goT, ghT, hT);
    __syncthreads();
    // tile partials: dW1[j][k] = sum_m gH[j][m] c[k][m]; db1; dW2[i][j] = sum_m g_out[i][m] H[j][m]; db2
    rn_outer(ghT, h, cT, dc, pp, d);
    rn_rowsum(ghT, h, pp + (int64_t)h * d);
    rn_outer(goT, dtr, hT, h, pp + (int64_t)h * d + h, h);
    rn_rowsum(goT, dtr, pp + 2LL * h * d + h);
    // g_c[k][m] = sum_j W1[j][cond_k] gH[j][m], added to the conditioning dims
    rn_narrow(pk.W1c, sm.d4, nullptr, h, dc, ghT, gcT);
    __syncthreads();
    for (int o = tid; o < dc * RN_TS; o += RN_THREADS) {
      const int k = o / RN_TS, m = o - k * RN_TS;
      gb[m * ldx + cond[k]] += gcT[o];
    }
    __syncthreads();
  }
  for (int o = tid; o < RN_TS * d; o += RN_THREADS) {
    const int m = o / d, j = o - m * d;
    const int64_t row = m0 + m;
    if (row < a.n) a.gx[row * d + j] = gb[m * ldx + j];
  }
}

// Sum of the tile partials of one layer, in two fixed-order stages so that
// enough lanes stream the partial buffer: stage 1 sums chunk c of the tiles
// (tiles c, c + C, c + 2C, ...) into row n_tiles + c of the buffer; stage 2
// sums the C chunk rows in order and scatters the result to the
// reference-shaped leaves of the gradient vector.
constexpr int RN_RED_CHUNKS = 16;

__host__ __device__ inline int rn_chunks(int64_t n_tiles) {
  const int64_t c = (n_tiles + 15) / 16;
  return (int)(c < 1 ? 1 : (c > RN_RED_CHUNKS ? RN_RED_CHUNKS : c));
}

__global__ void __launch_bounds__(256) rnvp_wgrad_stage1(int64_t LS, float* part, int64_t n_tiles, int C) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (e >= LS) return;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  int64_t t = c;
  for (; t + 3 * C < n_tiles; t += 4 * C) {
    s0 += part[t * LS + e];
    s1 += part[(t + C) * LS + e];
    s2 += part[(t + 2 * C) * LS + e];
    s3 += part[(t + 3 * C) * LS + e];
  }
  for (; t < n_tiles; t += C) s0 += part[t * LS + e];
  part[(n_tiles + c) * LS + e] = (s0 + s1) + (s2 + s3);
}

__global__ void __launch_bounds__(256) rnvp_wgrad_stage2(RnvpDev f, int l, const float* __restrict__ part,
                                                         int64_t n_tiles, int C, float* __restrict__ grad) {
  const int d = f.d, h = f.h;
  const int64_t LS = rn_layer_size(d, h), MS = rn_mlp_size(d, h);
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= LS) return;
  const int32_t* lay = rn_lay(f, l);
  const int dc = lay[0], dtr = lay[1];
  const int32_t* cond = lay + 2;
  const int32_t* trans = lay + 2 + d;
  const int p = (int)(e / MS);
  const int64_t r = e - p * MS;
  int64_t dst = -1;
  if (r < (int64_t)h * d) {
    const int j = (int)(r / d), k = (int)(r - (int64_t)j * d);
    if (k < dc) dst = (int64_t)j * d + cond[k];
  } else if (r < (int64_t)h * d + h) {
    dst = r;
  } else if (r < 2LL * h * d + h) {
    const int64_t rr = r - (int64_t)h * d - h;
    const int i = (int)(rr / h), j = (int)(rr - (int64_t)i * h);
    if (i < dtr) dst = (int64_t)h * d + h + (int64_t)trans[i] * h + j;
  } else {
    const int i = (int)(r - 2LL * h * d - h);
    if (i < dtr) dst = 2LL * h * d + h + trans[i];
  }
  if (dst < 0) return;
  float s = 0.f;
  for (int c = 0; c < C; ++c) s += part[(n_tiles + c) * LS + e];
  grad[rn_mlp(d, h, l, p) + dst] = s;
}

static int check_rnvp(const fmc_rnvp* r, RnvpDev& f, bool need_packed) {
  FMC_ARG(r != nullptr, "RealNVP description is NULL");
  FMC_ARG(r->n_dim >= 1 && r->n_layers >= 1 && r->n_hidden >= 1, "n_dim, n_layers and n_hidden must be >= 1");
  FMC_ARG(r->theta != nullptr && r->layout != nullptr, "theta or layout is NULL");
  FMC_ARG(!need_packed || r->packed != nullptr, "packed buffer is NULL");
  const RnSmem sm(r->n_dim, r->n_hidden, true);
  FMC_ARG(sm.total <= 160 * 1024, "n_dim %d / n_hidden %d exceed the LDS budget of the RealNVP kernels",
          r->n_dim, r->n_hidden);
  f = RnvpDev{r->n_dim, r->n_layers, r->n_hidden, r->dt, r->theta, r->packed, r->layout};
  return FMC_OK;
}

}  // namespace fmc

using namespace fmc;

extern "C" int fmc_rnvp_sizes(const fmc_rnvp* r, int64_t* theta_size, int64_t* packed_size,
                              int64_t* partial_per_tile, int32_t* tile) {
  RnvpDev f;
  int rc = check_rnvp(r, f, false);
  if (rc) return rc;
  if (theta_size) *theta_size = rn_theta_size(f.d, f.h, f.L);
  if (packed_size) *packed_size = rn_packed_size(f.d, f.h, f.L);
  if (partial_per_tile) *partial_per_tile = rn_layer_size(f.d, f.h);  // rows: tiles + chunk rows
  if (tile) *tile = RN_TS;
  return FMC_OK;
}

extern "C" int fmc_rnvp_pack(void* stream, const fmc_rnvp* r) {
  RnvpDev f;
  int rc = check_rnvp(r, f, true);
  if (rc) return rc;
  const int64_t n = rn_pk_mlp(f.d, f.h);
  const unsigned gx = (unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
  hipLaunchKernelGGL(rnvp_pack_kernel, dim3(gx, 2 * f.L), dim3(256), 0, (hipStream_t)stream, f, r->packed);
  if ((rc = check_launch("realnvp pack"))) return rc;
  const int64_t nf = rn_fr_slot(f.d, f.h);
  hipLaunchKernelGGL(rnvp_pack_frag_kernel, dim3((unsigned)((nf + 255) / 256 < 4096 ? (nf + 255) / 256 : 4096), 2 * f.L),
                     dim3(256), 0, (hipStream_t)stream, f, r->packed);
  return check_launch("realnvp pack (fragments)");
}

extern "C" int fmc_rnvp_pass(void* stream, const fmc_rnvp* r, int32_t dir, int32_t flags, const float* x_in,
                             int64_t n, uint32_t key0, uint32_t key1, int64_t sample0, float* x_out, float* logdet,
                             float* saved, const float* g_logp, float* gy_out) {
  RnvpDev f;
  int rc = check_rnvp(r, f, true);
  if (rc) return rc;
  FMC_ARG(dir == 0 || dir == 1, "dir must be 0 (forward) or 1 (inverse)");
  FMC_ARG(n >= 0, "n < 0");
  FMC_ARG(x_in != nullptr || (flags & RN_SAMPLE), "x_in is NULL and base sampling is off");
  FMC_ARG(!(flags & RN_SAMPLE) || dir == 1, "base sampling needs the inverse direction");
  FMC_ARG(!(flags & RN_BASE) || dir == 0, "the base log-prob is added in the forward direction only");
  FMC_ARG(saved == nullptr || dir == 0, "saved layer inputs need the forward direction");
  FMC_ARG(gy_out == nullptr || (g_logp != nullptr && (flags & RN_BASE)), "gy_out needs g_logp and BASE_LOGP");
  if (n == 0) return FMC_OK;
  RnPassArgs a{dir, flags, x_in, n, key0, key1, sample0, x_out, logdet, saved, g_logp, gy_out};
  hipStream_t st = (hipStream_t)stream;
  if (saved) {
    const RnSmem sm(f.d, f.h, false);
    if ((rc = rn_set_lds(rnvp_train_pass_kernel, (size_t)sm.total))) return rc;
    const int64_t grid = (n + RN_TS - 1) / RN_TS;
    FMC_ARG(grid <= 0x7fffffffLL, "too many samples for one launch");
    hipLaunchKernelGGL(rnvp_train_pass_kernel, dim3((unsigned)grid), dim3(RN_THREADS), (size_t)sm.total, st, f, a);
    return check_launch("realnvp training pass");
  }
  const int nb = rn_b16((f.d + 1) / 2);  // blocks of a mask that halves the dims
  const int var = rn_pass_variant(n, f.d, f.h);
  if (nb <= 1) return rn_pass_nb<1>(st, f, a, var);
  if (nb <= 2) return rn_pass_nb<2>(st, f, a, var);
  return rn_pass_nb<4>(st, f, a, var);
}

extern "C" int fmc_rnvp_backward_layer(void* stream, const fmc_rnvp* r, int32_t layer, const float* x_in, int64_t n,
                                       const float* g_logp, const float* gy, float* gx, float* partials,
                                       int64_t n_partial_tiles) {
  RnvpDev f;
  int rc = check_rnvp(r, f, true);
  if (rc) return rc;
  FMC_ARG(layer >= 0 && layer < f.L, "layer %d out of range", layer);
  FMC_ARG(n >= 0, "n < 0");
  FMC_ARG(x_in && g_logp && gy && gx && partials, "NULL pointer");
  FMC_ARG(gy != gx, "gx must not alias gy");
  const int64_t tiles = (n + RN_TS - 1) / RN_TS;
  FMC_ARG(n_partial_tiles >= tiles, "partials hold %lld tiles, %lld needed", (long long)n_partial_tiles,
          (long long)tiles);
  if (n == 0) return FMC_OK;
  const RnSmem sm(f.d, f.h, true);
  if ((rc = rn_set_lds(rnvp_bwd_kernel, (size_t)sm.total))) return rc;
  RnBwdArgs a{layer, x_in, n, g_logp, gy, gx, partials};
  hipLaunchKernelGGL(rnvp_bwd_kernel, dim3((unsigned)tiles), dim3(RN_THREADS), (size_t)sm.total,
                     (hipStream_t)stream, f, a);
  return check_launch("realnvp adjoint");
}

extern "C" int fmc_rnvp_weight_grad(void* stream, const fmc_rnvp* r, int32_t layer, float* partials,
                                    int64_t n_tiles, int64_t partial_rows, float* grad) {
  RnvpDev f;
  int rc = check_rnvp(r, f, false);
  if (rc) return rc;
  FMC_ARG(layer >= 0 && layer < f.L, "layer %d out of range", layer);
  FMC_ARG(partials && grad, "NULL pointer");
  FMC_ARG(n_tiles >= 1, "n_tiles must be >= 1");
  const int C = rn_chunks(n_tiles);
  FMC_ARG(partial_rows >= n_tiles + C, "partials hold %lld rows, %lld needed (tiles + %d reduction rows)",
          (long long)partial_rows, (long long)(n_tiles + C), C);
  const int64_t LS = rn_layer_size(f.d, f.h);
  const unsigned gx = (unsigned)((LS + 255) / 256);
  hipLaunchKernelGGL(rnvp_wgrad_stage1, dim3(gx, C), dim3(256), 0, (hipStream_t)stream, LS, partials, n_tiles, C);
  if ((rc = check_launch("realnvp weight gradient (tile sums)"))) return rc;
  hipLaunchKernelGGL(rnvp_wgrad_stage2, dim3(gx), dim3(256), 0, (hipStream_t)stream, f, layer, partials, n_tiles,
                     C, grad);
  return check_launch("realnvp weight gradient");
}
