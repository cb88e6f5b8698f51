// RealNVP flow kernels for gfx950 (src/flowMC/resource/model/nf_model/
// realNVP.py). Per layer a masked coupling layer whose scale and shift MLPs
// ([d, hidden, d], ReLU; common.py:68-112, 171-208) read the conditioning
// dims and drive the transformed dims:
//   s = tanh(MLP_s(c)) dt,  t = MLP_t(c) dt,  y = (x + t) e^s,  log-det = sum s.
// The model is FP32 end to end and every product runs on the FP32 matrix
// cores (v_mfma_f32_16x16x4: the FP32 vector rate without packed forms is half
// of it; one instruction is four FMAs in k order, bit for bit, so a chain of
// them sums in the order its operands are laid out in). A hidden block of 16
// features x 16 samples stays in registers from the first product to the
// next: a lane's four accumulators are the second product's four k-steps.
//   passes   409,600 samples at d = 32, 8 layers, hidden 256 drawn in 1.17 ms,
//            92 TFLOP/s (FMA register tiles over LDS: 4.05 ms)
//   training one step of 10,000 samples, same flow: 0.32 ms (1.10 ms with FMA
//            tiles, one adjoint launch a layer and a partial weight gradient
//            for every 16 samples): forward 72 us, adjoint of all layers 205,
//            weight-gradient sums 19
// Sums keep short chains that are added pairwise (rn_mlp, RnOrder, the adjoint):
// the matrix cores would as well add everything in one.
#include "fmc_common.h"

namespace fmc {

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
// ---- layout: per layer [n_cond, n_trans, cond[d], trans[d]]
__host__ __device__ inline const int32_t* rn_lay(const RnvpDev& f, int l) { return f.layout + (int64_t)l * (2 + 2 * f.d); }

__host__ __device__ inline int rn_rup16(int v) { return (v + 15) & ~15; }
__host__ __device__ inline int rn_b16(int v) { return (v + 15) >> 4; }

// ---- packed copy: MFMA fragment images per (layer, p). Blocks of 16
// conditioning dims (kg < KC), 16 transformed dims (r < R) and 16 hidden
// features (hb < HB); one 16 x 16 weight block is 64 lanes x float4, lane l
// (c = l % 16, q = l / 16) holding element e of four k-steps:
//   W1f [hb][kg]: W1[16 hb + c][cond(16 kg + 4e + q)]   (k in dim order)
//   W2f [hb][r]:  W2[trans(16 r + c)][16 hb + 4q + e]
//   W2t [hb][r]:  W2[trans(16 r + 4e + q)][16 hb + c]
//   W1t [hb][kg]: W1[16 hb + 4q + e][cond(16 kg + c)]
// b1 [16 HB], b2 [16 R]; the training forward's images W1s [blk][kg],
// W2s [blk][r], b1s [16 blk] with the hidden features in its summation order
// (RnOrder: row 4q + i of block blk is feature (blk, q, i)); and the index
// words cond [16 KC], the same in fragment order (word 4q + e of a block is
// cond 4e + q), trans [16 R], padding entries 0. Slots have a fixed size: KC +
// R <= ceil(d / 16) + 1 whatever the mask, and at most HB + 16 ordered blocks.
struct RnOrder {
  // The sum over the hidden features of one output: S strided partial sums
  // (features s, s + S, ..: one chain each), then pairs at distance S/2, S/4,
  // .., 1. S = 256 / (4 ceil(n_trans / 4)) rounded down to a power of two <= 64.
  // An ordered block holds 16 features: its k-step i (element i of all four
  // q) belongs to one chain, so the four chains s, s + S/2, s + S/4, s + 3S/4
  // (S >= 4) advance by four features each and end in two levels of pairs.
  int S, Sg, G, U;  // chains; chains of a block; blocks side by side; blocks along a chain
  __host__ __device__ RnOrder(int dtr, int h) {
    const int tiles = 4 * ((dtr + 3) >> 2);
    S = 1;
    while (S < 64 && tiles * S * 2 <= 256) S <<= 1;
    Sg = S < 4 ? S : 4;
    G = S / Sg;
    U = (h + S * (16 / Sg) - 1) / (S * (16 / Sg));
  }
  __host__ __device__ int blocks() const { return G * U; }
  __host__ __device__ int feature(int blk, int q, int i) const {
    const int g = blk / U, u = blk - g * U, k = i % Sg;
    const int s = S >= 4 ? g + (k & 1) * (S >> 1) + (k >> 1) * (S >> 2) : k;
    return s + S * ((u * (4 / Sg) + i / Sg) * 4 + q);
  }
};
__host__ __device__ inline int64_t rn_slot(int d, int h) {
  const int kr = rn_b16(d) + 1, hb = rn_b16(h);
  const int64_t w = 512LL * hb * kr + 16LL * hb + 16LL * rn_b16(d) + 256LL * (hb + 16) * kr + 16LL * (hb + 16) + 32LL * kr;
  return (w + 15) & ~15LL;
}
__host__ __device__ inline int64_t rn_packed_size(int d, int h, int L) { return 2LL * L * rn_slot(d, h); }
struct RnFr {
  int KC, R, HB;
  const float *W1f, *W2f, *W2t, *W1t, *b1, *b2, *W1s, *W2s, *b1s;
  const int32_t *cond, *condf, *trans;
  __device__ RnFr(const float* packed, int d, int h, int l, int p, int dc, int dtr) {
    KC = rn_b16(dc);
    R = rn_b16(dtr);
    HB = rn_b16(h);
    const int nb = RnOrder(dtr, h).blocks();
    W1f = packed + (2LL * l + p) * rn_slot(d, h);
    W1t = W1f + 256LL * HB * KC;
    W2f = W1t + 256LL * HB * KC;
    W2t = W2f + 256LL * HB * R;
    b1 = W2t + 256LL * HB * R;
    b2 = b1 + 16 * HB;
    W1s = b2 + 16 * R;
    W2s = W1s + 256LL * nb * KC;
    b1s = W2s + 256LL * nb * R;
    cond = reinterpret_cast<const int32_t*>(b1s + 16 * nb);
    condf = cond + 16 * KC;
    trans = condf + 16 * KC;
  }
};

// ------------------------------------------------------------- packing ---
// One thread per float4 of one (layer, p) slot (whose size fits 31 bits: d and
// h are bounded by the kernels' LDS).
__global__ void __launch_bounds__(256) rnvp_pack_kernel(RnvpDev f, float* packed) {
  const int d = f.d, h = f.h;
  const int lp = blockIdx.y, l = lp >> 1, p = lp & 1;
  const int32_t* lay = rn_lay(f, l);
  const int dc = lay[0], dtr = lay[1];
  const int32_t* cond = lay + 2;
  const int32_t* trans = lay + 2 + d;
  const RnFr fr(packed, d, h, l, p, dc, dtr);
  const RnOrder ord(dtr, h);
  const float* W1 = f.theta + rn_mlp(d, h, l, p);
  const float* b1 = W1 + (int64_t)h * d;
  const float* W2 = b1 + h;
  const float* b2 = W2 + (int64_t)d * h;
  float* dst = const_cast<float*>(fr.W1f);
  const int64_t n = reinterpret_cast<const float*>(fr.trans + 16 * fr.R) - dst;
  const int n4 = (int)(n >> 2), oW1t = (int)(fr.W1t - dst), oW2f = (int)(fr.W2f - dst), oW2t = (int)(fr.W2t - dst);
  const int ob1 = (int)(fr.b1 - dst), ob2 = (int)(fr.b2 - dst), oW1s = (int)(fr.W1s - dst), oW2s = (int)(fr.W2s - dst);
  const int ob1s = (int)(fr.b1s - dst), oc = (int)(reinterpret_cast<const float*>(fr.cond) - dst);
  const int ocf = oc + 16 * fr.KC, ot = ocf + 16 * fr.KC;
  for (int e4 = blockIdx.x * 256 + threadIdx.x; e4 < n4; e4 += gridDim.x * 256) {
    const int e0 = 4 * e4;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (e0 < ob1 || (e0 >= oW1s && e0 < ob1s)) {  // a weight image
      const bool sorted = e0 >= oW1s;
      const bool w1 = sorted ? e0 < oW2s : e0 < oW2f;  // W1f, W1t, W1s
      const bool tr = !sorted && ((e0 >= oW1t && e0 < oW2f) || e0 >= oW2t);
      const int r = e0 - (sorted ? (w1 ? oW1s : oW2s) : w1 ? (tr ? oW1t : 0) : (tr ? oW2t : oW2f));
      const int nb = w1 ? fr.KC : fr.R;
      const int blk = r >> 8, hb = blk / nb, b = blk - hb * nb, lane = (r >> 2) & 63, c = lane & 15, q = lane >> 4;
      const bool rows = w1 != tr;  // W1f, W1s, W2t: lane c is a feature, k the dims; else k the features
      const int jr = sorted ? ord.feature(hb, c >> 2, c & 3) : 16 * hb + c;
#pragma unroll
      for (int el = 0; el < 4; ++el) {
        const int j = rows ? jr : sorted ? ord.feature(hb, q, el) : 16 * hb + 4 * q + el;
        const int i = rows ? 16 * b + 4 * el + q : 16 * b + c;
        if (j < h && i < (w1 ? dc : dtr)) v[el] = w1 ? W1[(int64_t)j * d + cond[i]] : W2[(int64_t)trans[i] * h + j];
      }
    } else {
#pragma unroll
      for (int el = 0; el < 4; ++el) {
        const int e = e0 + el;
        if (e < ob2) {
          if (e - ob1 < h) v[el] = b1[e - ob1];
        } else if (e < oW1s) {
          if (e - ob2 < dtr) v[el] = b2[trans[e - ob2]];
        } else if (e < oc) {
          const int w = e - ob1s, j = ord.feature(w >> 4, (w >> 2) & 3, w & 3);
          if (j < h) v[el] = b1[j];
        } else {
          int w = 0;
          if (e < ocf) {
            w = e - oc < dc ? cond[e - oc] : 0;
          } else if (e < ot) {
            const int u = e - ocf, i = (u & ~15) + 4 * (u & 3) + ((u >> 2) & 3);
            w = i < dc ? cond[i] : 0;
          } else {
            w = e - ot < dtr ? trans[e - ot] : 0;
          }
          v[el] = __int_as_float(w);
        }
      }
    }
    reinterpret_cast<float4*>(dst)[e4] = make_float4(v[0], v[1], v[2], v[3]);
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

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t rn_mfma(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// (partial weight gradients may start at any float of a caller's buffer)
typedef float f32x4_a4_t __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f32x4_t rn_ld4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
__device__ __forceinline__ float rn_relu(float v) { return __builtin_amdgcn_fmed3f(v, 0.f, INFINITY); }

// A state row's conditioning dims 16 k + 4e + q, e = 0..3, as a lane's four
// k-steps (padding 0); xr: the row of the lane's sample
__device__ __forceinline__ f32x4_t rn_cond4(const RnFr& f, const float* xr, int k, int q, int dc) {
  const int4 ci = *reinterpret_cast<const int4*>(f.condf + 16 * k + 4 * q);
  const f32x4_t v{xr[ci.x], xr[ci.y], xr[ci.z], xr[ci.w]};
  const int i = 16 * k + q;
  return f32x4_t{i < dc ? v[0] : 0.f, i + 4 < dc ? v[1] : 0.f, i + 8 < dc ? v[2] : 0.f, i + 12 < dc ? v[3] : 0.f};
}

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

// Adds the hidden blocks' outputs pairwise in groups of 2^LV and the groups
// one after the other: the count of blocks so far says which partials merge.
template <int MB, int LV>
struct RnPairSum {
  static_assert(LV == 2 || LV == 3, "levels of pairs");
  f32x4_t l0[MB], l1[MB], l2[LV == 3 ? MB : 1], total[MB];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      l0[m] = l1[m] = total[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (LV == 3) l2[m] = total[m];
    }
  }
  __device__ __forceinline__ void add(f32x4_t (&v)[MB], int j) {  // block j (0, 1, ..)
    auto merge = [&](f32x4_t (&l)[MB], bool up) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        if (up)
          v[m] = l[m] + v[m];
        else
          l[m] = v[m];
      }
      return up;
    };
    if (!merge(l0, j & 1) || !merge(l1, j & 2)) return;
    if constexpr (LV == 3)
      if (!merge(l2, j & 4)) return;
#pragma unroll
    for (int m = 0; m < MB; ++m) total[m] += v[m];
  }
  // the sum after n blocks (partials without a partner, smallest first)
  __device__ __forceinline__ void finish(int n, f32x4_t (&out)[MB]) const {
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      f32x4_t v{0.f, 0.f, 0.f, 0.f};
      if (n & 1) v = l0[m];
      if (n & 2) v = l1[m] + v;
      if constexpr (LV == 3)
        if (n & 4) v = l2[m] + v;
      out[m] = total[m] + v;
    }
  }
};

// out[r][m] = W2 relu(W1 c + b1) over the hidden blocks hb0, hb0 + hs, ..,
// for the row blocks r0 .. r0 + NB - 1. The hidden block (16 features x 16
// samples) never leaves the registers: a lane's four accumulators are the
// second product's four k-steps. The sum over the features starts a chain
// anew every LEAF of them and adds the chains pairwise: one chain through the
// whole layer had 1.5 times the error of the outputs at d = 32, hidden 256
// (rms against FP64 2.8e-7 / 1.8e-7) and 2.3 times at hidden 1000.
template <int NB, int MB, int LEAF>
__device__ __forceinline__ void rn_mlp(const RnFr& f, int r0, int hb0, int hs, int dc, const f32x4_t (&c)[NB][MB],
                                       const float* xs, int ldx, f32x4_t (&out)[NB][MB], int lane) {
  constexpr int N = 16 / LEAF;  // chains of a block, one every LEAF / 4 k-steps
  static_assert(N == 2 || N == 4, "chains of a block");
  RnPairSum<MB, N == 4 ? 3 : 2> sum[NB];  // (three levels beside chains of eight spill)
#pragma unroll
  for (int r = 0; r < NB; ++r) sum[r].clear();
  RnFrag<NB> cur, nxt;
  if (hb0 < f.HB) cur.load(f, hb0, r0, lane);
  int j = 0;
  for (int hb = hb0; hb < f.HB; hb += hs, ++j) {
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
      for (int m = 0; m < MB; ++m) {
        const f32x4_t cv = rn_cond4(f, xs + (16 * m + (lane & 15)) * ldx, k, lane >> 4, dc);
#pragma unroll
        for (int e = 0; e < 4; ++e) a[m] = rn_mfma(w[e], cv[e], a[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) a[m][e] = rn_relu(a[m][e]);
#pragma unroll
    for (int r = 0; r < NB; ++r)
      if (r0 + r < f.R) {
        f32x4_t t[N][MB], v[MB];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int m = 0; m < MB; ++m)
            t[e * N / 4][m] = rn_mfma(cur.w2[r][e], a[m][e],
                                      e % (4 / N) == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : t[e * N / 4][m]);
#pragma unroll
        for (int m = 0; m < MB; ++m)
          v[m] = N == 2 ? t[0][m] + t[N - 1][m] : (t[0][m] + t[1][m]) + (t[N / 2][m] + t[N - 1][m]);
        sum[r].add(v, j);
      }
    cur = nxt;
  }
#pragma unroll
  for (int r = 0; r < NB; ++r) sum[r].finish(j, out[r]);
}

// fine: chains of four features instead of eight, where the sum over S strided
// chains and their pairs (RnOrder) has chains that short: the error is then no
// larger than that sum's at any width.
template <int NB, int MB>
__device__ __forceinline__ void rn_mlp(bool fine, const RnFr& f, int r0, int hb0, int hs, int dc,
                                       const f32x4_t (&c)[NB][MB], const float* xs, int ldx, f32x4_t (&out)[NB][MB],
                                       int lane) {
  if (fine)
    rn_mlp<NB, MB, 4>(f, r0, hb0, hs, dc, c, xs, ldx, out, lane);
  else
    rn_mlp<NB, MB, 8>(f, r0, hb0, hs, dc, c, xs, ldx, out, lane);
}

// All layers of a pass for 16 MB samples on the FP32 matrix cores, which bound
// it at large n (61 % of a large FP32 product's rate at 409,600 samples, the
// rest the pairwise sums, tails, tanh / exp and weight reads; one chain a layer
// for 1.10 ms, see rn_mlp); small batches are bound by the serial chain of
// hidden blocks and layers.
// SPLIT = false: every wavefront owns 16 MB samples and runs alone (no
// barrier); SPLIT = true: the eight wavefronts of a workgroup share one
// 16-sample tile, each taking one MLP (wave & 1) and every fourth hidden
// block, their partial outputs summed in LDS in a fixed order. NB: blocks of
// 16 conditioning / transformed dims held in registers; masks that leave more
// on one side take the loops over the rest.
template <int NB, int MB, bool SPLIT>
__global__ void __launch_bounds__(SPLIT ? 512 : 256) __attribute__((amdgpu_waves_per_eu(NB <= 1 || (SPLIT && NB == 2) ? 4 : 2)))
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
    const RnFr fs(f.packed, d, h, l, 0, dc, dtr), ft(f.packed, d, h, l, 1, dc, dtr);
    const bool fine = h < 8 * RnOrder(dtr, h).S;
    float ls[MB];  // the layer's share of the log-dets
#pragma unroll
    for (int m = 0; m < MB; ++m) ls[m] = 0.f;
    f32x4_t c[NB][MB];  // conditioning inputs as MFMA operands
#pragma unroll
    for (int k = 0; k < NB; ++k)
      if (k < fs.KC) {
#pragma unroll
        for (int m = 0; m < MB; ++m) c[k][m] = rn_cond4(fs, xs + (16 * m + col) * ldx, k, q, dc);
      }
    for (int r0 = 0; r0 < fs.R; r0 += NB) {
      f32x4_t os[NB][MB], ot[NB][MB];
      if constexpr (SPLIT) {
        rn_mlp<NB, MB>(fine, (wave & 1) ? ft : fs, r0, wave >> 1, 4, dc, c, xs, ldx, os, lane);
#pragma unroll
        for (int r = 0; r < NB; ++r) *reinterpret_cast<f32x4_t*>(red + ((wave * NB + r) * 64 + lane) * 4) = os[r][0];
        __syncthreads();
      } else {
        rn_mlp<NB, MB>(fine, fs, r0, 0, 1, dc, c, xs, ldx, os, lane);
        rn_mlp<NB, MB>(fine, ft, r0, 0, 1, dc, c, xs, ldx, ot, lane);
      }
      // coupling on the transformed dims: a lane holds the scale and shift of
      // dims 16 r + 4 q + e of its sample (SPLIT: row block r by wave r)
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        if (r0 + r >= fs.R || (SPLIT && wave != r)) continue;
        if constexpr (SPLIT) {
          auto part = [&](int w) { return rn_ld4(red + ((w * NB + r) * 64 + lane) * 4); };
          os[r][0] = (part(0) + part(2)) + (part(4) + part(6));
          ot[r][0] = (part(1) + part(3)) + (part(5) + part(7));
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
              ls[m] += s;
            }
      }
      sync();
    }
#pragma unroll
    for (int m = 0; m < MB; ++m) ldacc[m] += ls[m];
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
  if (a.x_out) {
    for (int o = t; o < S * d; o += NT) {
      const int m = o / d, j = o - m * d;
      if (m0 + m >= a.n) continue;
      float v = xs[m * ldx + j];
      if (a.dir != 0 && (a.flags & RN_STD)) v = v * sqrtf(dcov[(int64_t)j * d + j]) + dmean[j];
      a.x_out[m0 * d + o] = v;
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
// layers, hidden 256 | d = 64, 10 layers, hidden 128 | d = 5, 4 layers, hidden
// 64 | d = 32, 4 layers, hidden 32):
//   n         shared tile (8 waves)     16 samples a wave       32 samples a wave
//   1000        39 |   49 |  17 |  16    106 |  119 |  25 |  22   156 |  183 |  34 |  31
//   4000        41 |   51 |  17 |  16    107 |  119 |  25 |  22   157 |  183 |  34 |  31
//   10000       90 |  111 |  36 |  33    106 |  120 |  25 |  23   157 |  183 |  33 |  32
//   20000      140 |  173 |  55 |  50    140 |  165 |  30 |  27   157 |  184 |  33 |  32
//   50000      332 |  415 | 132 | 121    225 |  307 |  45 |  39   221 |  270 |  43 |  39
//   409600    2500 | 3108 | 981 | 906   1290 | 1686 | 231 | 195  1173 | 1696 | 193 | 166
// A shared tile spreads the serial hidden blocks of a layer over eight waves,
// which pays up to two workgroups a CU (512 tiles) and, with eight and more
// blocks to spread, until a wave for every 16 samples fills the chip's SIMDs;
// 32 samples a wave halve the weight reads once the grid is several waves a
// SIMD deep. Wide states, whose four tiles would not leave room for two
// workgroups a CU, share one.
static int rn_pass_variant(int64_t n, int d, int h) {
  const int64_t tiles = (n + 15) / 16, hb = rn_b16(h), split_to = hb < 8 ? 512 : hb < 13 ? 100 * hb : 1280;
  if (4 * rn_rup16(16 * (d + 1) * 4) > 64 * 1024 || tiles <= split_to) return 0;
  return tiles <= 2048 ? 1 : 2;
}

template <int NB>
static int rn_pass_nb(hipStream_t st, const RnvpDev& f, const RnPassArgs& a, int var) {
  switch (var) {
    case 0: return rn_launch_pass<NB, 1, true>(st, f, a);
    case 1: return rn_launch_pass<NB, 1, false>(st, f, a);
    default: return rn_launch_pass<NB, NB <= 2 ? 2 : 1, false>(st, f, a);  // (four blocks and 32 samples spill)
  }
}

// ------------------------------------------------------------ training ---
// The forward pass of a training step (which saves every layer's input) and
// the adjoint sweep. Both use workgroups of eight wavefronts on tiles of 16 MS
// samples; wave 2k + p takes MLP p and share k of its hidden features.
// The hidden layers of both, and of the outputs that carry the state from
// layer to layer, are summed in one order (RnOrder): a ReLU mask that rounds
// differently in two evaluations changes a weight gradient by a whole sample's
// share.

// One ordered block's weights (a lane's share). The first block's are requested
// ahead of the barrier before their use, the others one block ahead.
template <int NB>
struct RnOrdW {
  f32x4_t w1[NB], w2, b;
  __device__ __forceinline__ void load(const RnFr& f, int blk, int r, int lane) {
    const int kc = f.KC > 0 ? f.KC : 1;
#pragma unroll
    for (int k = 0; k < NB; ++k) w1[k] = rn_ld4(f.W1s + ((int64_t)blk * kc + (k < kc ? k : kc - 1)) * 256 + 4 * lane);
    w2 = rn_ld4(f.W2s + ((int64_t)blk * f.R + r) * 256 + 4 * lane);
    b = rn_ld4(f.b1s + 16 * blk + 4 * (lane >> 4));
  }
};

// What share k (of four) of an MLP's waves does in a round: row block r of
// the round's 4 / Gw, chain groups gcol, gcol + Gw, .. (Gc of them).
struct RnShare {
  int lgw, rsel, gcol, lgc;  // log2 Gw; log2 Gc
  __device__ RnShare(const RnOrder& od, int k) {
    lgw = od.G >= 4 ? 2 : od.G >> 1;
    lgc = od.G >= 16 ? 2 : od.G >= 8 ? 1 : 0;  // G is a power of two <= 16
    rsel = k >> lgw;
    gcol = k & ((1 << lgw) - 1);
  }
  __device__ int rows() const { return 4 >> lgw; }  // row blocks of a round
  // first block of chain group gi (four groups pair up at twice their distance first: 0, 2, 1, 3)
  __device__ int group(const RnOrder& od, int gi) const {
    return (gcol + ((lgc == 2 ? ((gi & 1) << 1 | gi >> 1) : gi) << lgw)) * od.U;
  }
};

// Row block r of an MLP's output for the wave's share of the hidden features:
// out[m] = the pairwise sum of its chains. cF: the conditioning inputs as
// fragments, [KC][MS][64] float4 in LDS (rn_cond4 of every lane); nx: the
// weights of block group(od, 0).
template <int NB, int MS>
__device__ __forceinline__ void rn_ordered_out(const RnFr& f, const RnOrder& od, const RnShare& sh, int r,
                                               RnOrdW<NB>& nx, const float* cF, f32x4_t (&out)[MS], int lane) {
  const int groups = 1 << sh.lgc;
  f32x4_t part[MS], c[NB][MS];
#pragma unroll
  for (int k = 0; k < NB; ++k)
    if (k < f.KC) {
#pragma unroll
      for (int m = 0; m < MS; ++m) c[k][m] = rn_ld4(cF + ((k * MS + m) * 64 + lane) * 4);
    }
  for (int gi = 0; gi < groups; ++gi) {
    const int blk0 = sh.group(od, gi);
    f32x4_t acc[4][MS];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int m = 0; m < MS; ++m) acc[i][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int u = 0; u < od.U; ++u) {
      const RnOrdW<NB> w = nx;
      const int blk = blk0 + u;
      nx.load(f, u + 1 < od.U ? blk + 1 : gi + 1 < groups ? sh.group(od, gi + 1) : blk, r, lane);
      f32x4_t a[MS];
#pragma unroll
      for (int m = 0; m < MS; ++m) a[m] = w.b;
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (k < f.KC) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int m = 0; m < MS; ++m) a[m] = rn_mfma(w.w1[k][e], c[k][m][e], a[m]);
        }
      for (int k = NB; k < f.KC; ++k) {
        const f32x4_t x1 = rn_ld4(f.W1s + ((int64_t)blk * f.KC + k) * 256 + 4 * lane);
#pragma unroll
        for (int m = 0; m < MS; ++m) {
          const f32x4_t cv = rn_ld4(cF + ((k * MS + m) * 64 + lane) * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) a[m] = rn_mfma(x1[e], cv[e], a[m]);
        }
      }
#pragma unroll
      for (int m = 0; m < MS; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) a[m][e] = rn_relu(a[m][e]);
      if (od.Sg == 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int m = 0; m < MS; ++m) acc[i][m] = rn_mfma(w.w2[i], a[m][i], acc[i][m]);
      } else if (od.Sg == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int m = 0; m < MS; ++m) acc[i & 1][m] = rn_mfma(w.w2[i], a[m][i], acc[i & 1][m]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int m = 0; m < MS; ++m) acc[0][m] = rn_mfma(w.w2[i], a[m][i], acc[0][m]);
      }
    }
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      // the accumulators of absent chains are zero: v + 0 = v
      const f32x4_t v = (acc[0][m] + acc[1][m]) + (acc[2][m] + acc[3][m]);
      // group sums in the order 0, 1 | 2, 3: (0 + 1) + (2 + 3)
      if (gi == 0)
        out[m] = v;
      else if (gi == 1)
        out[m] = out[m] + v;
      else if (gi == 2)
        part[m] = v;
      else
        out[m] = out[m] + (part[m] + v);
    }
  }
}

// A wave's output for row block rd * rows() + rsel, 16 MS samples, into red.
template <int NB, int MS>
__device__ __forceinline__ void rn_round_out(const RnFr& f, const RnOrder& od, const RnShare& sh, int rd,
                                             RnOrdW<NB>& nx, const float* cF, float* red, int wave, int lane) {
  const int r = rd * sh.rows() + sh.rsel;
  if (r >= f.R) return;
  f32x4_t o[MS];
  if (rd > 0) nx.load(f, sh.group(od, 0), r, lane);
  rn_ordered_out<NB, MS>(f, od, sh, r, nx, cF, o, lane);
#pragma unroll
  for (int m = 0; m < MS; ++m) *reinterpret_cast<f32x4_t*>(red + ((wave * MS + m) * 64 + lane) * 4) = o[m];
}
// ... and the sum of the waves' outputs for row block rsel of the round and
// 16-sample group m (waves at distance 2 first)
template <int MS>
__device__ __forceinline__ f32x4_t rn_round_sum(const float* red, int p, int rsel, int lgw, int m, int lane) {
  auto at = [&](int g) { return rn_ld4(red + (((2 * ((rsel << lgw) + g) + p) * MS + m) * 64 + lane) * 4); };
  if (lgw == 2) return (at(0) + at(2)) + (at(1) + at(3));
  if (lgw == 1) return at(0) + at(1);
  return at(0);
}

// What the coupling of a row block needs from memory besides the outputs.
struct RnCpl {
  f32x4_t bs, bt;
  int tj[4];
  __device__ __forceinline__ void load(const RnFr& fs, const RnFr& ft, int r, int q) {
    const int k0 = 16 * r + 4 * q;
    bs = rn_ld4(fs.b2 + k0);
    bt = rn_ld4(ft.b2 + k0);
    const int4 ti = *reinterpret_cast<const int4*>(fs.trans + k0);
    tj[0] = ti.x, tj[1] = ti.y, tj[2] = ti.z, tj[3] = ti.w;
  }
};

template <int NB, int MS>
__global__ void __launch_bounds__(512) rnvp_train_pass_kernel(RnvpDev f, RnPassArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int S = 16 * MS, NT = 512;
  const int d = f.d, h = f.h, ldx = d + 1, t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), col = lane & 15, q = lane >> 4;
  float* xs = reinterpret_cast<float*>(smem);
  float* red = xs + rn_rup16(S * ldx * 4) / 4;  // [8][MS][64] float4
  float* ldp = red + 8 * MS * 256;              // [8][S] log-dets by wave
  float* cF = ldp + 8 * S;                      // [KC][MS][64] float4
  const int64_t m0 = (int64_t)blockIdx.x * S;
  const float* dmean = f.theta + rn_stats(d, h, f.L);
  const float* dcov = dmean + d;
  for (int o = t; o < S * d; o += NT) {
    const int m = o / d, j = o - m * d;
    float v = 0.f;
    if (m0 + m < a.n) {
      v = a.x_in[m0 * d + o];
      if (a.flags & RN_STD) v = (v - dmean[j]) / sqrtf(dcov[(int64_t)j * d + j]);
    }
    xs[m * ldx + j] = v;
  }
  for (int o = t; o < 8 * S; o += NT) ldp[o] = 0.f;
  __syncthreads();
  for (int l = 0; l < f.L; ++l) {
    if (a.saved) {
      for (int o = t; o < S * d; o += NT) {
        const int m = o / d, j = o - m * d;
        if (m0 + m < a.n) a.saved[((int64_t)l * a.n + m0) * d + o] = xs[m * ldx + j];
      }
    }
    const int32_t* lay = rn_lay(f, l);
    const int dc = lay[0], dtr = lay[1];
    const RnFr fs(f.packed, d, h, l, 0, dc, dtr), ft(f.packed, d, h, l, 1, dc, dtr);
    const RnOrder od(dtr, h);
    const RnShare sh(od, wave >> 1);
    const RnFr& fp = (wave & 1) ? ft : fs;
    const int rpr = sh.rows();
    RnOrdW<NB> nx;
    if (sh.rsel < fs.R) nx.load(fp, sh.group(od, 0), sh.rsel, lane);
    RnCpl cp;  // of the wave's first coupling task
    if (wave < rpr * MS && wave / MS < fs.R) cp.load(fs, ft, wave / MS, q);
    for (int u = wave; u < fs.KC * MS; u += 8)
      *reinterpret_cast<f32x4_t*>(cF + (u * 64 + lane) * 4) = rn_cond4(fs, xs + (16 * (u % MS) + col) * ldx, u / MS, q, dc);
    __syncthreads();
    for (int rd = 0; rd * rpr < fs.R; ++rd) {
      rn_round_out<NB, MS>(fp, od, sh, rd, nx, cF, red, wave, lane);
      __syncthreads();
      for (int k = wave; k < rpr * MS; k += 8) {
        const int rsel = k / MS, m = k - rsel * MS, r = rd * rpr + rsel;
        if (r >= fs.R) continue;
        const int k0 = 16 * r + 4 * q;
        if (rd > 0 || k >= 8) cp.load(fs, ft, r, q);
        const f32x4_t sv = rn_round_sum<MS>(red, 0, rsel, sh.lgw, m, lane), tv = rn_round_sum<MS>(red, 1, rsel, sh.lgw, m, lane);
        const f32x4_t bs = cp.bs, bt = cp.bt;
        const int (&tj)[4] = cp.tj;
        float ls = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (k0 + e < dtr) {
            float* xp = xs + (16 * m + col) * ldx + tj[e];
            const float s = tanhf(sv[e] + bs[e]) * f.dt;
            const float tt = (tv[e] + bt[e]) * f.dt;
            *xp = (*xp + tt) * expf(s);
            ls += s;
          }
        ls += __shfl_xor(ls, 16, 64);
        ls += __shfl_xor(ls, 32, 64);
        if (lane < 16) ldp[wave * S + 16 * m + col] += ls;
      }
      __syncthreads();
    }
  }
  for (int m = t; m < S; m += NT) {
    if (m0 + m >= a.n) continue;
    float ld = 0.f;
    for (int w = 0; w < 8; ++w) ld += ldp[w * S + m];
    if (a.flags & RN_BASE) {
      // log N(y; 0, I) (realNVP.py:211-213: the standard normal, not base_dist)
      float s2 = 0.f;
      for (int j = 0; j < d; ++j) s2 += xs[m * ldx + j] * xs[m * ldx + j];
      ld += -0.5f * s2 - 0.91893853320467274f * (float)d;
    }
    if (a.logdet) a.logdet[m0 + m] = ld;
  }
  if (a.gy_out || a.x_out) {
    for (int o = t; o < S * d; o += NT) {
      const int m = o / d, j = o - m * d;
      if (m0 + m >= a.n) continue;
      const float v = xs[m * ldx + j];
      if (a.gy_out) a.gy_out[m0 * d + o] = -a.g_logp[m0 + m] * v;
      if (a.x_out) a.x_out[m0 * d + o] = v;
    }
  }
}

// ------------------------------------------------------------- adjoint ---
// Layers l1-1 .. l0 of the forward direction for one tile: recompute s, t;
// the coupling's reverse sweep; per MLP the hidden gradient gH = W2^T g, its
// ReLU mask, the tile's weight gradients and W1^T gH into the conditioning
// dims. H and gH are formed in both orientations (features x samples for the
// next product, samples x features as the operands of the weight gradients,
// whose k runs over the samples): swapping the operands of the product costs
// one more pass of the matrix core where a transpose would go through LDS.
// Weight gradients of a tile go to memory in fragment order, per (layer,
// tile) and p: dW1 [hb][kg][64] float4 (element i of lane l: feature 16 hb +
// 4 (l / 16) + i, dim 16 kg + l % 16), dW2 [hb][r][64] (dim 16 r + 4 (l / 16)
// + i, feature 16 hb + l % 16), db1 [16 HB], db2 [16 R]. A workgroup takes the
// tiles b, b + grid, .. and adds their weight gradients up in its own row.
struct RnBwdArgs {
  int l0, l1;
  const float* x;  // [l1 - l0, n, d] layer inputs, from layer l0
  int64_t n;
  const float* g_logp;
  const float* gy;  // [n, d] dL/d(output of layer l1 - 1)
  float* gx;        // [n, d] dL/d(input of layer l0)
  float* part;      // [l1 - l0, workgroups, rn_part_row]
};

__host__ __device__ inline int64_t rn_part_mlp(int hb, int kc, int r) { return 256LL * hb * (kc + r) + 16 * hb + 16 * r; }
__host__ __device__ inline int64_t rn_part_row(int d, int h) {  // KC + R <= ceil(d / 16) + 1, R <= ceil(d / 16)
  return 2 * (256LL * rn_b16(h) * (rn_b16(d) + 1) + 16LL * rn_b16(h) + 16LL * rn_b16(d));
}

template <int NB>
struct RnBwdFrag {
  f32x4_t w1[NB], w2t[NB], w1t[NB], b;
  float bc;
  __device__ __forceinline__ void load(const RnFr& f, int hb, int k0, int lane) {
    const int kc = f.KC > 0 ? f.KC : 1, rc = f.R > 0 ? f.R : 1;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      w1[k] = rn_ld4(f.W1f + ((int64_t)hb * kc + (k < kc ? k : kc - 1)) * 256 + 4 * lane);
      w2t[k] = rn_ld4(f.W2t + ((int64_t)hb * rc + (k < rc ? k : rc - 1)) * 256 + 4 * lane);
      w1t[k] = rn_ld4(f.W1t + ((int64_t)hb * kc + (k0 + k < kc ? k0 + k : kc - 1)) * 256 + 4 * lane);
    }
    b = rn_ld4(f.b1 + 16 * hb + 4 * (lane >> 4));
    bc = f.b1[16 * hb + (lane & 15)];
  }
};

template <int NB, int MS>
__device__ __forceinline__ void rn_bwd_tile(const RnvpDev& f, const RnBwdArgs& a, int64_t m0, bool first,
                                            unsigned char* smem) {
  constexpr int S = 16 * MS, NT = 512;
  const int d = f.d, h = f.h, ldx = d + 1, t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), col = lane & 15, q = lane >> 4;
  const int p = wave & 1, share = wave >> 1;
  float* gb = reinterpret_cast<float*>(smem);  // [S][ldx] gradient of the state
  float* glp = gb + rn_rup16(S * ldx * 4) / 4;  // [S]
  float* red = glp + S;                         // [8][NB][MS][64] float4
  // fragments [block][MS][64] float4 of the conditioning inputs, then of the
  // gradients of the scale and of the shift outputs: F with the product's k
  // over the dims, T with k over the samples
  float* cF = red + 8 * NB * MS * 256;
  const f32x4_t zero{0.f, 0.f, 0.f, 0.f};
  // (every entry of the row is one lane's, tile after tile)
  auto keep4 = [&](float* p, f32x4_t v) {
    f32x4_a4_t* p4 = reinterpret_cast<f32x4_a4_t*>(p);
    if (!first) v += *p4;
    *p4 = v;
  };
  auto keep = [&](float* p, float v) { *p = first ? v : *p + v; };

  for (int o = t; o < S * d; o += NT) {
    const int m = o / d, j = o - m * d;
    gb[m * ldx + j] = m0 + m < a.n ? a.gy[m0 * d + o] : 0.f;
  }
  for (int m = t; m < S; m += NT) glp[m] = m0 + m < a.n ? a.g_logp[m0 + m] : 0.f;

  for (int l = a.l1 - 1; l >= a.l0; --l) {
    const float* x = a.x + (int64_t)(l - a.l0) * a.n * d;
    auto x_at = [&](int m, int j) {  // entry j of the tile's sample m (0 past the batch)
      const int64_t row = m0 + m < a.n ? m0 + m : a.n - 1;
      const float v = x[row * d + j];
      return m0 + m < a.n ? v : 0.f;
    };
    const int32_t* lay = rn_lay(f, l);
    const int dc = lay[0], dtr = lay[1];
    const RnFr fs(f.packed, d, h, l, 0, dc, dtr), ft(f.packed, d, h, l, 1, dc, dtr);
    const RnFr& fp = p ? ft : fs;
    const RnOrder od(dtr, h);
    const RnShare sh(od, share);
    const int rpr = sh.rows(), KC = fs.KC, R = fs.R, HB = fs.HB;
    float* cT = cF + KC * MS * 256;
    float* gF = cT + KC * MS * 256;       // [2][R]
    float* gT = gF + 2 * R * MS * 256;    // [2][R]
    for (int u = wave; u < 2 * KC * MS; u += 8) {
      const int v = u >> 1, k = v / MS, m = v - k * MS;
      f32x4_t o;
      int ci[4];
      if (u & 1) {
        ci[0] = ci[1] = ci[2] = ci[3] = fs.cond[16 * k + col];
      } else {
        const int4 c4 = *reinterpret_cast<const int4*>(fs.condf + 16 * k + 4 * q);
        ci[0] = c4.x, ci[1] = c4.y, ci[2] = c4.z, ci[3] = c4.w;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float xv = x_at(16 * m + ((u & 1) ? 4 * q + e : col), ci[e]);
        o[e] = 16 * k + ((u & 1) ? col : 4 * e + q) < dc ? xv : 0.f;
      }
      *reinterpret_cast<f32x4_t*>(((u & 1) ? cT : cF) + (v * 64 + lane) * 4) = o;
    }
    RnOrdW<NB> nx;
    if (sh.rsel < R) nx.load(fp, sh.group(od, 0), sh.rsel, lane);
    RnCpl cp;  // of the wave's first coupling task, with its samples' inputs
    float xv[4];
    auto cpl = [&](int r, int m) {
      cp.load(fs, ft, r, q);
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[e] = x_at(16 * m + col, cp.tj[e]);
    };
    if (wave < rpr * MS && wave / MS < R) cpl(wave / MS, wave % MS);
    __syncthreads();
    RnBwdFrag<NB> w, wn;
    // ---- scale / shift, then the coupling's reverse sweep: y = (x + t) e^s,
    // log-det += s:  g_x = g e^s, g_t = g e^s, g_s = g y + g_logp;
    // g_spre = g_s dt (1 - tanh^2), g_tpre = g_t dt
    for (int rd = 0; rd * rpr < R; ++rd) {
      rn_round_out<NB, MS>(fp, od, sh, rd, nx, cF, red, wave, lane);
      if (rd == 0 && share < HB) wn.load(fp, share, 0, lane);
      __syncthreads();
      for (int k = wave; k < rpr * MS; k += 8) {
        const int rsel = k / MS, m = k - rsel * MS, r = rd * rpr + rsel;
        if (r >= R) continue;
        const int k0 = 16 * r + 4 * q, ms = 16 * m + col;
        if (rd > 0 || k >= 8) cpl(r, m);
        const f32x4_t sv = rn_round_sum<MS>(red, 0, rsel, sh.lgw, m, lane), tv = rn_round_sum<MS>(red, 1, rsel, sh.lgw, m, lane);
        const f32x4_t bs = cp.bs, bt = cp.bt;
        const int (&tj)[4] = cp.tj;
        float* oF = gF + (r * MS + m) * 256;
        float* oT = gT + (r * MS + m) * 256;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float g1 = 0.f, g2 = 0.f;
          if (k0 + e < dtr) {
            const float tn = tanhf(sv[e] + bs[e]);
            const float s = tn * f.dt;
            const float tt = (tv[e] + bt[e]) * f.dt;
            const float es = expf(s);
            const float y = (xv[e] + tt) * es;
            const float g = gb[ms * ldx + tj[e]];
            const float ge = g * es;
            gb[ms * ldx + tj[e]] = ge;
            g1 = (g * y + glp[ms]) * f.dt * (1.f - tn * tn);
            g2 = ge * f.dt;
          }
          // dim 4q + e of sample col: k-step q of lane (col, e) / k-step col % 4
          // of lane (4q + e, col / 4)
          const int iF = (col + 16 * e) * 4 + q, iT = (4 * q + e + 16 * (col >> 2)) * 4 + (col & 3);
          oF[iF] = g1;
          oT[iT] = g1;
          oF[R * MS * 256 + iF] = g2;
          oT[R * MS * 256 + iT] = g2;
        }
      }
      __syncthreads();
    }
    // ---- per MLP (p) and hidden block (share, share + 4, ..)
    const float* gpF = gF + p * R * MS * 256;
    const float* gpT = gT + p * R * MS * 256;
    auto frag = [&](const float* v, int blk, int m) { return rn_ld4(v + ((blk * MS + m) * 64 + lane) * 4); };
    float* pp = a.part + ((int64_t)(l - a.l0) * gridDim.x + blockIdx.x) * rn_part_row(d, h) + p * rn_part_mlp(HB, KC, R);
    float* pw2 = pp + 256LL * HB * KC;
    float* pb1 = pw2 + 256LL * HB * R;
    for (int k0 = 0; k0 == 0 || k0 < KC || k0 < R; k0 += NB) {
      f32x4_t gc[NB][MS];
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int m = 0; m < MS; ++m) gc[k][m] = zero;
      if ((k0 > 0 || R == 0) && share < HB) wn.load(fp, share, k0, lane);
      for (int hb = share; hb < HB; hb += 4) {
        w = wn;
        wn.load(fp, hb + 4 < HB ? hb + 4 : hb, k0, lane);
        f32x4_t o1[NB], o2[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) o1[k] = o2[k] = zero;
        float sb = 0.f;
#pragma unroll
        for (int m = 0; m < MS; ++m) {
          f32x4_t H = w.b, Ht{w.bc, w.bc, w.bc, w.bc}, g = zero, gt = zero;
#pragma unroll
          for (int k = 0; k < NB; ++k)
            if (k < KC) {
              const f32x4_t cv = frag(cF, k, m);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                H = rn_mfma(w.w1[k][e], cv[e], H);
                Ht = rn_mfma(cv[e], w.w1[k][e], Ht);
              }
            }
          for (int k = NB; k < KC; ++k) {
            const f32x4_t cv = frag(cF, k, m), x1 = rn_ld4(fp.W1f + ((int64_t)hb * KC + k) * 256 + 4 * lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              H = rn_mfma(x1[e], cv[e], H);
              Ht = rn_mfma(cv[e], x1[e], Ht);
            }
          }
#pragma unroll
          for (int r = 0; r < NB; ++r)
            if (r < R) {
              const f32x4_t gv = frag(gpF, r, m);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                g = rn_mfma(w.w2t[r][e], gv[e], g);
                gt = rn_mfma(gv[e], w.w2t[r][e], gt);
              }
            }
          for (int r = NB; r < R; ++r) {
            const f32x4_t gv = frag(gpF, r, m), x2 = rn_ld4(fp.W2t + ((int64_t)hb * R + r) * 256 + 4 * lane);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              g = rn_mfma(x2[e], gv[e], g);
              gt = rn_mfma(gv[e], x2[e], gt);
            }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            g[e] = H[e] > 0.f ? g[e] : 0.f;
            gt[e] = Ht[e] > 0.f ? gt[e] : 0.f;
            Ht[e] = rn_relu(Ht[e]);
            sb += gt[e];
          }
          // (chains of 16 features / samples, then their sums: with one chain
          // through all of them the input gradients' error was up to 1.14 times
          // that of short chains, at hidden 1000)
#pragma unroll
          for (int k = 0; k < NB; ++k)
            if (k0 + k < KC) {
              const f32x4_t cv = frag(cT, k0 + k, m);
              f32x4_t t1 = zero, t2 = zero;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                t1 = rn_mfma(w.w1t[k][e], g[e], t1);
                t2 = rn_mfma(gt[e], cv[e], t2);
              }
              gc[k][m] += t1;
              o1[k] += t2;
            }
#pragma unroll
          for (int r = 0; r < NB; ++r)
            if (k0 + r < R) {
              const f32x4_t gv = frag(gpT, k0 + r, m);
              f32x4_t t = zero;
#pragma unroll
              for (int e = 0; e < 4; ++e) t = rn_mfma(gv[e], Ht[e], t);
              o2[r] += t;
            }
        }
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          if (k0 + k < KC) keep4(pp + ((int64_t)hb * KC + k0 + k) * 256 + 4 * lane, o1[k]);
          if (k0 + k < R) keep4(pw2 + ((int64_t)hb * R + k0 + k) * 256 + 4 * lane, o2[k]);
        }
        if (k0 == 0) {
          sb += __shfl_xor(sb, 16, 64);
          sb += __shfl_xor(sb, 32, 64);
          if (lane < 16) keep(pb1 + 16 * hb + lane, sb);
        }
      }
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (k0 + k < KC) {
#pragma unroll
          for (int m = 0; m < MS; ++m)
            *reinterpret_cast<f32x4_t*>(red + (((wave * NB + k) * MS + m) * 64 + lane) * 4) = gc[k][m];
        }
      __syncthreads();
      for (int u = wave; u < NB * MS; u += 8) {  // conditioning-input gradients: all shares of both MLPs
        const int k = u / MS, m = u - k * MS;
        if (k0 + k >= KC) continue;
        auto at = [&](int w8) { return rn_ld4(red + (((w8 * NB + k) * MS + m) * 64 + lane) * 4); };
        const f32x4_t v = ((at(0) + at(2)) + (at(4) + at(6))) + ((at(1) + at(3)) + (at(5) + at(7)));
        const int i0 = 16 * (k0 + k) + 4 * q;
        const int4 ci = *reinterpret_cast<const int4*>(fs.cond + i0);
        const int cj[4] = {ci.x, ci.y, ci.z, ci.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i0 + e < dc) gb[(16 * m + col) * ldx + cj[e]] += v[e];
      }
      __syncthreads();
    }
    if (share == 0) {  // db2: sums over the samples
      for (int r = 0; r < R; ++r) {
        float s = 0.f;
        for (int m = 0; m < MS; ++m) {
          const f32x4_t gv = frag(gpT, r, m);
          s += (gv[0] + gv[1]) + (gv[2] + gv[3]);
        }
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (lane < 16) keep(pb1 + 16 * HB + 16 * r + lane, s);
      }
    }
    __syncthreads();  // the fragments are rewritten by the next layer
  }
  for (int o = t; o < S * d; o += NT) {
    const int m = o / d, j = o - m * d;
    if (m0 + m < a.n) a.gx[m0 * d + o] = gb[m * ldx + j];
  }
}

// MORE: more tiles than workgroups (a kernel of its own: what the loop keeps
// over the tiles takes 92 bytes of scratch a lane instead of 32 at one block and
// three groups)
template <int NB, int MS, bool MORE>
__global__ void __launch_bounds__(512) rnvp_bwd_kernel(RnvpDev f, RnBwdArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int S = 16 * MS;
  if constexpr (MORE) {
    // (a tile starts where every thread has read what it overwrites: its own
    // entries of the state gradient, the rest before the last barrier)
    for (int64_t tile = blockIdx.x; tile * S < a.n; tile += gridDim.x)
      rn_bwd_tile<NB, MS>(f, a, tile * S, tile == blockIdx.x, smem);
  } else {
    rn_bwd_tile<NB, MS>(f, a, (int64_t)blockIdx.x * S, true, smem);
  }
}

// Sum of the rows of weight gradients, scattered to the reference-shaped
// leaves of the gradient vector: a workgroup takes 64 float4 of one layer,
// wave w the rows w, w + 4, .. in four sums that take turns; the sixteen meet
// in LDS pairwise (four sums over a quarter of all tiles each had twice the
// error at 60,000 samples and 4.5 times at 400,000). Bound by reading the
// rows (a wave reads 1 KB of one row at a time).
__global__ void __launch_bounds__(256) rnvp_wgrad_kernel(RnvpDev f, int l0, const float* __restrict__ part, int rows,
                                                         float* __restrict__ grad) {
  __shared__ f32x4_t sh[4][64];
  const int d = f.d, h = f.h, l = l0 + blockIdx.y;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int32_t* lay = rn_lay(f, l);
  const int dc = lay[0], dtr = lay[1], KC = rn_b16(dc), R = rn_b16(dtr), HB = rn_b16(h);
  const int64_t pm = rn_part_mlp(HB, KC, R), row = rn_part_row(d, h);
  const int64_t e4 = (int64_t)blockIdx.x * 64 + lane;
  const bool in = 4 * e4 < 2 * pm;
  f32x4_t v{0.f, 0.f, 0.f, 0.f};
  if (in) {
    const float* src = part + (int64_t)blockIdx.y * rows * row + 4 * e4;
    auto at = [&](int t) -> f32x4_t { return *reinterpret_cast<const f32x4_a4_t*>(src + (int64_t)t * row); };
    f32x4_t u[4] = {v, v, v, v};
    int t = w;
    for (; t + 12 < rows; t += 16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) u[k] += at(t + 4 * k);
    }
    for (int k = 0; t < rows; t += 4, ++k) {
      const f32x4_t x = at(t);
      if (k == 0) u[0] += x;
      else if (k == 1) u[1] += x;
      else u[2] += x;
    }
    v = (u[0] + u[1]) + (u[2] + u[3]);
  }
  sh[w][lane] = v;
  __syncthreads();
  if (w != 0 || !in) return;
  v = (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]);
  const int p = 4 * e4 >= pm;
  const int64_t r = 4 * e4 - p * pm, n1 = 256LL * HB * KC, n2 = n1 + 256LL * HB * R, n3 = n2 + 16 * HB;
  float* W1 = grad + rn_mlp(d, h, l, p);
  float* b1 = W1 + (int64_t)h * d;
  float* W2 = b1 + h;
  float* b2 = W2 + (int64_t)d * h;
  const int32_t* cond = lay + 2;
  const int32_t* trans = lay + 2 + d;
  const int fl = (int)(r >> 2) & 63, c = fl & 15, q = fl >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (r < n1) {
      const int b = (int)(r >> 8), hb = b / KC, j = 16 * hb + 4 * q + i, k = 16 * (b - hb * KC) + c;
      if (j < h && k < dc) W1[(int64_t)j * d + cond[k]] = v[i];
    } else if (r < n2) {
      const int b = (int)((r - n1) >> 8), hb = b / R, k = 16 * (b - hb * R) + 4 * q + i, j = 16 * hb + c;
      if (j < h && k < dtr) W2[(int64_t)trans[k] * h + j] = v[i];
    } else if (r < n3) {
      const int j = (int)(r - n2) + i;
      if (j < h) b1[j] = v[i];
    } else {
      const int k = (int)(r - n3) + i;
      if (k < dtr) b2[trans[k]] = v[i];
    }
  }
}

// ---------------------------------------------------------------- host ---
// blocks of 16 dims held in registers: a mask that halves the dims fits (up
// to 128 dims; past 256, two, for the adjoint's LDS)
static inline int rn_nb(int d) {
  const int nb = rn_b16((d + 1) / 2);
  return nb <= 1 ? 1 : (nb <= 2 || d > 256) ? 2 : 4;
}
static inline int64_t rn_bwd_lds(int d, int nb, int ms) {
  // fragments: 2 KC + 4 R blocks of 1 KB, KC + R <= ceil(d / 16) + 1
  return (int64_t)rn_rup16(16 * ms * (d + 1) * 4) + 64 * ms + 8192LL * nb * ms + 1024LL * ms * (4 * rn_b16(d) + 2);
}
static int check_rnvp(const fmc_rnvp* r, RnvpDev& f, bool need_packed) {
  FMC_ARG(r != nullptr, "RealNVP description is NULL");
  FMC_ARG(r->n_dim >= 1 && r->n_layers >= 1 && r->n_hidden >= 1, "n_dim, n_layers and n_hidden must be >= 1");
  FMC_ARG(r->theta != nullptr && r->layout != nullptr, "theta or layout is NULL");
  FMC_ARG(!need_packed || r->packed != nullptr, "packed buffer is NULL");
  // the sizes taken: a bound from kernels that kept hidden rows in LDS, kept so
  // that what is refused stays refused. It admits d <= 424 and hidden <= 1268,
  // and the tiles of these kernels (a 16-sample adjoint the largest) fit 160 KB
  // for all of them (checked below).
  const int64_t d4 = (r->n_dim + 3) & ~3, h4 = (r->n_hidden + 3) & ~3;
  const int64_t need = 2 * ((64LL * (r->n_dim + 1) + 15) & ~15LL) + 64 * (4 * d4 + 2 * h4) + 128;
  FMC_ARG(need <= 160 * 1024, "n_dim %d / n_hidden %d exceed the LDS budget of the RealNVP kernels", r->n_dim,
          r->n_hidden);
  FMC_ARG(rn_bwd_lds(r->n_dim, rn_nb(r->n_dim), 1) <= 160 * 1024, "n_dim %d exceeds the LDS of the RealNVP adjoint",
          r->n_dim);
  f = RnvpDev{r->n_dim, r->n_layers, r->n_hidden, r->dt, r->theta, r->packed, r->layout};
  return FMC_OK;
}

// 16-sample groups per workgroup of the training kernels: as many as leave one
// workgroup a CU, up to three (four spill; measured at d = 32, 8 layers,
// hidden 256, adjoint + forward, n = 10,000: one group 433 + 120 us, two 353 +
// 134, three 237 + 85; n = 4000: 141 + 54, 177 + 68, 220 + 82)
static int rn_ms(int64_t tiles16, int d) {
  const int nb = rn_nb(d), cap = nb <= 2 ? 3 : 1;
  int64_t ms = (tiles16 + 255) / 256;
  ms = ms < 1 ? 1 : ms > cap ? cap : ms;
  while (ms > 1 && rn_bwd_lds(d, nb, (int)ms) > 160 * 1024) --ms;
  return (int)ms;
}

// How a sweep over all layers is cut: rows of weight gradients (workgroups) and
// layers a launch. The rows hold what a tile leaves, two workgroups a CU at
// most (more tiles are added up in them: with a row a tile the workspace grew
// with the batch and the rows' sum had chains of hundreds of terms), and as
// many layers share a launch as keep the rows within 256 MB (10,000 samples
// at d = 32, 8 layers, hidden 256 take 168 MB; d = 128, 10 layers would 1.5 GB).
struct RnSweep {
  int ms, layers;
  int64_t rows;
  RnSweep(const RnvpDev& f, int64_t n) {
    const int64_t t16 = (n + 15) / 16;
    ms = rn_ms(t16, f.d);
    rows = (t16 + ms - 1) / ms;
    if (rows > 512) rows = 512;
    const int64_t fit = (64LL << 20) / (rows * rn_part_row(f.d, f.h));
    layers = fit < 1 ? 1 : fit > f.L ? f.L : (int)fit;
  }
};

template <int NB, int MS>
static int rn_launch_train(hipStream_t st, const RnvpDev& f, const RnPassArgs& a) {
  const size_t shm = (size_t)rn_rup16(16 * MS * (f.d + 1) * 4) + (8192 + 512 + 1024 * rn_b16(f.d)) * MS;
  if (const int rc = rn_set_lds(rnvp_train_pass_kernel<NB, MS>, shm)) return rc;
  const int64_t grid = (a.n + 16 * MS - 1) / (16 * MS);
  FMC_ARG(grid <= 0x7fffffffLL, "too many samples for one launch");
  hipLaunchKernelGGL((rnvp_train_pass_kernel<NB, MS>), dim3((unsigned)grid), dim3(512), shm, st, f, a);
  return check_launch("realnvp training pass");
}

template <int NB, int MS>
static int rn_launch_bwd(hipStream_t st, const RnvpDev& f, const RnBwdArgs& a, int64_t rows) {
  const size_t shm = (size_t)rn_bwd_lds(f.d, NB, MS);
  FMC_ARG(rows <= 0x7fffffffLL, "too many samples for one launch");
  const auto k = rows * (16 * MS) < a.n ? rnvp_bwd_kernel<NB, MS, true> : rnvp_bwd_kernel<NB, MS, false>;
  if (const int rc = rn_set_lds(k, shm)) return rc;
  hipLaunchKernelGGL(k, dim3((unsigned)rows), dim3(512), shm, st, f, a);
  return check_launch("realnvp adjoint");
}

// ms: 16-sample groups a tile; rows: workgroups, at most the tiles
static int rn_bwd(hipStream_t st, const RnvpDev& f, const RnBwdArgs& a, int ms, int64_t rows) {
  switch (4 * rn_nb(f.d) + ms) {
    case 5: return rn_launch_bwd<1, 1>(st, f, a, rows);
    case 6: return rn_launch_bwd<1, 2>(st, f, a, rows);
    case 7: return rn_launch_bwd<1, 3>(st, f, a, rows);
    case 9: return rn_launch_bwd<2, 1>(st, f, a, rows);
    case 10: return rn_launch_bwd<2, 2>(st, f, a, rows);
    case 11: return rn_launch_bwd<2, 3>(st, f, a, rows);
    default: return rn_launch_bwd<4, 1>(st, f, a, rows);
  }
}

static int rn_train_pass(hipStream_t st, const RnvpDev& f, const RnPassArgs& a) {
  switch (4 * rn_nb(f.d) + rn_ms((a.n + 15) / 16, f.d)) {
    case 5: return rn_launch_train<1, 1>(st, f, a);
    case 6: return rn_launch_train<1, 2>(st, f, a);
    case 7: return rn_launch_train<1, 3>(st, f, a);
    case 9: return rn_launch_train<2, 1>(st, f, a);
    case 10: return rn_launch_train<2, 2>(st, f, a);
    case 11: return rn_launch_train<2, 3>(st, f, a);
    default: return rn_launch_train<4, 1>(st, f, a);
  }
}

static int rn_wgrad(hipStream_t st, const RnvpDev& f, int l0, int nl, const float* part, int64_t rows, float* grad) {
  const unsigned gx = (unsigned)((rn_part_row(f.d, f.h) / 4 + 63) / 64);
  hipLaunchKernelGGL(rnvp_wgrad_kernel, dim3(gx, (unsigned)nl), dim3(256), 0, st, f, l0, part, (int)rows, grad);
  return check_launch("realnvp weight gradient");
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
  if (partial_per_tile) *partial_per_tile = rn_part_row(f.d, f.h);
  if (tile) *tile = 16;
  return FMC_OK;
}

extern "C" int fmc_rnvp_pack(void* stream, const fmc_rnvp* r) {
  RnvpDev f;
  int rc = check_rnvp(r, f, true);
  if (rc) return rc;
  const unsigned gx = (unsigned)((rn_slot(f.d, f.h) / 4 + 255) / 256);
  hipLaunchKernelGGL(rnvp_pack_kernel, dim3(gx, 2 * f.L), dim3(256), 0, (hipStream_t)stream, f, r->packed);
  return check_launch("realnvp pack");
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
  if (saved || gy_out) return rn_train_pass(st, f, a);
  const int nb = rn_nb(f.d);
  const int var = rn_pass_variant(n, f.d, f.h);
  if (nb == 1) return rn_pass_nb<1>(st, f, a, var);
  if (nb == 2) return rn_pass_nb<2>(st, f, a, var);
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
  const int64_t tiles = (n + 15) / 16;
  FMC_ARG(n_partial_tiles >= tiles, "partials hold %lld tiles, %lld needed", (long long)n_partial_tiles,
          (long long)tiles);
  if (n == 0) return FMC_OK;
  // one row of partials for every 16 samples, whatever n: a caller may sum the rows of several calls
  return rn_bwd((hipStream_t)stream, f, RnBwdArgs{layer, layer + 1, x_in, n, g_logp, gy, gx, partials}, 1, tiles);
}

extern "C" int fmc_rnvp_weight_grad(void* stream, const fmc_rnvp* r, int32_t layer, float* partials,
                                    int64_t n_tiles, int64_t partial_rows, float* grad) {
  RnvpDev f;
  int rc = check_rnvp(r, f, false);
  if (rc) return rc;
  FMC_ARG(layer >= 0 && layer < f.L, "layer %d out of range", layer);
  FMC_ARG(partials && grad, "NULL pointer");
  FMC_ARG(n_tiles >= 1 && n_tiles <= 0x7fffffffLL, "n_tiles must be >= 1");
  const int64_t c = n_tiles < 256 ? (n_tiles + 15) / 16 : 16;  // (spare rows that the interface asks for)
  FMC_ARG(partial_rows >= n_tiles + c, "partials hold %lld rows, %lld needed (tiles + %lld more)",
          (long long)partial_rows, (long long)(n_tiles + c), (long long)c);
  return rn_wgrad((hipStream_t)stream, f, layer, 1, partials, n_tiles, grad);
}

extern "C" int fmc_rnvp_backward_ws_size(const fmc_rnvp* r, int64_t n, int64_t* floats) {
  RnvpDev f;
  int rc = check_rnvp(r, f, false);
  if (rc) return rc;
  FMC_ARG(n >= 1 && floats != nullptr, "n must be >= 1 and floats not NULL");
  const RnSweep sw(f, n);
  *floats = sw.layers * sw.rows * rn_part_row(f.d, f.h);
  return FMC_OK;
}

extern "C" int fmc_rnvp_backward(void* stream, const fmc_rnvp* r, const float* saved, int64_t n, const float* g_logp,
                                 const float* gy, float* gx, float* grad, float* workspace, int64_t workspace_floats) {
  RnvpDev f;
  int rc = check_rnvp(r, f, true);
  if (rc) return rc;
  FMC_ARG(n >= 1, "n must be >= 1");
  FMC_ARG(saved && g_logp && gy && gx && grad && workspace, "NULL pointer");
  FMC_ARG((uintptr_t)workspace % 16 == 0, "workspace must be 16-byte aligned");
  const RnSweep sw(f, n);
  const int64_t need = sw.layers * sw.rows * rn_part_row(f.d, f.h);
  FMC_ARG(workspace_floats >= need, "workspace holds %lld floats, need %lld (fmc_rnvp_backward_ws_size)",
          (long long)workspace_floats, (long long)need);
  hipStream_t st = (hipStream_t)stream;
  for (int l1 = f.L; l1 > 0; l1 -= sw.layers) {
    const int l0 = l1 > sw.layers ? l1 - sw.layers : 0;
    // (a tile reads its gradient rows before it writes them: gx in place)
    const RnBwdArgs a{l0, l1, saved + (int64_t)l0 * n * f.d, n, g_logp, l1 == f.L ? gy : gx, gx, workspace};
    if ((rc = rn_bwd(st, f, a, sw.ms, sw.rows))) return rc;
    if ((rc = rn_wgrad(st, f, l0, l1 - l0, workspace, sw.rows, grad))) return rc;
  }
  return FMC_OK;
}
