// The wide flow pass (fmc_flow_wide.hip): its LDS layout and what it takes.
#pragma once

#include "fmc_flow_common.h"

namespace fmc {

constexpr int WIDE_MT = 64;  // samples a workgroup
constexpr int WD_P = 4;      // k-steps of weight fragments in flight

struct WideSmem {
  int xs, ldw, h, b, total;  // byte offsets: tile, the wavefronts' partial log-dets, activations, a layer's biases
  int ldx, lh;
  __host__ __device__ explicit WideSmem(const FlowDims& dm) {
    ldx = dm.d | 1;
    lh = dm.hmaxp() + PBF16::PAD;
    xs = 0;
    ldw = rup(WIDE_MT * ldx * 4, 16);
    h = ldw + 4 * WIDE_MT * 4;
    b = h + WIDE_MT * lh * 2;
    const int b0 = (int)dm.pb_size(0), b1 = (int)dm.pb_size(1);
    total = b + 4 * (b0 > b1 ? b0 : b1);
  }
  // dims whose base log-density terms fit the activation region at once
  // (WIDE_MT + 1 rows of an odd stride)
  __host__ __device__ int base_cols(int d) const {
    const int c = WIDE_MT * lh * 2 / 4 / (WIDE_MT + 1) - 1;
    return d < c ? d : c;
  }
};

// Whether a pass goes the wide way. It takes a BF16 conditioner of up to 256
// units a layer (a wavefront holds a whole layer's share of a tile across the
// barrier), register splines, a diagonal base and no saved layer inputs; two
// workgroups a CU have to fit the LDS, and the ring's reads the packed buffer.
// More samples than the small-grid passes (whose eight wavefronts sum the
// log-dets in another order).
// The general pass has 96 samples a CU in flight (three workgroups of 32), the
// wide one 128 (two of 64), and either takes about the same time for its first
// sample as for a full chip: what decides is in how many rounds the chip takes
// the call. In as many rounds the wide pass gains where a layer keeps its four
// wavefronts busy and loses where each layer's barrier is most of it. wide /
// general, log-density, n on 256 CUs (general : wide rounds):
//                                       20000  26000  33000  41000  50000  66000  82000  100000
//                                       (1:1)  (2:1)  (2:2)  (2:2)  (3:2)  (3:3)  (4:3)  (5:4)
//   d = 100, 2 layers, [256, 256]        0.91   0.62   0.92   0.89   0.74   0.85   0.73   0.81
//   d = 64,  4 layers, [256, 256]        0.95   0.70   1.00   0.90   0.81   0.90   0.76   0.81
//   d = 8,   4 layers, [256]             1.15   0.76   1.12   1.01   0.92   1.03   0.93   0.96
//   d = 32,  8 layers, [128, 128]        1.01   0.68   1.00   0.92   0.83   0.93   0.85   0.87
//   d = 16,  4 layers, [64, 64]          1.12   0.75   1.06   0.99   0.93   1.01   0.91   0.93
//   d = 32,  4 layers, [256, 128, 64]    1.09   0.75   1.09   0.98   0.92   1.01   0.94   0.94
//   d = 5,   4 layers, [32, 32]          1.15   0.74   1.13   1.09   0.92   1.09   0.94   0.99
//   d = 33,  4 layers, [128,256,64,32]   1.24   0.85   1.34   1.21   1.06   1.26   1.11   1.13
inline bool flow_wide(const FlowDims& dm, const PassArgs& a, int cus) {
  if (!dm.reg_spline() || dm.base_dense || dm.hmaxp() > 256 || a.saved || a.gy_out) return false;
  if (dm.pk_total() * 2 >= (1LL << 31) || WideSmem(dm).total > 80 * 1024) return false;
  if (dm.pk_read_end(WD_P) > dm.pk_total()) return false;  // (no layout so far: w3rt is at least as long as w3r's last steps)
  if (a.n <= 64 * (int64_t)cus) return false;
  int narrowest = dm.hp(0);
  for (int i = 1; i < dm.nh; ++i) narrowest = dm.hp(i) < narrowest ? dm.hp(i) : narrowest;
  if (narrowest > 128 && dm.d >= 64) return true;
  if (narrowest > 64 && dm.d >= 16 && a.n > 160 * (int64_t)cus) return true;
  const int64_t rg = (a.n + 96 * (int64_t)cus - 1) / (96 * (int64_t)cus), rw = (a.n + 128 * (int64_t)cus - 1) / (128 * (int64_t)cus);
  // a round of the wide pass in tenths of the general pass's
  const int round = dm.hp(dm.nh - 1) > 32 ? 10 : dm.nh > 2 ? 16 : 13;
  return rw * round < rg * 10;
}

void launch_flow_wide(hipStream_t st, const FlowDev& fd, const PassArgs& a);

}  // namespace fmc
