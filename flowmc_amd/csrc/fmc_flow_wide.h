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
// workgroups a CU have to fit the LDS, and the ring's reads the packed buffer. More samples than the small-grid
// passes (whose eight wavefronts sum the log-dets in another order), and
// enough for its half as many workgroups to fill the chip: general / wide, us,
// n = 20000 | 33000 | 50000 | 100000:
//   d = 64, 10 layers, [256, 256]    302 / 271 | 499 / 482 | 712 / 539 | 1246 / 1014
//   d = 32,  8 layers, [128, 128]    120 / 119 | 196 / 184 | 261 / 220 |  452 /  381
//   d = 16,  4 layers, [64, 64]       42 /  48 |  70 /  72 |  96 /  88 |  165 /  150
//   d = 32,  4 layers, [256, 128, 64] 80 /  88 | 134 / 142 | 182 / 170 |  312 /  298
inline bool flow_wide(const FlowDims& dm, const PassArgs& a, int cus) {
  if (!dm.reg_spline() || dm.base_dense || dm.hmaxp() > 256 || a.saved || a.gy_out) return false;
  if (dm.pk_total() * 2 >= (1LL << 31) || WideSmem(dm).total > 80 * 1024) return false;
  if (dm.pk_read_end(WD_P) > dm.pk_total()) return false;  // (no layout so far: w3rt is at least as long as w3r's last steps)
  bool broad = true;
  for (int i = 0; i < dm.nh; ++i) broad = broad && dm.hp(i) > 128;
  return a.n > (broad ? 64 : 160) * (int64_t)cus;
}

void launch_flow_wide(hipStream_t st, const FlowDev& fd, const PassArgs& a);

}  // namespace fmc
