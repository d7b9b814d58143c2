// Which kernel and which form of it a convolution of the U-Net takes: rules on
// the level's size and the channel counts, without device code.
#pragma once

#include <algorithm>
#include <cstdint>

#include "unet_internal.h"

namespace hlbn {

inline int64_t positions(const ConvGeom& g) { return (int64_t)g.N * g.D * g.H * g.W; }

// Launch plan of k_conv_fwd: NT output-channel tiles per wave (an A fragment
// feeds NT MFMAs), MT position tiles (a B fragment feeds MT) and the number of
// K slices.  Fine levels keep MT = 4 or 2; coarse levels, with few positions,
// first take fewer position tiles per wave and then split K so that the grid
// has about four waves per SIMD and each wave a short chain of K steps.
struct FwdPlan {
  int mt, nt, nsplit, hpw;
  int64_t waves;
};
inline FwdPlan fwd_plan(const ConvGeom& cg, int ci, int co) {
  const int64_t P = positions(cg);
  const int tiles = co / 16;
  FwdPlan f;
  f.nt = tiles >= 8 ? 8 : (tiles >= 3 ? 4 : tiles);
  f.mt = f.nt >= 8 ? 2 : 4;
  const int ngroups = (tiles + f.nt - 1) / f.nt;
  constexpr int64_t kTarget = 4096;
  while (f.mt > 1 && ((P + 16 * f.mt - 1) / (16 * f.mt)) * ngroups < kTarget) f.mt /= 2;
  f.waves = ((P + 16 * f.mt - 1) / (16 * f.mt)) * ngroups;
  const int nhalf = 27 * (ci / 16);
  const int ksteps = (nhalf + 1) / 2;
  int ns = (int)std::min<int64_t>(ksteps, (kTarget + f.waves - 1) / f.waves);
  int kps = (ksteps + ns - 1) / ns;  // K steps per slice
  f.hpw = 2 * kps;
  f.nsplit = (nhalf + f.hpw - 1) / f.hpw;
  if (f.nsplit <= 1) {
    f.nsplit = 1;
    f.hpw = nhalf + 1;
  }
  return f;
}

// A form of k_conv_box: ng groups of 16 input channels, nt output-channel and
// mt position tiles per wave, wm waves along the positions (4 / wm along the
// channels), a box of bd x bh x bw positions.  ng 0: none.
struct BoxForm {
  int ng, nt, mt, wm, bd, bh, bw;
  bool operator==(const BoxForm& o) const {
    return ng == o.ng && nt == o.nt && mt == o.mt && wm == o.wm && bd == o.bd && bh == o.bh &&
           bw == o.bw;
  }
};
// Every form that box_form returns, 16 wide (H = 4) and 8 wide (H = 8).
#define HLBN_BOX_FORMS_OF(X, H, BW)                                                       \
  X(1, 1, 1, 4, 1, H, BW) X(1, 2, 2, 4, 2, H, BW) X(1, 1, 2, 4, 2, H, BW)                  \
  X(1, 3, 4, 4, 4, H, BW) X(1, 2, 4, 4, 4, H, BW) X(1, 1, 8, 4, H, 8, BW)                  \
  X(2, 1, 1, 4, 1, H, BW) X(2, 2, 2, 4, 2, H, BW) X(2, 1, 2, 4, 2, H, BW)                  \
  X(2, 3, 4, 4, 4, H, BW) X(2, 2, 4, 4, 4, H, BW) X(2, 1, 4, 4, 4, H, BW)                  \
  X(3, 1, 1, 4, 1, H, BW) X(3, 1, 2, 4, 2, H, BW) X(3, 1, 4, 4, 4, H, BW)                  \
  X(4, 1, 2, 2, 2, H / 2, BW) X(4, 1, 4, 1, 2, H / 2, BW) X(4, 1, 2, 1, 1, H / 2, BW)      \
  X(6, 1, 2, 2, 2, H / 2, BW)                                                             \
  X(8, 1, 4, 1, 2, H / 2, BW) X(8, 1, 1, 2, 1, H / 2, BW)                                  \
  X(12, 1, 4, 1, 2, H / 2, BW)
#define HLBN_BOX_FORMS(X) HLBN_BOX_FORMS_OF(X, 4, 16) HLBN_BOX_FORMS_OF(X, 8, 8)

// The box for a level and channel counts.  Boxes are 16 wide where that pads
// the width no more than 8, and hold as many positions as still leave about
// two workgroups per CU: a large box re-reads less halo, a small one fills the
// chip (32 -> 32 channels at 2 x 32^3: 21 us in boxes of 64 positions and one
// output tile, 13 in boxes of 128 and two).  Many input channels bound the box
// by LDS instead; there half the box (12 groups) and twice (6) measured the
// same within 3 %.
inline BoxForm box_for(const ConvGeom& g, int ci, int co) {
  const bool wide = (g.W + 15) / 16 * 16 == (g.W + 7) / 8 * 8;
  const int w = wide ? 16 : 8, h = wide ? 4 : 8;
  const int64_t P = positions(g);
  const int T = co / 16;
  const bool large = P >= 512 * 256, medium = P >= 256 * 128;
  switch (ci / 16) {
    case 1:
      if (!medium) return {1, 1, 1, 4, 1, h, w};
      if (!large) return T % 2 == 0 ? BoxForm{1, 2, 2, 4, 2, h, w} : BoxForm{1, 1, 2, 4, 2, h, w};
      if (T % 3 == 0) return {1, 3, 4, 4, 4, h, w};
      if (T % 2 == 0) return {1, 2, 4, 4, 4, h, w};
      return {1, 1, 8, 4, h, 8, w};
    case 2:
      if (!medium) return {2, 1, 1, 4, 1, h, w};
      if (!large) return T % 2 == 0 ? BoxForm{2, 2, 2, 4, 2, h, w} : BoxForm{2, 1, 2, 4, 2, h, w};
      if (T % 3 == 0) return {2, 3, 4, 4, 4, h, w};
      if (T % 2 == 0) return {2, 2, 4, 4, 4, h, w};
      return {2, 1, 4, 4, 4, h, w};
    case 3:
      if (!medium) return {3, 1, 1, 4, 1, h, w};
      return large ? BoxForm{3, 1, 4, 4, 4, h, w} : BoxForm{3, 1, 2, 4, 2, h, w};
    case 4:
      if (T <= 2) return {4, 1, 2, 2, 2, h / 2, w};
      return P >= 64 * 256 ? BoxForm{4, 1, 4, 1, 2, h / 2, w} : BoxForm{4, 1, 2, 1, 1, h / 2, w};
    case 6:
      return {6, 1, 2, 2, 2, h / 2, w};
    case 8:
      return P >= 64 * 256 ? BoxForm{8, 1, 4, 1, 2, h / 2, w} : BoxForm{8, 1, 1, 2, 1, h / 2, w};
    case 12:
      return {12, 1, 4, 1, 2, h / 2, w};
  }
  return {0, 0, 0, 0, 0, 0, 0};
}

// The form that a convolution takes, or none: k_conv_fwd.  A box holds
// positions of one sample, so on levels of side 1 to 4 most of it is padding,
// while k_conv_fwd fills its tiles from several samples.  That costs nothing
// while the chip is not full, where a box wins by its shorter chain of loads.
// Timed over the default network at sides 8 to 56 with up to 3000 samples:
// * boxes more than half empty, up to 2e9 padded products: 104 convolutions
//   1.33 ms in boxes and 2.39 in k_conv_fwd, 4 of them up to 1.2 x slower;
// * more products: 50 convolutions 5.43 and 2.12 ms, up to 15 x slower (side
//   8, 1000 samples: 128 -> 128 at 1^3 219.8 and 34.4 us, 32 -> 64 at 2^3
//   63.3 and 19.4);
// * half empty: 34 convolutions 0.77 and 1.27 ms (16^3 x 300: 192 -> 64 at
//   4^3 77.4 and 115.9 us).
inline BoxForm box_form(const ConvGeom& g, int ci, int co) {
  const BoxForm f = box_for(g, ci, co);
  if (!f.ng) return f;
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b * b; };
  const int64_t padded = g.N * up(g.D, f.bd) * up(g.H, f.bh) * up(g.W, f.bw);
  const double products = (double)padded * up(co, 16 * f.nt * (4 / f.wm)) * 27 * ci;
  return padded <= 2 * positions(g) || products <= 2e9 ? f : BoxForm{0, 0, 0, 0, 0, 0, 0};
}

// Box width of the LDS-staged weight gradient for this level (0: the level
// does not tile into 4 x BH x BW boxes and takes the direct kernel).
inline int wgrad_box_width(const ConvGeom& g) {
  if (g.D % 4) return 0;
  if (g.W % 16 == 0 && g.H % 4 == 0) return 16;
  if (g.W % 8 == 0 && g.H % 8 == 0) return 8;
  return 0;
}

}  // namespace hlbn
