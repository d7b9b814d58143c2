// Prints what the U-Net's launch rules choose: for every line "N side ci co" on
// stdin the form of the LDS convolution (seven numbers, zeros: none), whether K
// is summed in slices, and the width of the weight gradient's boxes; with an
// argument, every form that is compiled.
#include <cstdio>

#include "unet_plan.h"

int main(int argc, char**) {
  using namespace hlbn;
  if (argc > 1) {
#define PRINT(NG, NT, MT, WM, BD, BH, BW) \
  std::printf("%d %d %d %d %d %d %d\n", NG, NT, MT, WM, BD, BH, BW);
    HLBN_BOX_FORMS(PRINT)
    return 0;
  }
  int N, side, ci, co;
  while (std::scanf("%d %d %d %d", &N, &side, &ci, &co) == 4) {
    const ConvGeom g{N, side, side, side};
    const BoxForm f = box_form(g, ci, co);
    std::printf("%d %d %d %d %d %d %d %d %d\n", f.ng, f.nt, f.mt, f.wm, f.bd, f.bh, f.bw,
                fwd_plan(g, ci, co).nsplit > 1, wgrad_box_width(g));
  }
}
