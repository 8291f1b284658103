// FP64 instantiations of the fused step in 64-cell row segments.
#include "fused_seg.h"

namespace pm {

int launch_yee_seg_f64(const KGrid& g, int ck, const FusedBufs& fb, int ty, int kchunk, int order,
                       hipStream_t s) {
  KFz z;
  if (!make_kfz(g, fb, (int)sizeof(double), &z)) return -1;
  if (ck == PM_COEFF_CB) return launch_seg_ck<double, PM_COEFF_CB>(g, z, ty, kchunk, order, s);
  if (ck == PM_COEFF_CACB)
    return launch_seg_ck<double, PM_COEFF_CACB>(g, z, ty, kchunk, order, s);
  return -1;
}

}  // namespace pm
