// FP32 instantiations of the fused step in 64-cell row segments.
#include "fused_seg.h"

namespace pm {

int launch_yee_seg_f32(const KGrid& g, int ck, const FusedBufs& fb, int ty, int kchunk, int order,
                       hipStream_t s) {
  KFz z;
  if (!make_kfz(g, fb, (int)sizeof(float), &z)) return -1;
  if (ck == PM_COEFF_CB) return launch_seg_ck<float, PM_COEFF_CB>(g, z, ty, kchunk, order, s);
  if (ck == PM_COEFF_CACB) return launch_seg_ck<float, PM_COEFF_CACB>(g, z, ty, kchunk, order, s);
  if (ck == PM_COEFF_CB_F16)
    return launch_seg_ck<float, PM_COEFF_CB_F16>(g, z, ty, kchunk, order, s);
  return -1;
}

bool seg_supported(int ck, int ty) {
  return (ty == 3 || ty == 7) && (ck == PM_COEFF_CB || ck == PM_COEFF_CACB || ck == PM_COEFF_CB_F16);
}

}  // namespace pm
