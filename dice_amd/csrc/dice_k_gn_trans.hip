// gn kernels of square subsets in the common case beside the lean one: the
// translation-only pass (one wave per subset) and the crews of four waves per
// subset (translation-only and six parameters).
#include "dice_device.h"

namespace dice_hip {

hipError_t launch_gn_trans(int storage, int interp, const Launch &L, const KParams &kp, const DImage &ref,
                           const DImage &def, const DSubsets &subs, double *fields, const PassArgs &pa,
                           hipStream_t stream) {
#define V(T, I) dev::launch_trans_variant<T, I>(L, kp, ref, def, subs, fields, pa, stream)
  if (storage == 0) return interp == 0 ? V(float, 0) : V(float, 2);
  return interp == 0 ? V(uint16_t, 0) : V(uint16_t, 2);
#undef V
}

hipError_t launch_gn_crew(int storage, int interp, int trans, const Launch &L, const KParams &kp, const DImage &ref,
                          const DImage &def, const DSubsets &subs, double *fields, const PassArgs &pa,
                          hipStream_t stream) {
#define V(T, I, X) dev::launch_crew_variant<T, I, X>(L, kp, ref, def, subs, fields, pa, stream)
  if (trans) {
    if (storage == 0) return interp == 0 ? V(float, 0, true) : V(float, 2, true);
    return interp == 0 ? V(uint16_t, 0, true) : V(uint16_t, 2, true);
  }
  if (storage == 0) return interp == 0 ? V(float, 0, false) : V(float, 2, false);
  return interp == 0 ? V(uint16_t, 0, false) : V(uint16_t, 2, false);
#undef V
}

}  // namespace dice_hip
