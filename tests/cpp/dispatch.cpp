// Reads "n S affine slot keys uncertainty listed" lines and, for 256 CUs, prints the kernel that common_kernel (dice_dispatch.h) names for each
// (0 none, 1 lean, 2 translation, 3 crew) and the dynamic LDS bytes of the translation and crew launches.
#include <cstdio>

#include "../../dice_amd/csrc/dice_dispatch.h"

int main() {
  int n, S, affine, slot, keys, unc, listed;
  while (std::scanf("%d %d %d %d %d %d %d", &n, &S, &affine, &slot, &keys, &unc, &listed) == 7)
    std::printf("%d %zu %zu\n",
                (int)dice_hip::common_kernel({n, S, affine != 0, slot, keys != 0, unc != 0, listed != 0, 256}),
                sizeof(float) * dice_hip::trans_lds_floats(S, slot, false),
                sizeof(float) * dice_hip::trans_lds_floats(S, slot, true));
  return 0;
}
