// With four arguments the VSG cell side.  Else reads "n S affine slot keys uncertainty listed border" lines and, for 256 CUs, prints the kernel that common_kernel (dice_dispatch.h) names for each
// (0 none, 1 lean, 2 translation, 3 crew) and the dynamic LDS bytes of the translation and crew launches.
#include <cstdio>
#include <cstdlib>

#include "../../dice_amd/csrc/dice_dispatch.h"

using dice_hip::reaches_border;
static_assert(reaches_border(21, 78, 17, 0, 100) == 0 && reaches_border(20, 50, 17, 0, 100) == 1 &&
                  reaches_border(50, 79, 17, 0, 100) == 2 && reaches_border(0, 99, 17, 0, 100) == 3,
              "a box from 4 to 95 of 100 pixels keeps them all");
static_assert(reaches_border(71, 128, 17, 50, 100) == 0 && reaches_border(21, 78, 17, 50, 100) == 1 &&
                  reaches_border(70, 71, 17, 50, 100) == 1 && reaches_border(128, 129, 17, 50, 100) == 2,
              "the same in an image that begins at 50");

int main(int argc, char **argv) {
  if (argc == 5) {  // the VSG cell side for radius, slack, area and number of subsets
    std::printf("%.17g\n", dice_hip::vsg_radius_cell(std::atof(argv[1]), std::atof(argv[2]), std::atof(argv[3]),
                                                     std::atoi(argv[4])));
    return 0;
  }
  int n, S, affine, slot, keys, unc, listed, border;
  while (std::scanf("%d %d %d %d %d %d %d %d", &n, &S, &affine, &slot, &keys, &unc, &listed, &border) == 8)
    std::printf("%d %zu %zu\n",
                (int)dice_hip::common_kernel(
                    {n, S, affine != 0, slot, keys != 0, unc != 0, listed != 0, border, 256}),
                sizeof(float) * dice_hip::trans_lds_floats(S, slot, false),
                sizeof(float) * dice_hip::trans_lds_floats(S, slot, true));
  return 0;
}
