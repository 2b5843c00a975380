// Register-resident stabilised solve (the kernel is in resident.h).
#include "resident.h"

namespace potamd {
hipError_t resident_launch_stab(int f32, const ResidentTile& t, const ResidentArgs& a, int grid,
                                size_t lds, hipStream_t s, int* per_cu) {
  return f32 ? on_tile<float, double, kResStab>(t, a, grid, lds, s, per_cu)
             : on_tile<double, double, kResStab>(t, a, grid, lds, s, per_cu);
}
}  // namespace potamd
