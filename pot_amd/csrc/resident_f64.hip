// Register-resident dense solve, double costs (the kernel is in resident.h).
#include "resident.h"

namespace potamd {
hipError_t resident_launch_f64(const ResidentTile& t, const ResidentArgs& a, int grid, size_t lds,
                               hipStream_t s, int* per_cu) {
  return a.logd ? on_tile<double, double, kResLog>(t, a, grid, lds, s, per_cu)
                : on_tile<double, double, kResScaling>(t, a, grid, lds, s, per_cu);
}
}  // namespace potamd
