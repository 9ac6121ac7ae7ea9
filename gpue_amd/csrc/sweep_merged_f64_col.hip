// merged col sweeps, double
#include "sweep_merged.h"
namespace gpue {
hipError_t merged_f64_col(int m, const SweepArgs* d, const MergeMap* map, int grid, int lds, hipStream_t s) {
  return launch_col_merged<double>(m, d, map, grid, lds, s);
}
int merged_f64_col_shape(int n, int* lds) { return merged_col_shape<double>(n, lds); }
}  // namespace gpue
