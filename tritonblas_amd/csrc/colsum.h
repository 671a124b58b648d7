// Host-visible entry of the column-sum kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tb {

struct ColumnSumParams {
  const uint8_t* x;
  int64_t m, n, stride;   // elements; unit stride along n
  void* out;
  float* partial;         // (parts, n), unused when parts == 1
  int parts;              // row ranges summed by workgroups of their own
};

// row ranges an (m, n) sum is cut into
int column_sum_parts(int64_t m, int64_t n, int n_cu);
hipError_t launch_column_sum(const ColumnSumParams& p, int x_type, hipStream_t stream);

}  // namespace tb
