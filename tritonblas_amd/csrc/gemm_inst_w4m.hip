// The hand-scheduled 4-wave 256x256 kernels of bf16 and fp16 with M-contiguous operands (see gemm_w4.h).
#include "gemm_w4.h"

namespace tb {

template <int DT>
static const void* w4_kernel_of(int alay, int blay) {
  if (alay == LAY_K) return (const void*)&gemm_kernel_w4<W4Tile<DT, LAY_K, LAY_M>>;
  if (blay == LAY_K) return (const void*)&gemm_kernel_w4<W4Tile<DT, LAY_M, LAY_K>>;
  return (const void*)&gemm_kernel_w4<W4Tile<DT, LAY_M, LAY_M>>;
}

const void* w4_kernel_m(int dt, int alay, int blay) {
  return dt == DT_BF16 ? w4_kernel_of<DT_BF16>(alay, blay) : w4_kernel_of<DT_F16>(alay, blay);
}

}  // namespace tb
