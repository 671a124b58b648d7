// Sums over the rows of a row-major matrix (a layer's bias gradient).
//
// Bound by reading the matrix once.  A workgroup takes 16 chunks of 16 bytes (128 columns of a 16-bit type) of a
// range of rows: 16 rows at a time, 256 contiguous bytes of each, eight loads per lane in flight.  There are few
// such column blocks (14336 columns: 112), so the rows are cut into parts until about four workgroups per CU exist;
// the parts' fp32 sums are added by a second launch, in a fixed order.
// 4096x14336 bf16: 203 us as a general reduction over tensor iterators, 25 us here (20 + 5).
#include "colsum.h"
#include "gemm_device.h"

namespace tb {

constexpr int CS_TX = 16, CS_TY = 16, CS_UNROLL = 8;

template <int DT>
__device__ __forceinline__ void cs_store(void* out, int64_t i, float v) {
  if constexpr (DT == DT_F32) ((float*)out)[i] = v;
  else if constexpr (DT == DT_F16) ((_Float16*)out)[i] = (_Float16)v;
  else ((__bf16*)out)[i] = (__bf16)v;
}

// VEC: columns a lane owns (one 16-byte load, or one element where rows do not start on 16 bytes)
template <int DT, int VEC>
__global__ void __launch_bounds__(CS_TX * CS_TY) column_sum_kernel(const ColumnSumParams p) {
  constexpr int ESZ = DT == DT_F32 ? 4 : 2;
  __shared__ float lds[CS_TY][CS_TX * VEC + 4];
  const int tx = threadIdx.x % CS_TX, ty = threadIdx.x / CS_TX;
  const int64_t c0 = (int64_t)blockIdx.x * (CS_TX * VEC);
  const int64_t col = c0 + tx * VEC;
  const int64_t per = (p.m + p.parts - 1) / p.parts;
  const int64_t r0 = (int64_t)blockIdx.y * per, r1 = r0 + per < p.m ? r0 + per : p.m;
  float acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
  if (col < p.n) {        // (n is a multiple of VEC)
    const uint8_t* src = p.x + col * ESZ;
    auto add = [&](const uint8_t* at) {
      if constexpr (VEC == 1) {
        acc[0] += load_as_f32(at, DT);
      } else {
        const v4i v = *(const v4i*)at;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          if constexpr (DT == DT_F32) acc[e] += __builtin_bit_cast(v4f, v)[e];
          else if constexpr (DT == DT_F16) acc[e] += (float)__builtin_bit_cast(h8, v)[e];
          else acc[e] += __builtin_bit_cast(float, (e & 1) ? ((uint32_t)v[e / 2] & 0xffff0000u) : ((uint32_t)v[e / 2] << 16));
        }
      }
    };
    const int64_t pitch = p.stride * ESZ;
    int64_t r = r0 + ty;
    for (; r + (CS_UNROLL - 1) * CS_TY < r1; r += CS_UNROLL * CS_TY)
#pragma unroll
      for (int u = 0; u < CS_UNROLL; ++u) add(src + (r + u * CS_TY) * pitch);
    for (; r < r1; r += CS_TY) add(src + r * pitch);
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) lds[ty][tx * VEC + e] = acc[e];
  __syncthreads();
  for (int c = threadIdx.x; c < CS_TX * VEC && c0 + c < p.n; c += CS_TX * CS_TY) {
    float s = 0.f;
#pragma unroll
    for (int y = 0; y < CS_TY; ++y) s += lds[y][c];
    if (p.parts == 1) cs_store<DT>(p.out, c0 + c, s);
    else p.partial[(int64_t)blockIdx.y * p.n + c0 + c] = s;
  }
}

template <int DT>
__global__ void __launch_bounds__(256) column_sum_parts_kernel(const ColumnSumParams p) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= p.n) return;
  float s = 0.f;
#pragma unroll 8
  for (int i = 0; i < p.parts; ++i) s += p.partial[(int64_t)i * p.n + c];
  cs_store<DT>(p.out, c, s);
}

int column_sum_parts(int64_t m, int64_t n, int n_cu) {
  // (at least 128 rows, one round of the unrolled loop, per part)
  const int64_t blocks = (n + 127) / 128, want = (4 * (int64_t)n_cu + blocks - 1) / blocks, most = (m + 127) / 128;
  const int64_t parts = want < most ? want : most;
  return (int)(parts < 1 ? 1 : (parts > 64 ? 64 : parts));
}

template <int DT>
hipError_t launch_typed(const ColumnSumParams& p, hipStream_t stream) {
  constexpr int ESZ = DT == DT_F32 ? 4 : 2, VEC = 16 / ESZ;
  const bool vec = p.n % VEC == 0 && (p.stride * ESZ) % 16 == 0 && ((uintptr_t)p.x & 15) == 0;
  const int64_t cols = CS_TX * (vec ? VEC : 1), blocks = (p.n + cols - 1) / cols;
  const dim3 grid((unsigned)blocks, (unsigned)p.parts);
  if (vec) hipLaunchKernelGGL((column_sum_kernel<DT, VEC>), grid, dim3(CS_TX * CS_TY), 0, stream, p);
  else hipLaunchKernelGGL((column_sum_kernel<DT, 1>), grid, dim3(CS_TX * CS_TY), 0, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.parts == 1) return e;
  hipLaunchKernelGGL((column_sum_parts_kernel<DT>), dim3((unsigned)((p.n + 255) / 256)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_column_sum(const ColumnSumParams& p, int x_type, hipStream_t stream) {
  // (a launch takes less than 2^32 threads, and a workgroup of 256 may have as few as 16 columns)
  constexpr int64_t MOST = 1ll << 27;
  const int64_t esz = x_type == DT_F32 ? 4 : 2;
  for (int64_t c = 0; c < p.n; c += MOST) {
    ColumnSumParams part = p;
    part.x += c * esz;
    part.out = (uint8_t*)p.out + c * esz;
    part.n = p.n - c < MOST ? p.n - c : MOST;
    const hipError_t e = x_type == DT_F32 ? launch_typed<DT_F32>(part, stream)
                         : x_type == DT_F16 ? launch_typed<DT_F16>(part, stream) : launch_typed<DT_BF16>(part, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace tb
