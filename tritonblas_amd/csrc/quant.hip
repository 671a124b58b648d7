// Fused blockwise Hadamard-32 rotation + MXFP4 quantisation (e2m1 codes, E8M0 scale per 32 values).
//
// HBM-bound: every input element is read once (16-byte loads, a wave covers 1 KiB of a row) and
// 4.25 bits per element are written; loads and stores are marked non-temporal (nothing is touched
// twice), which together with the division-free index arithmetic is worth 15 % on 8192x16384 bf16.  Four neighbouring lanes own one 32-value block (8 values
// each); the butterfly stages with stride 8 and 16 and the block maximum cross lanes with
// quad-permute DPP moves, so nothing goes through LDS.
//
// Bit-level definition of the quantiser (must stay integer-exact):
//   amax -> (bits + 0x200000) & 0xFF800000 -> e = exponent - 2, clamped to [-127, 127]
//   scale byte = (e + 127) & 0xFF ; q = x * 2^-e ; code = round-half-up-in-magnitude(q), saturated to 6.0
// The last step runs on v_cvt_scalef32_pk_fp4_f32 (two values per instruction); see the tie handling below.
// This file is compiled with -ffp-contract=off: the rotation is fp32 adds/subs and one multiply.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <type_traits>
#include "quant.h"

namespace tb {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float dpp_xor1(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_xor2(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));
}

template <int XT>
__device__ __forceinline__ void load8(const uint8_t* p, float (&v)[8]) {
  if constexpr (XT == QT_F32) {
    const v4f a = __builtin_nontemporal_load((const v4f*)p);
    const v4f b = __builtin_nontemporal_load((const v4f*)(p + 16));
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const v4i raw = __builtin_nontemporal_load((const v4i*)p);
    const uint32_t w[4] = {(uint32_t)raw.x, (uint32_t)raw.y, (uint32_t)raw.z, (uint32_t)raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (XT == QT_BF16) {
        v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
        v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
      } else {
        v[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] & 0xffffu));
        v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] >> 16));
      }
    }
  }
}

// MAGIC: the item count fits 31 bits and p.div_magic / p.div_shift divide by the items per row
template <int XT, bool HAD, int UNROLL, bool MAGIC>
__global__ __launch_bounds__(256) void quant_kernel(const QuantParams p) {
  const int64_t nc = p.n >> 3;  // 8-value items per row
  const int64_t items = p.m * nc;
  const int64_t base = ((int64_t)blockIdx.x * UNROLL) * 256 + threadIdx.x;
  const int sub = threadIdx.x & 3;
  constexpr int XB = (XT == QT_F32) ? 4 : 2;

  float v[UNROLL][8];
  int64_t row[UNROLL], col[UNROLL];
  bool ok[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    int64_t it = base + (int64_t)u * 256;
    ok[u] = it < items;
    if (!ok[u]) it = items - 1;  // keep the quad complete; nothing is stored for it
    if constexpr (MAGIC) {
      const uint32_t it32 = (uint32_t)it;
      const uint32_t q = p.div_shift < 0 ? it32 : (__umulhi(it32, p.div_magic) >> p.div_shift);
      row[u] = q;
      col[u] = it32 - q * (uint32_t)nc;
    } else {
      row[u] = it / nc;
      col[u] = it - row[u] * nc;
    }
    load8<XT>(p.x + (row[u] * p.x_stride + col[u] * 8) * XB, v[u]);
  }

#pragma unroll
  for (int u = 0; u < UNROLL; ++u) {
    float(&x)[8] = v[u];
    if constexpr (HAD) {
#pragma unroll
      for (int h = 1; h < 8; h <<= 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if ((i & h) == 0) {
            float a = x[i], b = x[i + h];
            x[i] = a + b;
            x[i + h] = a - b;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {  // stride 8: partner is lane ^ 1
        float o = dpp_xor1(x[i]);
        x[i] = (sub & 1) ? (o - x[i]) : (x[i] + o);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {  // stride 16: partner is lane ^ 2
        float o = dpp_xor2(x[i]);
        x[i] = (sub & 2) ? (o - x[i]) : (x[i] + o);
      }
      const float inv_sqrt32 = __builtin_bit_cast(float, 0x3E3504F3u);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = x[i] * inv_sqrt32;
    }
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[i]));
    amax = fmaxf(amax, dpp_xor1(amax));
    amax = fmaxf(amax, dpp_xor2(amax));

    uint32_t ab = (__builtin_bit_cast(uint32_t, amax) + 0x200000u) & 0xFF800000u;
    int field = (int)((ab >> 23) & 0xFFu);
    int e = field - 129;
    if (field == 0) e = -127;
    if (field == 255) e = 127;
    e = e < -127 ? -127 : (e > 127 ? 127 : e);
    // 2^-e as fp32 bits: normal for -e >= -126, the sub-normal 2^-127 for e = 127
    uint32_t qb = (e == 127) ? 0x00400000u : ((uint32_t)(127 - e) << 23);
    const float qs = __builtin_bit_cast(float, qb);
    // e2m1 conversion on the hardware converter.  It rounds to nearest-even; the quantiser's rule is
    // round-half-up in magnitude.  Setting the lowest fp32 mantissa bit moves every exact tie just
    // above the tie point and changes no other rounding decision (tie points have zero low bits).
    uint32_t packed = 0;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float q0 = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[i] * qs) | 1u);
      const float q1 = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[i + 1] * qs) | 1u);
      if (i == 0) packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, q0, q1, 1.0f, 0);
      if (i == 2) packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, q0, q1, 1.0f, 1);
      if (i == 4) packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, q0, q1, 1.0f, 2);
      if (i == 6) packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, q0, q1, 1.0f, 3);
    }
    if (ok[u]) {
      __builtin_nontemporal_store(packed, (uint32_t*)(p.codes + row[u] * p.codes_stride + col[u] * 4));
      if (sub == 0) p.scales[row[u] * p.scales_stride + (col[u] >> 2)] = (uint8_t)((e + 127) & 0xFF);
    }
  }
}

template <int XT, bool HAD>
static hipError_t launch_t(const QuantParams& p0, bool force_div64, hipStream_t stream) {
  constexpr int UNROLL = 4;
  QuantParams p = p0;
  const int64_t nc = p.n >> 3;
  const int64_t items = p.m * nc;
  const int64_t per_block = 256 * UNROLL;
  const int64_t grid = (items + per_block - 1) / per_block;
  // (force_div64: testing hook, takes the kernel for 2^31 items and more at any size)
  if (items < (1ll << 31) && !force_div64) {
    // floor(i / nc) for i < 2^31: with l = ceil(log2 nc) and magic = floor(2^(31+l) / nc) + 1 < 2^32,
    // (i * magic) >> (31 + l) is exact; the kernel takes the high product word and shifts by l - 1
    int l = 0;
    while ((1ll << l) < nc) ++l;
    if (l == 0) { p.div_magic = 0; p.div_shift = -1; }
    else { p.div_magic = (uint32_t)(((1ull << (31 + l)) / (uint64_t)nc) + 1); p.div_shift = l - 1; }
    hipLaunchKernelGGL((quant_kernel<XT, HAD, UNROLL, true>), dim3((unsigned)grid), dim3(256), 0, stream, p);
  } else {
    hipLaunchKernelGGL((quant_kernel<XT, HAD, UNROLL, false>), dim3((unsigned)grid), dim3(256), 0, stream, p);
  }
  return hipGetLastError();
}

hipError_t launch_quant(const QuantParams& p, int x_type, bool hadamard, bool force_div64, hipStream_t stream) {
  if (x_type == QT_BF16) return hadamard ? launch_t<QT_BF16, true>(p, force_div64, stream) : launch_t<QT_BF16, false>(p, force_div64, stream);
  if (x_type == QT_F16) return hadamard ? launch_t<QT_F16, true>(p, force_div64, stream) : launch_t<QT_F16, false>(p, force_div64, stream);
  return hadamard ? launch_t<QT_F32, true>(p, force_div64, stream) : launch_t<QT_F32, false>(p, force_div64, stream);
}

// ---- one 8-bit scale per row -----------------------------------------------------------------------
// amax of a row -> scale = max(amax, min_scale) * (1 / top) -> q = x * (1 / scale) in fp32 -> e4m3 / e5m2 / int8.
//
// Bound by HBM: the row is read once and stays in registers between the two uses, so a row costs its own bytes, the codes and
// one float.  Written as tensor operations (convert, abs, amax, clamp, two scalings, product, convert) the same values cost nine
// launches and five passes over fp32 copies of x: quantising 512x14336 bf16 and multiplying by a 4096x14336 e4m3 weight took
// 114 us as tensor operations + GEMM and takes 54 us with this kernel (49 us of it the GEMM).
// RT threads share a row: one while a chunk of eight values holds it, eight up to 64 values, a wave while 4096 values fit its
// registers, a workgroup of 256 up to 16384, 1024 threads beyond.  Few rows: more threads per row, so that the loads of a row are
// spread over the CU (launch_row_quant).  Short rows are bound by wavefronts, not by bytes: 2^24 rows of 8 bf16 take
// 81 us with a thread each, 4360 with a wave each and 1273 as tensor operations; 2^20 rows of 64 take 39, 286 and 640.
// Rows longer than 65536 values are read twice (LOOP), the second time mostly from the caches, or cut into parts, see below.
struct RowChunk16 { v4i a; };
struct RowChunk32 { v4i a, b; };

template <int XT> using row_chunk = typename std::conditional<XT == QT_F32, RowChunk32, RowChunk16>::type;

// eight values of a row, zero past its end.  VEC: rows start on 16 bytes and hold whole chunks.
template <int XT, bool VEC>
__device__ __forceinline__ row_chunk<XT> row_load(const uint8_t* row, int64_t c, int64_t n) {
  row_chunk<XT> r;
  if constexpr (XT == QT_F32) { r.a = v4i{0, 0, 0, 0}; r.b = v4i{0, 0, 0, 0}; } else { r.a = v4i{0, 0, 0, 0}; }
  const int64_t left = n - c * 8;
  if (left <= 0) return r;
  if constexpr (VEC) {
    if constexpr (XT == QT_F32) { r.a = *(const v4i*)(row + c * 32); r.b = *(const v4i*)(row + c * 32 + 16); }
    else r.a = *(const v4i*)(row + c * 16);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < left) {
        if constexpr (XT == QT_F32) {
          const int v = *(const int*)(row + (c * 8 + j) * 4);
          if (j < 4) r.a[j & 3] = v; else r.b[j & 3] = v;
        } else {
          r.a[j >> 1] |= (int)((uint32_t)*(const uint16_t*)(row + (c * 8 + j) * 2) << (16 * (j & 1)));
        }
      }
    }
  }
  return r;
}

template <int XT>
__device__ __forceinline__ void row_values(const row_chunk<XT>& r, float (&v)[8]) {
  if constexpr (XT == QT_F32) {
    const v4f a = __builtin_bit_cast(v4f, r.a), b = __builtin_bit_cast(v4f, r.b);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const uint32_t w[4] = {(uint32_t)r.a.x, (uint32_t)r.a.y, (uint32_t)r.a.z, (uint32_t)r.a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (XT == QT_BF16) {
        v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
        v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
      } else {
        v[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] & 0xffffu));
        v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] >> 16));
      }
    }
  }
}

// |x| as the integer its bits are: the order of the magnitudes, with NaN above everything (so that a NaN reaches the scale)
template <int XT>
__device__ __forceinline__ uint32_t row_amax(const row_chunk<XT>& r, uint32_t m) {
  float v[8];
  row_values<XT>(r, v);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v[j]) & 0x7fffffffu;
    m = b > m ? b : m;
  }
  return m;
}

// Whether every |x / scale| of a row is at most `top` but for one rounding: its largest magnitude and the scale's reciprocal are finite, and the scale is no
// denormal number, which would be off by more.  (m: the bits of the largest magnitude; NaN lies above infinity.)  Decided once for a row: with a look at every value
// the codes take 5 times the instructions of their products and conversions, which rows of few loads a thread do not hide.  bf16 to e4m3, us, every value and once a
// row: 512x14336 8.9 and 7.1, 4096x4096 14.2 and 12.1, 256x16384 6.1 and 4.6, 128x28672 5.7 and 4.5, 2048x1024 3.7 and 3.3, 8192x8192 37.5 and 36.3.
__device__ __forceinline__ bool row_fits(uint32_t m, float scale) { return m < 0x7f800000u && scale >= 1.17549435e-38f; }

// Eight codes of one chunk, lowest byte first.  FITS: see row_fits; the converters then round what they get and no value overflows.  Otherwise their own
// overflow rule is not relied on: the float formats take what lies half a step above
// the largest finite value to NaN (e4m3) or infinity (e5m2), as a conversion without saturation does.
template <int XT, int OT, bool FITS>
__device__ __forceinline__ uint64_t row_codes(const row_chunk<XT>& r, float inv) {
  float v[8];
  row_values<XT>(r, v);
  uint32_t w[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float q[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) q[j] = v[4 * h + j] * inv;
    if constexpr (OT == RQ_I8) {
      w[h] = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float t = __builtin_rintf(q[j]);
        if constexpr (!FITS) t = t != t ? 0.f : fminf(fmaxf(t, -127.f), 127.f);
        w[h] |= ((uint32_t)(int)t & 0xffu) << (8 * j);
      }
    } else if constexpr (FITS) {
      int p = 0;
      if constexpr (OT == RQ_E4M3) {
        p = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], p, false);
        p = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], p, true);
      } else {
        p = __builtin_amdgcn_cvt_pk_bf8_f32(q[0], q[1], p, false);
        p = __builtin_amdgcn_cvt_pk_bf8_f32(q[2], q[3], p, true);
      }
      w[h] = (uint32_t)p;
    } else {
      constexpr float over = OT == RQ_E4M3 ? 464.f : 61440.f;        // half a step above the largest finite value
      constexpr float lim = OT == RQ_E4M3 ? 448.f : 57344.f;
      constexpr uint32_t high = OT == RQ_E4M3 ? 0x7fu : 0x7cu;
      float s[4];
      bool any = false;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[j] = q[j] != q[j] ? 0.f : fminf(fmaxf(q[j], -lim), lim);
        any |= !(fabsf(q[j]) < over) || (OT == RQ_E4M3 && fabsf(q[j]) == over);
      }
      int p = 0;
      if constexpr (OT == RQ_E4M3) {
        p = __builtin_amdgcn_cvt_pk_fp8_f32(s[0], s[1], p, false);
        p = __builtin_amdgcn_cvt_pk_fp8_f32(s[2], s[3], p, true);
      } else {
        p = __builtin_amdgcn_cvt_pk_bf8_f32(s[0], s[1], p, false);
        p = __builtin_amdgcn_cvt_pk_bf8_f32(s[2], s[3], p, true);
      }
      w[h] = (uint32_t)p;
      if (any) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t sign = (__builtin_bit_cast(uint32_t, q[j]) >> 24) & 0x80u;
          const bool nan = q[j] != q[j];
          const bool big = OT == RQ_E4M3 ? fabsf(q[j]) > over : fabsf(q[j]) >= over;   // (464 is a tie: to even, 448)
          if (nan || big) w[h] = (w[h] & ~(0xffu << (8 * j))) | ((sign | (nan ? 0x7fu : high)) << (8 * j));
        }
      }
    }
  }
  return (uint64_t)w[0] | ((uint64_t)w[1] << 32);
}

// the largest m of the RT threads (a power of two) that share a row; `part`: one word per wave of the workgroup
template <int RT>
__device__ __forceinline__ uint32_t row_max(uint32_t m, uint32_t* part) {
#pragma unroll
  for (int d = (RT < 64 ? RT : 64) / 2; d > 0; d >>= 1) {
    const uint32_t o = (uint32_t)__shfl_xor((int)m, d);
    m = o > m ? o : m;
  }
  if constexpr (RT > 64) {
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < RT / 64; ++w) m = part[w] > m ? part[w] : m;
  }
  return m;
}

__device__ __forceinline__ float row_scale(const RowQuantParams& p, uint32_t m) {
  const float amax = __builtin_bit_cast(float, m);
  return (amax < p.min_scale ? p.min_scale : amax) * p.inv_top;     // (a NaN stays)
}

// codes of chunk c of a row to where they belong
template <int XT, int OT, bool VEC, bool FITS>
__device__ __forceinline__ void row_store(uint8_t* qr, int64_t c, int64_t n, const row_chunk<XT>& x, float inv) {
  const int64_t left = n - c * 8;
  if (left <= 0) return;
  const uint64_t w = row_codes<XT, OT, FITS>(x, inv);
  if constexpr (VEC) {
    *(uint64_t*)(qr + c * 8) = w;
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) if (j < left) qr[c * 8 + j] = (uint8_t)(w >> (8 * j));
  }
}

template <int XT, int OT, int RT, int CH, bool VEC, bool LOOP>
__global__ __launch_bounds__(RT < 256 ? 256 : RT) void row_quant_kernel(const RowQuantParams p) {
  constexpr int ROWS = RT < 256 ? 256 / RT : 1;
  constexpr int XB = XT == QT_F32 ? 4 : 2;
  __shared__ uint32_t part[RT > 64 ? RT / 64 : 1];
  const int t = threadIdx.x % RT;
  const int64_t stride = (int64_t)gridDim.x * ROWS;
  for (int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / RT; row < p.m; row += stride) {
    const uint8_t* xr = p.x + row * p.x_stride * XB;
    row_chunk<XT> r[CH];
    uint32_t m = 0;
    const int64_t chunks = LOOP ? (p.n + 7) >> 3 : 1;
    for (int64_t c0 = 0; c0 < chunks; c0 += (int64_t)RT * CH) {
#pragma unroll
      for (int i = 0; i < CH; ++i) r[i] = row_load<XT, VEC>(xr, c0 + i * RT + t, p.n);
#pragma unroll
      for (int i = 0; i < CH; ++i) m = row_amax<XT>(r[i], m);
    }
    m = row_max<RT>(m, part);
    const float scale = row_scale(p, m), inv = 1.0f / scale;
    if (t == 0) p.scale[row] = scale;
    auto codes = [&](auto fits) {
      for (int64_t c0 = 0; c0 < chunks; c0 += (int64_t)RT * CH) {
        if constexpr (LOOP) {
#pragma unroll
          for (int i = 0; i < CH; ++i) r[i] = row_load<XT, VEC>(xr, c0 + i * RT + t, p.n);
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) row_store<XT, OT, VEC, decltype(fits)::value>(p.q + row * p.n, c0 + i * RT + t, p.n, r[i], inv);
      }
    };
    if (__builtin_expect(row_fits(m, scale), 1)) codes(std::true_type{});
    else codes(std::false_type{});
    if constexpr (RT > 64) { if (row + stride < p.m) __syncthreads(); }      // (`part` is read before it is written again)
  }
}

// Few very long rows, in parts of 16384 values with a workgroup each and three launches: amax of the parts, scale of the row, codes
// of the parts.  The parts' amax wait where the row's first codes will be, which the third launch writes.  One workgroup for a row
// reads 40 GB/s: a row of 2^22 bf16 418 us, 21 in parts, 49 as tensor operations; of 2^24 1650, 21 and 99.
constexpr int ROW_PART_T = 256, ROW_PART_CH = 8;
constexpr int64_t ROW_PART_CHUNKS = ROW_PART_T * ROW_PART_CH;

template <int XT, bool VEC>
__global__ __launch_bounds__(ROW_PART_T) void row_part_amax_kernel(const RowQuantParams p, int parts) {
  constexpr int XB = XT == QT_F32 ? 4 : 2;
  __shared__ uint32_t lds[ROW_PART_T / 64];
  const int64_t row = blockIdx.x / (unsigned)parts, part = blockIdx.x % (unsigned)parts;
  const uint8_t* xr = p.x + row * p.x_stride * XB;
  row_chunk<XT> r[ROW_PART_CH];
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < ROW_PART_CH; ++i) r[i] = row_load<XT, VEC>(xr, part * ROW_PART_CHUNKS + i * ROW_PART_T + threadIdx.x, p.n);
#pragma unroll
  for (int i = 0; i < ROW_PART_CH; ++i) m = row_amax<XT>(r[i], m);
  m = row_max<ROW_PART_T>(m, lds);
  if (threadIdx.x == 0) __builtin_memcpy(p.q + row * p.n + part * 4, &m, 4);
}

__global__ __launch_bounds__(64) void row_part_scale_kernel(const RowQuantParams p, int parts) {
  const int64_t row = blockIdx.x;
  uint32_t m = 0;
  for (int i = threadIdx.x; i < parts; i += 64) {
    uint32_t v;
    __builtin_memcpy(&v, p.q + row * p.n + (int64_t)i * 4, 4);
    m = v > m ? v : m;
  }
  m = row_max<64>(m, nullptr);
  if (threadIdx.x == 0) p.scale[row] = row_scale(p, m);
}

template <int XT, int OT, bool VEC>
__global__ __launch_bounds__(ROW_PART_T) void row_part_codes_kernel(const RowQuantParams p, int parts) {
  constexpr int XB = XT == QT_F32 ? 4 : 2;
  const int64_t row = blockIdx.x / (unsigned)parts, part = blockIdx.x % (unsigned)parts;
  const uint8_t* xr = p.x + row * p.x_stride * XB;
  const float inv = 1.0f / p.scale[row];
  row_chunk<XT> r[ROW_PART_CH];
#pragma unroll
  for (int i = 0; i < ROW_PART_CH; ++i) r[i] = row_load<XT, VEC>(xr, part * ROW_PART_CHUNKS + i * ROW_PART_T + threadIdx.x, p.n);
#pragma unroll
  for (int i = 0; i < ROW_PART_CH; ++i)
    row_store<XT, OT, VEC, false>(p.q + row * p.n, part * ROW_PART_CHUNKS + i * ROW_PART_T + threadIdx.x, p.n, r[i], inv);
}

template <int XT>
static bool row_vec(const RowQuantParams& p) {
  constexpr int XB = XT == QT_F32 ? 4 : 2;
  return p.n % 8 == 0 && ((uintptr_t)p.x & 15) == 0 && (p.x_stride * XB) % 16 == 0 && ((uintptr_t)p.q & 7) == 0;
}

template <int XT, int OT, int RT, int CH, bool LOOP = false>
static hipError_t row_quant_t(const RowQuantParams& p, hipStream_t stream) {
  constexpr int ROWS = RT < 256 ? 256 / RT : 1, THREADS = RT < 256 ? 256 : RT;
  // (a launch takes less than 2^32 threads; a workgroup goes on to further rows)
  const int64_t blocks = (p.m + ROWS - 1) / ROWS, most = (1ll << 31) / THREADS;
  const dim3 grid((unsigned)(blocks < most ? blocks : most));
  if (row_vec<XT>(p)) hipLaunchKernelGGL((row_quant_kernel<XT, OT, RT, CH, true, LOOP>), grid, dim3(THREADS), 0, stream, p);
  else hipLaunchKernelGGL((row_quant_kernel<XT, OT, RT, CH, false, LOOP>), grid, dim3(THREADS), 0, stream, p);
  return hipGetLastError();
}

template <int XT, int OT>
static hipError_t row_quant_parts(const RowQuantParams& p, hipStream_t stream) {
  const int64_t parts = ((p.n + 7) / 8 + ROW_PART_CHUNKS - 1) / ROW_PART_CHUNKS;
  if (parts * p.m >= (1ll << 32) / ROW_PART_T) return hipErrorInvalidValue;      // (2^38 values)
  const dim3 grid((unsigned)(parts * p.m));
  const bool vec = row_vec<XT>(p);
  if (vec) hipLaunchKernelGGL((row_part_amax_kernel<XT, true>), grid, dim3(ROW_PART_T), 0, stream, p, (int)parts);
  else hipLaunchKernelGGL((row_part_amax_kernel<XT, false>), grid, dim3(ROW_PART_T), 0, stream, p, (int)parts);
  hipLaunchKernelGGL(row_part_scale_kernel, dim3((unsigned)p.m), dim3(64), 0, stream, p, (int)parts);
  if (vec) hipLaunchKernelGGL((row_part_codes_kernel<XT, OT, true>), grid, dim3(ROW_PART_T), 0, stream, p, (int)parts);
  else hipLaunchKernelGGL((row_part_codes_kernel<XT, OT, false>), grid, dim3(ROW_PART_T), 0, stream, p, (int)parts);
  return hipGetLastError();
}

template <int XT, int OT>
static hipError_t row_quant_o(const RowQuantParams& p, hipStream_t stream) {
  const int64_t chunks = (p.n + 7) / 8;
  if (chunks <= 1) return row_quant_t<XT, OT, 1, 1>(p, stream);
  if (chunks <= 8) return row_quant_t<XT, OT, 8, 1>(p, stream);
  // (a wave per row only where the rows alone fill the device: 256 CUs x 8 waves)
  if (chunks <= 64 * 2 && p.m >= 2048) return row_quant_t<XT, OT, 64, 2>(p, stream);
  if (chunks <= 64 * 8 && p.m >= 2048) return row_quant_t<XT, OT, 64, 8>(p, stream);
  if (chunks <= 256 * 2) return row_quant_t<XT, OT, 256, 2>(p, stream);
  if (chunks <= 256 * 8 && p.m >= 256) return row_quant_t<XT, OT, 256, 8>(p, stream);
  if (chunks <= 1024 * 4) return row_quant_t<XT, OT, 1024, 4>(p, stream);
  if (chunks <= 1024 * 8) return row_quant_t<XT, OT, 1024, 8>(p, stream);
  // (a row of up to 2^17 values takes one workgroup less time than two more launches; 256 rows keep every CU reading, and read the
  // second time from the caches: 512x131072 bf16 55 us, in parts 62)
  if (chunks <= 1 << 14 || p.m >= 256) return row_quant_t<XT, OT, 1024, 4, true>(p, stream);
  return row_quant_parts<XT, OT>(p, stream);
}

template <int XT>
static hipError_t row_quant_x(const RowQuantParams& p, int q_type, hipStream_t stream) {
  if (q_type == RQ_E4M3) return row_quant_o<XT, RQ_E4M3>(p, stream);
  if (q_type == RQ_E5M2) return row_quant_o<XT, RQ_E5M2>(p, stream);
  return row_quant_o<XT, RQ_I8>(p, stream);
}

hipError_t launch_row_quant(const RowQuantParams& p, int x_type, int q_type, hipStream_t stream) {
  if (x_type == QT_BF16) return row_quant_x<QT_BF16>(p, q_type, stream);
  if (x_type == QT_F16) return row_quant_x<QT_F16>(p, q_type, stream);
  return row_quant_x<QT_F32>(p, q_type, stream);
}

}  // namespace tb
