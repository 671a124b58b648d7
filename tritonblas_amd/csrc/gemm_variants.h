// Host-visible registry of the built GEMM kernel variants.
#pragma once
#include <stdint.h>
#include "gemm_device.h"

namespace tb {

struct Variant {
  int dt, bm, bn, bk;     // element type and tile in elements
  int alay, blay;         // operand loaders (LAY_K / LAY_M)
  int wm, wn, threads, lds_bytes, minb;
  int fast, stages;       // fast: LOAD_*; the tile selector chooses among the LOAD_DIRECT ones
  const void* kernel;     // __global__ void (*)(const GemmParams), whole-tile schedules
  const void* kernel_one; // one tile to a workgroup (null: this variant has none)
  const void* kernel_sk;  // same tile with the Stream-K tail (null: this variant has none)
  int k_step_pairs;       // 1: hand-scheduled 4-wave kernel -- K must hold four K steps at least (MXFP4, M-contiguous operands, results whose rows are off
                          // 16 bytes: be an even number of them); with a
                          // Stream-K tail a multiple of four (the K ranges of its pieces are cut at multiples of four steps)
};

template <class T>
constexpr Variant make_variant() {
  return Variant{T::DT, T::BM, T::BN, T::BK, T::ALAY, T::BLAY, T::WM, T::WN, T::THREADS, T::LDS_ALLOC, T::MINB,
                 T::LOADER, T::STAGES, (const void*)&gemm_kernel<T, false>, (const void*)&gemm_tile_kernel<T, OneTile<T>::WHOLE_STEP>, (const void*)&gemm_kernel<T, true>, 0};
}

// The hand-scheduled 4-wave kernels of gemm_w4.h (256x256 tile, 128-byte K steps) are compiled in a
// translation unit of their own (gemm_inst_w4.hip), which hands out their addresses.
// (the ones with an M-contiguous operand in gemm_inst_w4m.hip)
const void* w4_kernel(int dt);
const void* w4_kernel_m(int dt, int alay, int blay);
const void* w4_kernel_sk(int dt);
template <int DT, int ALAY = LAY_K, int BLAY = LAY_K>
using W4Tile = Tile<DT, 256, 256, 128, 2, 2, ALAY, BLAY, 1, LOAD_DIRECT, 2>;
// LDS of these kernels: two 64 KB stages, 16 KB of FP4 scale buffers, 1 KB per wave of epilogue scales,
// the schedule's broadcast word
constexpr int W4_EPS_OFFSET = 131072 + 16384;
constexpr int W4_LDS_BYTES = W4_EPS_OFFSET + 4096 + 16;
template <class T>
Variant make_variant_w4() {
  return Variant{T::DT, T::BM, T::BN, T::BK, T::ALAY, T::BLAY, T::WM, T::WN, T::THREADS, W4_LDS_BYTES, 1,
                 1, T::STAGES, T::ALAY == LAY_M || T::BLAY == LAY_M ? w4_kernel_m(T::DT, T::ALAY, T::BLAY) : w4_kernel(T::DT), nullptr,
                 T::ALAY == LAY_M || T::BLAY == LAY_M ? nullptr : w4_kernel_sk(T::DT), 1};
}

// the grouped kernel of a tile, one tile to a workgroup (null: the tile has none; gemm_inst_fp8.hip)
const void* group_kernel(const Variant& v);

// defined one per translation unit
extern const Variant g_variants_f16[];
extern const int g_num_variants_f16;
extern const Variant g_variants_bf16[];
extern const int g_num_variants_bf16;
extern const Variant g_variants_fp8[];
extern const int g_num_variants_fp8;
extern const Variant g_variants_e5m2[];
extern const int g_num_variants_e5m2;
extern const Variant g_variants_e4e5[];
extern const int g_num_variants_e4e5;
extern const Variant g_variants_e5e4[];
extern const int g_num_variants_e5e4;
extern const Variant g_variants_fp4[];
extern const int g_num_variants_fp4;
extern const Variant g_variants_f32[];
extern const int g_num_variants_f32;
extern const Variant g_variants_i8[];
extern const int g_num_variants_i8;
// further variants of these types (translation units of their own: compile time)
extern const Variant g_variants_mid_f16[];
extern const int g_num_variants_mid_f16;
extern const Variant g_variants_mid_bf16[];
extern const int g_num_variants_mid_bf16;

}  // namespace tb
