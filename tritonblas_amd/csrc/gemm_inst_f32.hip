// fp32 tile GEMM kernels (v_mfma_f32_16x16x4_f32: full fp32 products and sums; this target has no
// reduced-precision fp32 matrix mode) for the four operand layout combinations, plus one
// element-wise-gather kernel for operands the vector loaders cannot address.
#include "gemm_variants.h"

namespace tb {

#define TB_LAYOUTS(BM, BN, WM, WN, MINB)                                       \
  make_variant<Tile<DT_F32, BM, BN, 128, WM, WN, LAY_K, LAY_K, MINB, true, 2>>(),   \
  make_variant<Tile<DT_F32, BM, BN, 128, WM, WN, LAY_K, LAY_M, MINB, true, 2>>(),   \
  make_variant<Tile<DT_F32, BM, BN, 128, WM, WN, LAY_M, LAY_K, MINB, true, 2>>(),   \
  make_variant<Tile<DT_F32, BM, BN, 128, WM, WN, LAY_M, LAY_M, MINB, true, 2>>()

#define TB_REGS_LAYOUTS(BM, BN, MINB)                                          \
  make_variant<Tile<DT_F32, BM, BN, 128, 2, 2, LAY_K, LAY_K, MINB, LOAD_REGS, 2>>(),   \
  make_variant<Tile<DT_F32, BM, BN, 128, 2, 2, LAY_K, LAY_M, MINB, LOAD_REGS, 2>>(),   \
  make_variant<Tile<DT_F32, BM, BN, 128, 2, 2, LAY_M, LAY_K, MINB, LOAD_REGS, 2>>(),   \
  make_variant<Tile<DT_F32, BM, BN, 128, 2, 2, LAY_M, LAY_M, MINB, LOAD_REGS, 2>>()

const Variant g_variants_f32[] = {
    TB_LAYOUTS(256, 256, 2, 4, 1),
    TB_LAYOUTS(128, 128, 2, 2, 2),
    TB_LAYOUTS(64, 64, 2, 2, 4),
    // unit stride, any alignment of the rows
    TB_REGS_LAYOUTS(128, 128, 2),
    TB_REGS_LAYOUTS(64, 64, 4),
    make_variant<Tile<DT_F32, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, false, 2>>(),
};
const int g_num_variants_f32 = sizeof(g_variants_f32) / sizeof(Variant);

}  // namespace tb
