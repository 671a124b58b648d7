// bf16 tile GEMM kernels: every tile shape for the four operand layout combinations, plus one
// element-wise-gather kernel for operands the vector loaders cannot address.
#include "gemm_variants.h"

namespace tb {

#define TB_LAYOUTS(BM, BN, BK, WM, WN, MINB, STAGES)                                    \
  make_variant<Tile<DT_BF16, BM, BN, BK, WM, WN, LAY_K, LAY_K, MINB, true, STAGES>>(),   \
  make_variant<Tile<DT_BF16, BM, BN, BK, WM, WN, LAY_K, LAY_M, MINB, true, STAGES>>(),   \
  make_variant<Tile<DT_BF16, BM, BN, BK, WM, WN, LAY_M, LAY_K, MINB, true, STAGES>>(),   \
  make_variant<Tile<DT_BF16, BM, BN, BK, WM, WN, LAY_M, LAY_M, MINB, true, STAGES>>()

#define TB_REGS_LAYOUTS(BM, BN, WM, WN, MINB, STAGES)                                          \
  make_variant<Tile<DT_BF16, BM, BN, 128, WM, WN, LAY_K, LAY_K, MINB, LOAD_REGS, STAGES>>(),   \
  make_variant<Tile<DT_BF16, BM, BN, 128, WM, WN, LAY_K, LAY_M, MINB, LOAD_REGS, STAGES>>(),   \
  make_variant<Tile<DT_BF16, BM, BN, 128, WM, WN, LAY_M, LAY_K, MINB, LOAD_REGS, STAGES>>(),   \
  make_variant<Tile<DT_BF16, BM, BN, 128, WM, WN, LAY_M, LAY_M, MINB, LOAD_REGS, STAGES>>()

const Variant g_variants_bf16[] = {
    // hand-scheduled 4-wave kernel: K of four K steps at least (M-contiguous operands: an even number of them; others: where rest_of_k_pays),
    // no Stream-K tail (with one: K-major operands only)
    make_variant_w4<W4Tile<DT_BF16>>(),
    make_variant_w4<W4Tile<DT_BF16, LAY_K, LAY_M>>(),
    make_variant_w4<W4Tile<DT_BF16, LAY_M, LAY_K>>(),
    make_variant_w4<W4Tile<DT_BF16, LAY_M, LAY_M>>(),
    TB_LAYOUTS(256, 256, 128, 2, 4, 1, 2),
    TB_LAYOUTS(128, 128, 128, 2, 2, 2, 2),
    TB_LAYOUTS(64, 64, 128, 2, 2, 4, 2),
    // deeper copy pipelines of the small tile for problems with few tiles per CU (each K step then
    // waits less for its copy; fewer workgroups fit a CU)
    TB_LAYOUTS(64, 64, 128, 2, 2, 3, 3),
    TB_LAYOUTS(64, 64, 128, 2, 2, 2, 4),
    // a handful of rows against a long K: short, wide, deep tile with three copy stages
    TB_LAYOUTS(32, 128, 256, 1, 4, 1, 3),
    // few tiles: what a CU copies for a K step is what the step takes, so tiles of a quarter and half of 64x64 on the CUs that would be idle, with half the steps
    TB_LAYOUTS(32, 32, 256, 2, 2, 2, 4),
    TB_LAYOUTS(64, 32, 256, 2, 2, 1, 4),
    // unit stride, any alignment of the rows
    TB_REGS_LAYOUTS(128, 128, 2, 2, 2, 2),
    // (eight waves and a K step more in flight while every tile has a CU of its own)
    TB_REGS_LAYOUTS(128, 128, 4, 2, 1, 3),
    TB_REGS_LAYOUTS(64, 64, 2, 2, 2, 3),
    make_variant<Tile<DT_BF16, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, false, 2>>(),
};
const int g_num_variants_bf16 = sizeof(g_variants_bf16) / sizeof(Variant);

}  // namespace tb
