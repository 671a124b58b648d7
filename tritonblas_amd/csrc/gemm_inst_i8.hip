// INT8 tile GEMM kernels (v_mfma_i32_16x16x64_i8, exact int32 sums over the K range of a work item).
// K-major operands take the LDS-direct kernels, everything else the element-wise-gather kernel.
#include "gemm_variants.h"

namespace tb {

const Variant g_variants_i8[] = {
    make_variant_w4<W4Tile<DT_I8>>(),
    make_variant<Tile<DT_I8, 256, 256, 128, 2, 4, LAY_K, LAY_K, 1, true, 2>>(),
    make_variant<Tile<DT_I8, 128, 128, 128, 2, 2, LAY_K, LAY_K, 2, true, 2>>(),
    make_variant<Tile<DT_I8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 4, true, 2>>(),
    // few tiles: what a CU copies for a K step is what the step takes, so tiles of a quarter and half of 64x64 on the CUs that would be idle, with half the steps
    make_variant<Tile<DT_I8, 32, 32, 256, 2, 2, LAY_K, LAY_K, 2, true, 4>>(),
    make_variant<Tile<DT_I8, 64, 32, 256, 2, 2, LAY_K, LAY_K, 1, true, 4>>(),
    // deeper copy pipelines of the small tile for problems with few tiles per CU
    make_variant<Tile<DT_I8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 3, LOAD_DIRECT, 3>>(),
    make_variant<Tile<DT_I8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, LOAD_DIRECT, 4>>(),
    // about one tile per CU: eight waves, as many copy stages as the LDS holds (the first: the 128x128 tile while every tile has a CU of its own)
    make_variant<Tile<DT_I8, 128, 128, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 4>>(),
    make_variant<Tile<DT_I8, 256, 128, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 3>>(),
    make_variant<Tile<DT_I8, 128, 64, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 4>>(),
    make_variant<Tile<DT_I8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, false, 2>>(),
};
const int g_num_variants_i8 = sizeof(g_variants_i8) / sizeof(Variant);

}  // namespace tb
