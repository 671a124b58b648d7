// FP8 (OCP e4m3) tile GEMM kernels.  The fast kernels take K-major operands; everything else goes
// through the element-wise-gather kernel.
#include "gemm_variants.h"

namespace tb {

const Variant g_variants_fp8[] = {
    // hand-scheduled 4-wave kernel: K of four K steps at least, an even number of them or where rest_of_k_pays
    make_variant_w4<W4Tile<DT_FP8>>(),
    make_variant<Tile<DT_FP8, 256, 256, 128, 2, 4, LAY_K, LAY_K, 1, true, 2>>(),
    make_variant<Tile<DT_FP8, 128, 128, 128, 2, 2, LAY_K, LAY_K, 2, true, 2>>(),
    make_variant<Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 4, true, 2>>(),
    make_variant<Tile<DT_FP8, 32, 128, 256, 1, 4, LAY_K, LAY_K, 1, true, 3>>(),
    // few tiles: what a CU copies for a K step is what the step takes, so tiles of a quarter and half of 64x64 on the CUs that would be idle, with half the steps
    make_variant<Tile<DT_FP8, 32, 32, 256, 2, 2, LAY_K, LAY_K, 2, true, 4>>(),
    make_variant<Tile<DT_FP8, 64, 32, 256, 2, 2, LAY_K, LAY_K, 1, true, 4>>(),
    // deeper copy pipelines of the small tile for problems with few tiles per CU (each K step then
    // waits less for its copy; fewer workgroups fit a CU)
    make_variant<Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 3, true, 3>>(),
    make_variant<Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, true, 4>>(),
    // about one tile per CU: eight waves, as many copy stages as the LDS holds (the first: the 128x128 tile while every tile has a CU of its own)
    make_variant<Tile<DT_FP8, 128, 128, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 4>>(),
    make_variant<Tile<DT_FP8, 256, 128, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 3>>(),
    make_variant<Tile<DT_FP8, 128, 64, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 4>>(),
    make_variant<Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, false, 2>>(),
};
const int g_num_variants_fp8 = sizeof(g_variants_fp8) / sizeof(Variant);

template <class T>
static bool group_kernel_of(const Variant& v, const void** out) {
  if (v.dt != T::DT || v.bm != T::BM || v.bn != T::BN || v.bk != T::BK || v.threads != T::THREADS || v.stages != T::STAGES || v.fast != LOAD_DIRECT || v.k_step_pairs) return false;
  *out = (const void*)&gemm_group_kernel<T, OneTile<T>::WHOLE_STEP>;
  return true;
}
template <class... T>
static const void* group_kernel_among(const Variant& v) {
  const void* k = nullptr;
  (void)(group_kernel_of<T>(v, &k) || ...);
  return k;
}
const void* group_kernel(const Variant& v) {
  return group_kernel_among<Tile<DT_FP8, 256, 128, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 3>, Tile<DT_FP8, 128, 128, 128, 2, 2, LAY_K, LAY_K, 2, LOAD_DIRECT, 2>,
                            Tile<DT_FP8, 128, 128, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 4>, Tile<DT_FP8, 128, 64, 128, 4, 2, LAY_K, LAY_K, 1, LOAD_DIRECT, 4>,
                            Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 4, LOAD_DIRECT, 2>, Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 3, LOAD_DIRECT, 3>,
                            Tile<DT_FP8, 64, 64, 128, 2, 2, LAY_K, LAY_K, 2, LOAD_DIRECT, 4>, Tile<DT_FP8, 32, 128, 256, 1, 4, LAY_K, LAY_K, 1, LOAD_DIRECT, 3>>(v);
}

}  // namespace tb
