// Analytical tile selector for the gfx950 kernel family: scores every built tile variant with a
// small roofline-style model (MFMA issue time, LDS read time, L2->LDS fill time, wave quantisation
// over the CUs, HBM time) and derives the launch parameters that go with the winner (GROUP_M, XCD
// remap, Stream-K grid, work-stealing slots).
#include <algorithm>
#include <cmath>
#include <cstring>
#include "selector.h"

namespace tb {

static int type_bits(int t) {
  switch (t) {
    case TB_F16: case TB_BF16: return 16;
    case TB_FP8_E4M3: case TB_FP8_E5M2: case TB_I8: return 8;
    case TB_FP4_E2M1: return 4;
    case TB_F32: return 32;
  }
  return 0;
}

// dense MFMA flops per clock per CU
static double mfma_flops_per_clk(int t) {
  switch (t) {
    case TB_F16: case TB_BF16: return 4096.0;
    case TB_FP8_E4M3: case TB_FP8_E5M2: case TB_I8: return 8192.0;
    case TB_FP4_E2M1: return 16384.0;
    case TB_F32: return 256.0;
  }
  return 1024.0;
}

void default_hw(tb_hw* hw) {
  std::memset(hw, 0, sizeof(*hw));
  hw->n_cu = 256; hw->num_xcd = 8; hw->cu_per_xcd = 32; hw->lds_bytes = 163840; hw->l2_bytes = 4 << 20;
  hw->clock_khz = 2400000; hw->mem_clock_khz = 2000000; hw->wave_size = 64; hw->hbm_gbps = 8000.0;
  std::strncpy(hw->arch, "gfx950", sizeof(hw->arch) - 1);
}

int ws_counters_per_xcd(int64_t total_tiles) {
  if (total_tiles <= 512) return 8;
  if (total_tiles <= 1536) return 4;
  if (total_tiles <= 2048) return 2;
  return 1;
}

// Reference origami.py:288-311: up to 4 tiles per CU everything stays XCD-local; above that the local
// share falls by 5 % per extra tile per CU, down to one half.  The local queues never get more than
// divides evenly (the reference's formula hands out one tile per XCD even when there are fewer tiles
// than XCDs).
void hierarchical_split(int64_t total_tiles, int hw_cus, int num_xcds, int64_t* local_per_xcd, int64_t* global_tiles) {
  const double tiles_per_cu = (double)total_tiles / std::max(hw_cus, 1);
  const double local_frac = std::max(0.5, 1.0 - std::max(0.0, tiles_per_cu - 4.0) * 0.05);
  int64_t local = std::max<int64_t>((int64_t)((double)total_tiles * local_frac) / num_xcds, 1);
  local = std::min(local, total_tiles / num_xcds);
  *local_per_xcd = local;
  *global_tiles = total_tiles - local * num_xcds;
}

static int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Workgroups of one variant that fit a CU (LDS and wave slots), capped by what the kernel was built for.
int variant_occupancy(const TileInfo& v, const tb_hw& hw) {
  int by_lds = std::max(1, hw.lds_bytes / std::max(1, v.lds_bytes));
  int by_waves = std::max(1, (8 * 4) / (v.threads / 64));
  return std::max(1, std::min({by_lds, by_waves, v.minb}));
}

// What is left of K behind an even number of K steps costs the hand-scheduled kernel a fixed time per tile, 1.3 us for a part of a step and 3.2 to 3.6 for a
// whole one and more, a tile that ends inside C another 2 to 3 (they show where all tiles run at once), results of 32 or 8 bits, which the eight-wave kernel
// stores no slower, 3 to 6; each step of its K loop gains 0.15 us on the eight-wave kernel, and several tiles after one another 1 us a tile.
// Hand-scheduled against eight-wave kernel, us.  int8 to bf16, 4096x4096: 6 steps and a quarter 23.0 and 22.4, 10 27.5 and 27.5, 16 33.7 and 35.6, 64 89.5 and
// 99.6; 7 whole steps 24.6 and 21.5, 25 42.5 and 42.5, 33 50.3 and 51.9.  3000x5376: 10 steps and a quarter 13 % slower, 20 level; 11 whole ones 23 % slower,
// 41 level.  7000x9000: 4 and a quarter 59.1 and 60.7; 7 whole ones 73.0 and 68.2, 13 97.9 and 96.6.  FP8 to fp32, 4096x4096: 10 steps and a quarter 37.0 and 34.8,
// 32 level; 25 whole ones 54.1 and 51.6, 49 level; to e4m3: 10 40.0 and 36.0, 40 level; 25 56.0 and 51.1, 65 level.  The other types within 3 % of these ratios.
bool rest_of_k_pays(int64_t m, int64_t n, int64_t k, int bk, int c_bits, int n_cu) {
  const int64_t steps = k / bk, tiles = cdiv(m, 256) * cdiv(n, 256);
  const bool whole = steps % 2 != 0;      // (what is left holds a whole step)
  if (c_bits == 32) return steps >= (whole ? 48 : 32);
  if (c_bits == 8) return steps >= (whole ? 56 : 40);
  if (tiles > 2 * (int64_t)n_cu) return steps >= (whole ? 12 : 4);
  const bool ragged = tiles <= n_cu && (m % 256 != 0 || n % 256 != 0);
  return steps >= (whole ? (ragged ? 36 : 24) : (ragged ? 20 : 10));
}

// Whether they are the faster ones for an even number of K steps.  They store a tile under the next one's K loop, which one round of tiles has no use for, and
// the eight-wave kernel starts sooner (one tile to a workgroup).  Hand-scheduled by eight-wave time, 256x256 tiles: one round, 16-bit 1.28 at 4 steps, 1.16 at 8, 1.10 at 12, 1.03 at 16,
// 0.98 at 24, 0.92 at 40; int8 1.41, 1.22, 1.13, 1.09, 1.01 at 24, 0.98 at 36; FP8 1.54, 1.41, 1.25, 1.19, 1.05 at 24, 1.01 at 32, 0.97 at 40; MXFP4 1.55, 1.30, 1.20, 1.15,
// 0.97 at 24, 0.94 at 32 (7860x1552x1536 28.3 us and 19.5).  Two rounds: 1.08 to 1.10 at 4, 1.01 at 12, 0.92 to
// 0.97 at 16 (MXFP4 1.28, 1.10, 1.05 at 14).  More: 0.91 to 1.0 (8 bits 1.01 to 1.13 at 4).  Launches of one tile to a workgroup only: from a caller's grid or the
// work-stealing queues the eight-wave kernel loops too, without either advantage.  Hand-scheduled and eight-wave, us: bf16 4096x4096x1280 on 64 workgroups 96.6 and 122.5, from the
// queues 105 and 125, from those of the whole device 42.2 and 43.5; FP8 4096x4096x3840 on 128 70 and 83; int8 2048x4096x1536 on 128, a tile each, 22.3 and 25.6.
bool even_k_pays(int64_t m, int64_t n, int64_t k, int bk, int type, int n_cu) {
  const int64_t steps = k / bk, tiles = cdiv(m, 256) * cdiv(n, 256);
  if (tiles > 2 * (int64_t)n_cu) return true;
  if (tiles > n_cu) return steps >= (type == TB_FP4_E2M1 ? 16 : 12);
  return steps >= (type == TB_FP8_E4M3 || type == TB_FP8_E5M2 ? 32 : 24);
}

// Measured behaviour of the built kernels on MI355X that the model is anchored to:
//   * a CU that is kept busy by `occ` resident workgroups finishes one K step of one tile every
//     ideal_step / eff: eff = fraction of the MFMA peak the kernel family sustains for that tile;
//   * a workgroup cannot turn a K step around faster than ~0.3 us (barrier + L2 round trip) plus the
//     time its own copy takes at the ~100 GB/s one workgroup pulls, times `lat`: small problems want enough tiles to put several
//     workgroups on every CU or a variant with deep copy stages, and
//     long-K problems with few rows want the deep 32x128x256 tile;
//   * per tile: epilogue + first-copy latency, `tile_us`.
// The figures of the 16- and 8-bit types are a fit to 117 problems (80..8192 rows, operands that come from HBM, every tile timed): the tile the
// model picks takes 1.008 (bf16), 1.003 (FP8) and 1.022 (int8) times the fastest one's time in the geometric mean, 1.12, 1.09 and 1.26 at worst;
// 19 fp32 problems 1.000.
// w4: the hand-scheduled 4-wave kernel runs the 256x256 tile (four K steps at least, see rest_of_k_pays; rounds of 256 tiles at
// K = 4096 and 8192: FP8 46.5 and 85.7 us, bf16 89 and 178 us, MXFP4 8192x8192x16384 in 0.40-0.43 ms).
struct Family {
  double eff, tile_us, lat;
};
// lat: the deeper variants of the 64x64 tile run while at most two (three) tiles per CU exist, the eight-wave 128x128 tile while every tile has
// a CU of its own (find_variant)
static Family family(int dt, const TileInfo& v, bool w4, int64_t tiles, int n_cu, bool grouped, bool older) {
  const int area = v.bm * v.bn;
  const int cls = (v.bm < 64 || v.bn < 64) ? 5 : area >= 256 * 256 ? 0 : area >= 256 * 128 ? 1 : area >= 128 * 128 ? 2 : area >= 128 * 64 ? 3 : 4;
  if (dt == TB_FP4_E2M1 || dt == TB_F32) {
    static const double f4[6] = {0.50, 0.36, 0.36, 0.22, 0.22, 0.10};   // (256x256: 8192x8192x16384 in 0.43-0.47 ms)
    // (the fp32 matrix pipe is slow enough to hide everything else; four 64x64 workgroups to a CU hide more of it than two of 128x128:
    // 2048^3 130 us against 147, 1000x3000x1504 79 and 108.  One 64x64 workgroup to a CU hides nothing, its step takes twice the MFMAs' time: 32x32 tiles
    // fill the CUs better there, 1664x480x5568 164 us and 105, 512x2048x2848 86 and 59, 240x3552x4672 140 and 91.  Of 894 problems, 100..8192 a side, four orders, the tile
    // taken was 1.029 times the best one's time in the geometric mean, 1.57 at most; with these three figures 1.003 and 1.19.  Stream-K launches cut such tiles
    // instead and keep their own: `older`.)
    static const double f32[6] = {0.92, 0.77, 0.77, 0.86, 0.82, 0.70}, f32_sk[6] = {0.92, 0.77, 0.77, 0.86, 0.86, 0.65};
    // (MXFP4 256x256 with eight waves, a round of one tile to a workgroup: 2 to 16 K steps 13.9 to 34.1 us, within 1.5 of the hand-scheduled kernel's figures)
    const bool w8_one = cls == 0 && dt == TB_FP4_E2M1 && !older && !grouped && tiles <= n_cu;
    const double tile_us = cls == 0 ? (w4 || w8_one ? 8.0 : 12.0) : (cls <= 2 ? 4.0 : 3.0);
    double lat = dt != TB_F32 ? 1.0 : cls == 5 ? (older ? 0.6 : 0.4) : cls == 4 && !older ? 1.7 : 1.0;
    if (dt == TB_FP4_E2M1 && !grouped) {      // (three copy stages: see find_variant)
      if (cls == 2 && tiles <= n_cu && v.bk == 256) lat = 0.88;
      if (cls == 3) lat = 0.85;
      if (cls == 4 && tiles <= 2 * (int64_t)n_cu) lat = 0.66;
    }
    return {dt == TB_F32 ? (older ? f32_sk : f32)[cls] : ((w4 && cls == 0) || w8_one ? 0.56 : f4[cls]), tile_us, lat};
  }
  //                                     256x256  256x128 128x128 128x64 64x64  32x128
  static const double eff16[6] = {0.69, 0.506, 0.388, 0.357, 0.246, 0.12}, us16[6] = {9.5, 5.0, 3.8, 2.8, 3.0, 3.0};
  static const double eff8[6] = {0.716, 0.50, 0.403, 0.303, 0.232, 0.15}, us8[6] = {6.8, 6.2, 4.0, 2.3, 2.4, 3.0};
  // (int8: fitted on 700 problems, 65..8192 x 256..16384 x 256..16384: the tile taken 1.007 times the best one's time in the geometric mean where it was 1.020;
  // 4096x1488x8064 88 us in 128x64, 58 in 256x128, 2240x3712x768 25 in 256x256 and 16 in 64x64.  Stream-K launches keep theirs.)
  static const double effi[6] = {0.665, 0.46, 0.367, 0.293, 0.159, 0.15}, usi[6] = {6.3, 5.8, 4.4, 2.6, 1.8, 3.0};
  static const double effi_sk[6] = {0.705, 0.368, 0.367, 0.293, 0.211, 0.15}, usi_sk[6] = {7.0, 5.8, 3.5, 2.3, 2.4, 3.0};
  const bool half = dt == TB_F16 || dt == TB_BF16;
  // 32x32 and 64x32, 256-byte K steps: where 64x64 tiles leave CUs idle.  A step takes what its CU copies for it, about 26 bytes a cycle however deep the
  // pipeline; a quarter of the bytes on four times the CUs.  bf16, 64x64 and 32x32, us: 256x256x7904 32.2 and 17.8, 128x1024x14336 65.3 and 33.1, 96x1280x5120 22.0 and 12.6,
  // 200x1000x2000 11.4 and 6.9; FP8 256x256x7904 19.9 and 9.9, 130x520x3008 8.6 and 5.7.  64x32: bf16 128x4096x4096 21.6 and 16.6.  On 1500 problems of at most 768 tiles of 64x64 each in
  // bf16 and FP8 the choice among the three takes 1.003 and 1.015 times the best one's time, 1/1.35 and 1/1.26 of what 64x64 takes.
  if (v.bn == 32) return half ? (v.bm == 32 ? Family{0.10, 1.2, 0.33} : Family{0.12, 1.2, 0.36}) : v.bm == 32 ? Family{0.10, 1.2, 0.36} : Family{0.15, 1.5, 0.55};
  Family f = half ? Family{eff16[cls], us16[cls], 1.0} : dt == TB_I8 ? (older ? Family{effi_sk[cls], usi_sk[cls], 1.0} : Family{effi[cls], usi[cls], 1.0}) : Family{eff8[cls], us8[cls], 1.0};
  // (the eight-wave 256x256 kernel.  16-bit, M-contiguous operands and a rest of K, 44 problems of 256..8192 in three orders: the model's tile 1.013 times the
  // fastest one's time; 1.021 with 0.89 and 4 us more a tile, which kept the library's choice off this kernel: 7848x7808x528 86 us, 256x128 104)
  if (cls == 0 && !w4) { f.eff *= half ? 0.97 : dt == TB_I8 && !older ? 0.91 : 0.86; f.tile_us += half ? 0.0 : 4.0; }
  if (grouped) return f;
  if (cls == 1 && !half && dt != TB_I8) f.lat = 1.19;
  if (cls == 2 && tiles <= n_cu) f.lat = 0.825;
  if (cls == 3) f.lat = half ? 0.61 : 0.645;
  if (cls == 4) f.lat = tiles <= 2 * (int64_t)n_cu ? 0.47 : tiles <= 3 * (int64_t)n_cu ? 0.85 : dt == TB_I8 && !older ? 0.8 : 1.0;
  return f;
}

// Stream-K launch grid for `total` tiles of `k_iters` K steps on `slots` co-resident workgroups of `n_cu` CUs.
//   * at least one whole tile per CU, but fewer tiles than slots: one workgroup per tile, nothing is
//     split -- every CU is busy, and cutting tiles only to raise the occupancy costs more in partial-tile
//     traffic than it gains (measured: 64x28672x8192 fp8, 448 tiles of 64x64: 38 us whole, 60 us in halves);
//   * fewer tiles than CUs: every tile is cut into the same number s of K segments (grid = total * s).
//     s is a power of two (segment counts that do not divide the K steps evenly were up to 2x slower:
//     32x4096x14336 bf16, 112 steps: s = 4 and 8 28 us, s = 5..7 31..53 us), at most what fits the slots,
//     never leaving fewer than 8 K steps per segment, and the one that minimises
//     steps_per_segment * step_us + (s - 1) * fix_us -- the owner adds the other segments' partial tiles
//     one after the other;
//   * tiles >= slots: every slot takes part: whole tiles first, the last total % slots tiles are shared --
//     unless another round of whole tiles is expected to be as fast (large tiles have expensive partial
//     tiles: 2048x14336x4096 bf16, 448 tiles of 256x256 on 256 slots: 209 us in two rounds, 253 us with a
//     shared tail); the return value `total` means "whole tiles only".
// A last round that does not fill the CUs is cheaper than a full one for the 256x256 tiles (one workgroup per CU):
// the busy CUs run at a higher clock and share the L2s and the fabric with fewer others.  Measured, FP8 and bf16,
// K = 4096 and 8192, as a fraction of a full round: 0.66-0.69 with 6 % of the CUs busy, 0.84-0.91 with a quarter,
// 0.87-0.93 with half or three quarters.  f: the busy fraction.
static double partial_round_factor(double f) {
  if (f <= 0.0 || f >= 1.0) return 1.0;
  return f < 0.25 ? 0.65 + f : (f < 0.75 ? 0.9 : 0.9 + 0.4 * (f - 0.75));
}
static const double kSharedTailFactor = 4.0;
// What the exchange of partial tiles costs the workgroup that finishes a tile cut into `segments` pieces, when
// `partials` partial tiles are exchanged at about the same time.  xchg_us = 0 (the 8-wave kernels): fix_us per extra
// piece, one after the other, times `crowd` when a whole grid shares a tail.  xchg_us > 0 (the 4-wave 256x256 kernels,
// whose pieces exchange 256 KB each): the exchange is bound by what all of them move together -- 128 tiles cut in two
// 30 us, 64 tiles cut in four 43 us, a tail of 280 tiles shared by 256 workgroups 60 us: 0.23 us per partial tile,
// about 1.1 TB/s -- and never faster than one workgroup reads its partners' tiles (fix_us each).
static double exchange_us(double segments, double partials, double fix_us, double xchg_us, double crowd) {
  if (segments <= 1.0) return 0.0;
  if (xchg_us > 0.0) return std::max((segments - 1.0) * fix_us, partials * xchg_us);
  return (segments - 1.0) * fix_us * crowd;
}
int streamk_grid(int64_t total, int64_t k_iters, int slots, int n_cu, double step_us, double fix_us, double xchg_us) {
  if (total <= 0 || slots <= 0) return 1;
  if (total >= slots) {
    const int64_t tail = total % slots;
    if (tail == 0) return slots;
    // (a tail shared by the whole grid costs about four times the per-segment figure that the split of
    // a few tiles shows: 2048x28672x8192 FP8, 128 tiles of 256x256 shared by 256 workgroups, ~100 us on
    // top of their K steps; 1024x28672x8192, 192 shared tiles, the same)
    const double segments = std::ceil((double)slots / tail);
    const double shared = std::ceil((double)tail * k_iters / slots) * step_us +
                          exchange_us(segments, (double)(slots - tail), fix_us, xchg_us, kSharedTailFactor);
    const double whole = (double)k_iters * step_us * (xchg_us > 0.0 ? partial_round_factor((double)tail / slots) : 1.0);
    return shared < whole ? slots : (int)std::min<int64_t>(total, INT32_MAX);
  }
  if (total >= n_cu) return (int)total;
  const int64_t smax = std::max<int64_t>(1, slots / total);
  int64_t best_s = 1;
  double best = 0;
  for (int64_t s2 = 1; s2 <= smax && (s2 == 1 || k_iters / s2 >= 8); s2 *= 2) {
    // workgroups per CU grow with the split; beyond one per CU they share its matrix pipe
    const double share = std::max(1.0, (double)(total * s2) / n_cu);
    const double cost = std::ceil((double)k_iters / s2) * step_us * std::sqrt(share) +
                        exchange_us((double)s2, (double)(total * (s2 - 1)), fix_us, xchg_us, 1.0);
    if (s2 == 1 || cost < best) { best = cost; best_s = s2; }
  }
  return (int)(total * best_s);
}

// A selector for some of the CUs: its launches carry a grid, which is what these CUs hold of the tile.
static bool of_the_cus(const tb_hw& hw) { return hw.n_cu < hw.num_xcd * hw.cu_per_xcd; }
static int64_t workgroups_of(const TileInfo& v, const tb_hw& hw, TileUse use) { return use.workgroups > 0 ? use.workgroups : (int64_t)hw.n_cu * variant_occupancy(v, hw); }

static double score(const tb_problem& pr, const tb_hw& hw, const TileInfo& v, bool streamk, double* comp_us,
                    double* mem_us, int* sk_grid_out = nullptr, TileUse use = {}) {
  const double clk = hw.clock_khz * 1e3;
  const int bits = type_bits(pr.a_type);
  const double esz = bits / 8.0;
  const int64_t tiles_m = cdiv(pr.m, v.bm), tiles_n = cdiv(pr.n, v.bn);
  const int64_t tiles = tiles_m * tiles_n + (pr.num_groups > 0 ? (int64_t)pr.num_groups * tiles_n / 2 : 0);
  const int64_t k_iters = cdiv(pr.k, v.bk);
  const int occ = variant_occupancy(v, hw);
  const int area = v.bm * v.bn;

  const double ideal_step_us = 2.0 * v.bm * v.bn * v.bk / mfma_flops_per_clk(pr.a_type) / clk * 1e6;
  // (an even number of whole K steps; what is behind them, up to two steps at about 3.5 us each and 2 more, only from K-contiguous operands, not MXFP4, and
  // without an int8 result: the kernels that find_variant has.  Of the Stream-K launches those that share no tile have them too; the others are
  // priced alike: with the eight-wave kernel's figures for both FP8 1556x10016x1840 goes from 48 to 56 us, and 44 bf16 problems come out level)
  const bool part = of_the_cus(hw);
  const int64_t whole_k = pr.k / v.bk;
  const bool rest = pr.k % (2 * (int64_t)v.bk) != 0;
  const bool w4 = v.threads == 256 && area >= 256 * 256 && whole_k >= 4 &&
                  (!rest ? streamk || use.looped || part || pr.num_groups > 0 || even_k_pays(pr.m, pr.n, pr.k, v.bk, pr.a_type, hw.n_cu) : (pr.a_type != TB_FP4_E2M1 && pr.c_type != TB_I8 && pr.a_k_contiguous && pr.b_k_contiguous &&
                             rest_of_k_pays(pr.m, pr.n, pr.k, v.bk, type_bits(pr.c_type), hw.n_cu)));
  int64_t k_steps = k_iters;
  double rest_us = 0.0;
  if (w4 && rest && !streamk) {
    k_steps = whole_k & ~1ll;
    rest_us = 2.0 + 3.5 * (double)(k_iters - k_steps);
  }
  // (the figures of int8 and fp32 were fitted on launches of the whole device.  On 64 workgroups fp32 1664x480x5568 takes 418 us by the older ones, in 64x64 tiles, 563 by these in
  // 32x32, which are ahead there only where all of them run at once: 256x512x2048 on 128 42 and 20.  int8 640x1024x3072 on 32 CUs 16.8 us in 128x128, 24.6 in 256x128.)
  const bool kept = part || use.workgroups > 0;
  const bool at_once = pr.a_type == TB_F32 && cdiv(pr.m, 32) * cdiv(pr.n, 32) <= workgroups_of(v, hw, use);
  const Family fam = family(pr.a_type, v, w4, cdiv(pr.m, v.bm) * cdiv(pr.n, v.bn), hw.n_cu, pr.num_groups > 0, streamk || (kept && !at_once));
  const double t_thru = ideal_step_us / fam.eff;   // CU time per tile K step, saturated
  const double t_lat = (0.30 + (v.bm + v.bn) * (v.bk * esz) / 1.0e5) * fam.lat;   // floor per K step of one workgroup
  const double t_tile = fam.tile_us + rest_us;
  auto last_round = [&](int64_t n_tiles, int64_t per_round) {
    const int64_t r = n_tiles % per_round;
    if (r == 0 || area < 256 * 128) return 1.0;
    if (area < 256 * 256) return pr.a_type == TB_F16 || pr.a_type == TB_BF16 ? 1.0 : 0.6 + 0.4 * (double)r / per_round;
    return partial_round_factor((double)r / per_round);
  };

  double us;
  if (streamk) {
    // one extra K segment of a tile costs its partial tile written through, polled for and added by the
    // owner, one after the other: ~1.5 us + the fp32 tile at ~10 GB/s (fitted on segment-count sweeps:
    // 32x128 tiles ~3 us, 128x128 tiles ~8 us, 256x256 tiles ~30 us per extra segment)
    // The 4-wave 256x256 kernels (256 threads) exchange partial tiles straight from the accumulators with 16 loads in
    // flight per lane: 4.5 us per partner for one workgroup alone, and 0.23 us per partial tile of the whole launch
    // (see exchange_us).
    const bool big4 = w4 && pr.k % (4 * (int64_t)v.bk) == 0;   // (the 4-wave Stream-K kernel cuts K at multiples of four steps)
    const double fix_us = big4 ? 4.5 : 1.5 + area * 4.0 / 10e3;
    const double xchg_us = big4 ? 0.23 : 0.0;
    const int slots = hw.n_cu * occ;
    const int grid = streamk_grid(tiles, k_iters, slots, hw.n_cu, std::max(t_thru, t_lat), fix_us, xchg_us);
    if (sk_grid_out) *sk_grid_out = grid;
    const int launched = (int)std::min<int64_t>(grid, slots);     // (grid == tiles > slots: whole tiles, resident grid loops)
    const double w = (double)cdiv(launched, hw.n_cu);             // workgroups sharing the busiest CU
    const double t_step = std::max(w * t_thru, t_lat);
    if (grid >= tiles && tiles > slots) {
      us = ((double)(cdiv(tiles, slots) - 1) + last_round(tiles, slots)) * (k_iters * t_step + t_tile);
    } else {
      const int64_t dp_rounds = tiles / grid, tail = tiles % grid;
      us = (double)dp_rounds * (k_iters * t_step + t_tile);
      if (tail > 0) {
        const double iters = std::ceil((double)tail * k_iters / grid);
        const double segments = std::ceil((double)grid / tail);
        // (tiles < grid: every tile is cut into `segments` pieces; otherwise a tail shared by the whole grid)
        const double partials = dp_rounds > 0 ? (double)(grid - tail) : (double)tail * (segments - 1.0);
        us += iters * t_step + exchange_us(segments, partials, fix_us, xchg_us, dp_rounds > 0 ? kSharedTailFactor : 1.0) + t_tile;
      }
    }
  } else {
    // the busiest CU works through c tiles, occ at a time
    const int64_t c = cdiv(tiles, hw.n_cu);
    const int64_t full = c / occ, rem = c % occ;
    us = (double)full * (k_steps * std::max(occ * t_thru, t_lat) + t_tile);
    if (rem) us += k_steps * std::max((double)rem * t_thru, t_lat) + t_tile;
    if (occ == 1 && c > 1) us -= (1.0 - last_round(tiles, hw.n_cu)) * (k_steps * std::max(t_thru, t_lat) + t_tile);
  }
  *comp_us = us;

  // HBM: every operand once
  const double c_bytes = type_bits(pr.c_type) / 8.0;
  const double a_bytes = (double)pr.m * pr.k * esz, b_bytes = (double)pr.n * pr.k * esz * std::max(1, pr.num_groups);
  const double c_out = (double)pr.m * pr.n * c_bytes;
  // few workgroups cannot pull the full HBM rate: ~45 GB/s per busy CU
  const double busy_cus = std::min<double>(hw.n_cu, streamk ? hw.n_cu : (double)tiles);
  const double hbm = std::min(hw.hbm_gbps * 0.65, busy_cus * 45.0);
  *mem_us = (a_bytes + b_bytes + c_out) / (hbm * 1e9) * 1e6;
  return std::max(*comp_us, *mem_us) + 3.0;
}

int streamk_grid_for(const tb_problem& pr, const tb_hw& hw, const TileInfo& v) {
  double c, m;
  int grid = 1;
  score(pr, hw, v, true, &c, &m, &grid);
  return grid;
}

double estimate_tile_us(const tb_problem& pr, const tb_hw& hw, const TileInfo& v, bool streamk, TileUse use) {
  double c, m;
  return score(pr, hw, v, streamk, &c, &m, nullptr, use);
}

// A grouped FP8 launch.  The rows of an expert are taken as spread around their mean, by chance and by 7 % of it, which gives the row blocks to expect; per variant:
// us a 128-byte K step and tile keeps a CU busy, the least a step takes, us a tile costs beside its steps, us per MB of operands and results, and
// how much of a last round that is not full is waited for (a hundredth of a round more than whole ones is an expectation that chance makes, not a round: 16 experts of
// 1984x3584, 6786 rows, 256.2 tiles of 256x256 to expect).  The two times are those of different units and add up as squares do.  Fitted on 1298 random launches
// (4, 8 and 16 experts, 16..16384 rows, n 1024..14336, k 1024..8192) per variant: 8 to 17 % off at one sigma; the variant it picks takes 1.032 times (on 420 others, as built, 1.025) the best
// one's time in the geometric mean, one picked by the rows per expert alone (256x256 from 192, 128x128 from 96, else 64x64) 1.214 times.
// 4 experts of 1536x7168, 1000 rows: 89 us that way, 29 now; 16 of 1024x8192, 600 rows: 54 and 34.
double estimate_grouped_us(const tb_problem& pr, const tb_hw& hw, const TileInfo& v) {
  struct Fit { int bm, bn, waves, stages; double step, least, tile, mb, round; };
  static const Fit fits[] = {
      {256, 256, 4, 2, 1.080, 0.0, 15.9, 0.202, 1.0},    {256, 256, 8, 2, 1.318, 0.0, 10.0, 0.193, 1.0},   {256, 128, 8, 3, 0.743, 0.0, 6.55, 0.151, 1.0},
      {128, 128, 4, 2, 0.541, 0.805, 3.75, 0.130, 0.75}, {128, 128, 8, 4, 0.469, 0.0, 4.92, 0.148, 1.0},   {128, 64, 8, 4, 0.150, 0.348, 3.70, 0.101, 0.75},
      {64, 64, 4, 2, 0.075, 0.751, 2.65, 0.140, 1.0},    {64, 64, 4, 3, 0.075, 0.562, 2.71, 0.139, 0.75},  {64, 64, 4, 4, 0.075, 0.397, 3.01, 0.139, 0.5},
      {32, 128, 4, 3, 0.075, 0.299, 3.29, 0.158, 0.75}};
  const Fit* f = nullptr;
  for (auto& x : fits) if (x.bm == v.bm && x.bn == v.bn && x.waves == v.threads / 64 && x.stages == v.stages) f = &x;
  if (!f || pr.num_groups <= 0 || pr.m <= 0) return 0.0;
  const double e = pr.num_groups, rows = (double)pr.m, mean = rows / e;
  const double spread = std::max({std::sqrt(mean * (1.0 - 1.0 / e)), 0.07 * mean, 1e-6});
  const double used = e * (1.0 - std::pow(1.0 - 1.0 / e, rows));      // experts with rows at all
  double blocks = used;
  for (int64_t at = v.bm; (double)at < mean + 5.0 * spread; at += v.bm) blocks += e * 0.5 * std::erfc(((double)at + 0.5 - mean) / (spread * std::sqrt(2.0)));
  const double tiles = blocks * (double)cdiv(pr.n, v.bn), steps = (double)cdiv(pr.k, 128);
  const int occ = variant_occupancy(v, hw);
  const double rounds = tiles / hw.n_cu / occ, slack = 0.01;
  double us;
  if (rounds <= 1.0 + slack) us = steps * std::max(std::ceil(tiles / hw.n_cu - slack) * f->step, f->least) + f->tile;
  else us = (f->round * std::ceil(rounds - slack) + (1.0 - f->round) * rounds) * (steps * std::max(occ * f->step, f->least) + f->tile);
  // (in several rounds the four-wave kernel stores a tile under the next one's K loop, 4 us of its cost, and 256x128 tiles fall out of step: 16 experts of 4096x2048, 16384 rows
  // 157 us and 186 where one round of both is priced alike)
  if (rounds > 1.0 + slack && v.bm == 256) us = v.bn == 128 ? us * 1.05 : v.threads == 256 ? us - 4.0 * (rounds - 1.0) : us;
  const double mb = (used * pr.n * pr.k + rows * pr.k + rows * pr.n * type_bits(pr.c_type) / 8.0) * 1e-6;
  return 3.0 + std::hypot(us, mb * f->mb);
}

// The streaming kernel for a handful of rows (skinny.hip), `cols` columns of the weight to a workgroup.  Two things bound it, and the nearer they
// are to each other the more they add up: the weight from HBM (5.7 TB/s with non-temporal reads) and what all workgroups read
// through the L2s, A once per workgroup (15 TB/s).  More than 32 rows in more than one round of workgroups cost a cold start per round.
// (52 cold-weight points, M = 1..64, N = 1024..28672, K = 1024..28672, within 15 %.)
double estimate_streaming_us(const tb_problem& pr, const tb_hw& hw, int cols) {
  const double row_bytes = (double)pr.k * type_bits(pr.a_type) / 8.0;
  const double groups = std::ceil((double)pr.n / cols), rounds = std::ceil(groups / hw.n_cu);
  const double hbm = ((double)pr.n + pr.m) * row_bytes / (hw.hbm_gbps * 0.71 * 1e3);     // bytes per us
  const double l2 = groups * (double)(pr.m + cols) * row_bytes / (hw.hbm_gbps * 1.9 * 1e3);
  return 3.0 + std::cbrt(hbm * hbm * hbm + l2 * l2 * l2) + (pr.m > 32 ? 2.5 * (rounds - 1.0) : 0.0);
}

// What the streaming kernel takes at most, with room to spare: 13 us and the weight at 3.4 (16-bit) to 4.6 TB/s, A from the L2s once per 64 columns
// (8x14336x4096 bf16: 48 us here, 19 to 25 measured).  The line for launches whose grid is the caller's: of 4000 random ones with 1 to 32 rows and 32 to 128
// workgroups 1267 leave their grid for the whole device by it, by the estimate above all but three would.
double streaming_bound_us(const tb_problem& pr, const tb_hw& hw) {
  const double esz = type_bits(pr.a_type) / 8.0;
  const double weight = (double)pr.n * pr.k * esz, a_reread = std::ceil(pr.n / 64.0) * (double)pr.m * pr.k * esz;
  return 13.0 + weight / (hw.hbm_gbps * (esz > 1.0 ? 0.425 : 0.575) * 1e3) + a_reread / (hw.hbm_gbps * 2.125 * 1e3);
}

bool narrow_tile(const TileInfo& v) { return v.bn == 32 && v.dt != TB_F32; }

int select_tile(const tb_problem& pr, const tb_hw& hw, const TileInfo* tiles, int ntiles, tb_selection* out, TileUse use) {
  int best = -1;
  double best_t = 0, best_c = 0, best_m = 0;
  for (int i = 0; i < ntiles; ++i) {
    const TileInfo& v = tiles[i];
    if (!v.fast) continue;  // the gather kernels are a fallback, never a choice of the model
    if (v.lds_bytes > hw.lds_bytes) continue;
    if (use.block_k > 0 && v.bk != use.block_k) continue;
    // decode-like problems (a handful of rows): tiles taller than twice the row count only add
    // LDS traffic and idle MFMA rows when a shorter tile exists
    // (the small tiles of few-tile problems, see family(): whole tiles only, and not where the streaming kernel is at home, which is weighed against the others)
    if (narrow_tile(v) && (pr.streamk || pr.num_groups > 0 || (pr.m <= 64 && pr.n >= 1024 && pr.a_k_contiguous && pr.b_k_contiguous))) continue;
    // (they are for CUs that would be idle: a launch kept to some workgroups takes them where each has one tile at most.  bf16 512x512x8192 on 16 workgroups 125 us in 64x64,
    // 277 in 32x32; 256x256x7904 on 32 32 and 36, on 64 32 and 20.  From the work-stealing queues, where each workgroup more costs a walk over the counters, 64x32
    // alone, where every CU has a tile at most: 0.58 to 0.98 of the time of 64x64 on 14 such shapes in bf16, 0.45 to 1.02 in FP8; 32x32 up to 1.31, 64x32 with 304 tiles 1.27.)
    if (narrow_tile(v) && (use.queues || use.workgroups > 0 || of_the_cus(hw)) && (cdiv(pr.m, v.bm) * cdiv(pr.n, v.bn) > workgroups_of(v, hw, use) || (use.queues && v.bm == 32))) continue;
    bool shorter_exists = false;
    for (int q = 0; q < ntiles; ++q) shorter_exists |= tiles[q].fast && !narrow_tile(tiles[q]) && tiles[q].bm < v.bm && tiles[q].bm >= pr.m;
    if (shorter_exists && pr.num_groups == 0) continue;
    if (pr.num_groups > 0) {
      // grouped, with a tail that is cut into K ranges or short last blocks left to a second launch (other launches: estimate_grouped_us): the row counts live on the
      // device; size the tile for the average group so that the ragged last row block of each group wastes little
      const int64_t avg = std::max<int64_t>(1, pr.m / pr.num_groups);
      const int want = avg >= 192 ? 256 : (avg >= 96 ? 128 : 64);
      if (v.bm != want || v.bn != want) continue;
    }
    double c, m;
    double t = score(pr, hw, v, pr.streamk != 0, &c, &m, nullptr, use);
    // prefer the larger tile on ties (less L2 traffic than the model resolves)
    if (best < 0 || t < best_t * 0.995 || (t <= best_t * 1.005 && (int64_t)v.bm * v.bn > (int64_t)tiles[best].bm * tiles[best].bn)) {
      best = i; best_t = t; best_c = c; best_m = m;
    }
  }
  if (best < 0) return TB_ERR_BAD_TILE;
  const TileInfo& v = tiles[best];
  std::memset(out, 0, sizeof(*out));
  out->block_m = v.bm; out->block_n = v.bn; out->block_k = v.bk;
  const int64_t tiles_m = cdiv(pr.m, v.bm), tiles_n = cdiv(pr.n, v.bn);
  const int64_t total = tiles_m * tiles_n;
  out->group_m = (int)std::min<int64_t>(8, tiles_m);
  out->num_xcds = hw.num_xcd;
  out->occupancy = variant_occupancy(v, hw);
  out->num_stages = v.stages;
  out->lds_bytes = v.lds_bytes;
  out->counters_per_xcd = ws_counters_per_xcd(total);
  out->sk_grid = streamk_grid_for(pr, hw, v);
  out->est_compute_us = best_c; out->est_memory_us = best_m; out->est_total_us = best_t;
  return TB_OK;
}

}  // namespace tb
