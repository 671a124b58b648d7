// Host-only: analytical tile selector.
#pragma once
#include <stdint.h>
#include "../../include/tritonblas_amd.h"

namespace tb {

struct TileInfo {
  int dt, bm, bn, bk, threads, lds_bytes, minb, fast, stages;
};

void default_hw(tb_hw* hw);
int streamk_grid(int64_t total_tiles, int64_t k_iters, int slots, int n_cu, double step_us, double fix_us, double xchg_us = 0.0);
// the Stream-K grid the model picks for one tile variant on a problem
int streamk_grid_for(const tb_problem& pr, const tb_hw& hw, const TileInfo& v);
int ws_counters_per_xcd(int64_t total_tiles);
// (tiles per XCD-local queue, tiles in the shared pool) of the hierarchical work-stealing mode
void hierarchical_split(int64_t total_tiles, int hw_cus, int num_xcds, int64_t* local_per_xcd, int64_t* global_tiles);
// whether the hand-scheduled 256x256 kernels are the faster ones for a K that is no even number of K steps
bool rest_of_k_pays(int64_t m, int64_t n, int64_t k, int bk, int c_bits, int n_cu);
bool even_k_pays(int64_t m, int64_t n, int64_t k, int bk, int type, int n_cu);     // ... that is one (type: a public element type)
int variant_occupancy(const TileInfo& v, const tb_hw& hw);
// How a launch goes over its tiles.  looped: workgroups that take tile after tile, from a caller's grid or the work-stealing queues, and not one workgroup to a
// tile.  block_k: tiles of this K step only (0: any).  queues: they come from the work-stealing queues.  workgroups: as many as the caller keeps the launch to (0: as
// many as the device holds).
struct TileUse {
  bool looped = false;
  int block_k = 0;
  bool queues = false;
  int workgroups = 0;
};
int select_tile(const tb_problem& pr, const tb_hw& hw, const TileInfo* tiles, int ntiles, tb_selection* out, TileUse use = {});
// 32x32 and 64x32 tiles of the 16- and 8-bit types
bool narrow_tile(const TileInfo& v);
// model time (us) of one tile variant on a problem, and of the streaming small-M kernel
double estimate_tile_us(const tb_problem& pr, const tb_hw& hw, const TileInfo& v, bool streamk, TileUse use = {});
// ... of a grouped launch whose row counts only the device knows (FP8; 0: no figures for this variant)
double estimate_grouped_us(const tb_problem& pr, const tb_hw& hw, const TileInfo& v);
double estimate_streaming_us(const tb_problem& pr, const tb_hw& hw, int cols);
double streaming_bound_us(const tb_problem& pr, const tb_hw& hw);   // ... and what it takes at most

}  // namespace tb
