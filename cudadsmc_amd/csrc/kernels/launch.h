// Host launch wrappers of the DSMC kernels (implemented in step.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "../common/dsmc_dev.h"

namespace dsmc_launch {

using dsmc_dev::InstDesc;

constexpr uint32_t kScanMaxTiles = 4096;  // scan of up to 4096*4096 entries

void mt_seed(uint32_t* state, const uint32_t* seeds, uint32_t n_streams, hipStream_t st);
void mt_generate(const uint32_t* a, const uint32_t* b, const uint32_t* c, const uint32_t* seeds, uint32_t n_streams,
                 uint32_t n_draws, uint32_t* out, hipStream_t st);
void cell_ids(const InstDesc& I, const float* x, const float* y, const float* z, uint32_t n, uint32_t* keys,
              hipStream_t st);
void keys_count(const InstDesc* d, uint32_t par, uint32_t n, hipStream_t st);
// Exclusive scan of in[0..n) into out[0..n] (out[n] = total); in is cleared,
// total_out (device) receives the total. scratch: kScanMaxTiles uint32.
int scan(uint32_t* in, uint32_t n, uint32_t* out, uint32_t* scratch, uint32_t* total_out, hipStream_t st);
// Step kernels take an array of descriptors (scan and list: n_inst of them,
// grid.y = instance; the others by a map of blocks).
//
// Scan of the step: cell offsets and the inflow numbers of the freestream
// faces. One launch for instances of up to kScanSmall cells, else two. With
// 65536 cells (16 blocks of 4096) a block reads at most 240 KB of counts
// again to find its offset, 480 KB where the stayers are counted apart, which
// takes less than the second launch; beyond that the reading grows with the
// square of the cells. 64x32x32 cells, us per step with one / two launches:
// 100k particles 44.7 / 51.1, 655k (tile queues, stayers apart) 89.8 / 95.5,
// 1.3M (likewise) 136.3 / 140.8.
constexpr uint32_t kScanSmall = 65536;
struct StepScan {
  uint32_t n_cell = 0, n_face = 0;  // blocks of 4096 cells and faces (largest instance)
  bool small = false;
  uint32_t words() const { return n_cell + n_face; }  // scratch per instance (uint32)
};
StepScan step_scan_plan(uint32_t max_cells, uint32_t max_faces);
void step_scan(const InstDesc* d, const StepScan& p, uint32_t* ts, hipStream_t st, uint32_t n_inst = 1);
// Scatter, clearing of the counts, and the face offsets. blocks: the sum of
// scatter_blocks over the instances; map: {instance, its block} of each block
// (null for one instance).
uint32_t scatter_blocks(const InstDesc& I);
void scatter(const InstDesc* d, uint32_t par, uint32_t blocks, const uint2* map, const StepScan& p, const uint32_t* ts,
             hipStream_t st);
// Stable sort operator: cell offsets (n_cells + 1) and the permutation of a
// stable sort by key (keys >= n_cells dropped, listed last). work:
// op_sort_work_words(n, n_cells) uint32. No allocation, no memset.
uint64_t op_sort_work_words(uint32_t n, uint32_t n_cells);
int op_sort(const uint32_t* keys, uint32_t n, uint32_t n_cells, uint32_t* perm, uint32_t* cell_start,
            uint32_t* work, hipStream_t st);
// The tile kernel of instances with (narrow) or without tile_narrow: blocks =
// the sum of their n_tile_wg, map as for the scatter.
void tile(uint32_t mode, bool narrow, const InstDesc* d, uint32_t par, uint32_t flags, uint32_t blocks,
          const uint2* map, hipStream_t st);
// PHYSICS: the wall pass over the particles the tile kernel deferred (opar =
// the buffer it wrote) and the inflow; blocks and map as for the scatter.
// Before it, instances that are not wall_direct compact the deferred
// particles (`grid` workgroups per instance).
uint32_t wall_blocks(const InstDesc& I);
void defer_list(const InstDesc* d, uint32_t grid, hipStream_t st, uint32_t n_inst = 1);
void walls(const InstDesc* d, uint32_t opar, uint32_t flags, uint32_t blocks, const uint2* map, hipStream_t st);
// For host reads: folds the wall sums of the last step into wall_acc and sums
// the collision counters (2 * kAccSlots values, see k_totals).
void totals(const InstDesc* d, uint32_t n_acc, long long* out, hipStream_t st);
// n, u, v, w, T of the samples as float [5][ncells].
void fields(const InstDesc* d, uint32_t mode, uint32_t ncells, double samples, double kb, float* out, hipStream_t st);
void load_reference(const InstDesc* d, uint32_t par, uint32_t ppc, uint32_t n_threads, float sux, float suy,
                    float suz, float temp, hipStream_t st);
void move_zero(const InstDesc* d, uint32_t par, uint32_t n, hipStream_t st);
void load_count(const InstDesc* d, uint32_t n_streams, const float* fn, hipStream_t st);
void load_generate(const InstDesc* d, uint32_t par, uint32_t n_streams, const float* fu, const float* fv,
                   const float* fw, const float* fT, hipStream_t st);
void sample_cells(const InstDesc* d, uint32_t par, uint32_t mode, uint32_t ncells, hipStream_t st);
void validate(const InstDesc* d, uint32_t par, uint32_t n, uint32_t* bad, hipStream_t st);

enum TileFlags : uint32_t { kFlagSample = 1u, kFlagKeepPerm = 2u, kFlagHits = 4u };

}  // namespace dsmc_launch
