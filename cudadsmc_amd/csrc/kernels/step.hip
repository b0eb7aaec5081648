// HIP kernels of the DSMC step for gfx950 (CDNA4, wave64).
//
// Step = scan(count) -> scatter -> tile [-> walls and inject], replacing the
// reference's CalculateCellIDs -> thrust::sort_by_key -> cudaMemset ->
// FindCellBoundaries -> ComputeBird -> IntegrateAndProcessCollisions ->
// SampleCellStatistics sequence (include/gpu_dsmc.inl:221-274).
//
//  * Keys of the next step are computed by the move itself and counted per
//    cell, so the "sort" is a counting sort: an exclusive scan of the counts
//    gives the cell offsets (cellStartEnd of FindCellBoundariesDev,
//    dsmc_kernel.cu:1734-1787) and the scatter places each particle in its
//    cell's segment.
//  * The tile kernel owns a tile of consecutive cells: it restores the stable
//    order inside each cell segment (ascending storage index, i.e. the
//    permutation of a stable sort_by_key, dsmc_kernel.cu:2048), gathers the
//    particles (the REORDER gather, :1777-1786), runs the NTC out of LDS (one
//    lane per cell in REFERENCE mode, :1002-1089, rounds of disjoint pairs
//    in PHYSICS mode), moves each particle with walls and box faces
//    (:1596-1657), writes the next key and samples per cell (:856-890).
//  * RNG: PHYSICS draws are counter-based (Philox keyed by cell, slot and
//    step), so no result depends on which wave takes a tile.
//    REFERENCE mode keeps the reference's layout: cell c collides with
//    stream c and loading thread t draws from stream t.
#include <hip/hip_runtime.h>

#include "launch.h"
#include "physics.h"

using namespace dsmc_dev;

namespace {

constexpr uint32_t kScanThreads = 256;
constexpr uint32_t kScanItems = 16;
constexpr uint32_t kScanTile = kScanThreads * kScanItems;  // 4096

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Between phases of one wave: its own LDS and memory operations are in order,
// only the compiler has to keep them so.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ void mt_load(const InstDesc& I, uint32_t s, Mt& m) {
  const gptr<uint32_t> st = gmem(I.mt_state);
#pragma unroll
  for (int w = 0; w < kMtN; ++w) m.st[w] = st[(uint32_t)w * I.n_streams + s];
  m.a = gmem(I.mt_a)[s];
  m.b = gmem(I.mt_b)[s];
  m.c = gmem(I.mt_c)[s];
}

__device__ __forceinline__ void mt_store(const InstDesc& I, uint32_t s, const Mt& m) {
#pragma unroll
  for (int w = 0; w < kMtN; ++w) gmem(I.mt_state)[(uint32_t)w * I.n_streams + s] = m.st[w];
}

// Wave-aggregated atomicAdd(&cnt[key], 1) for keys of consecutive lanes,
// returning each lane's count before its own increment: one atomic per run
// of equal keys, whose lanes take consecutive values. Invalid keys are
// skipped (their result is meaningless). Split in two so that a caller can
// issue the atomics of several rounds before waiting for any: count_issue
// returns the run head's old count (0 elsewhere) and the wave's run heads,
// count_finish the lane's value.
__device__ __forceinline__ uint32_t count_issue(gptr<uint32_t> cnt, uint32_t key, uint64_t& heads) {
  const uint32_t lane = lane_id();
  const uint32_t prev = __shfl_up(key, 1);
  const bool head = (lane == 0) || (key != prev);
  heads = __ballot(head);
  uint32_t base = 0;
  if (head && key != kInvalidKey) {
    const uint64_t below_incl = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
    const uint64_t above = heads & ~below_incl;
    const uint32_t next = above ? (uint32_t)__ffsll((unsigned long long)above) - 1u : 64u;
    base = gatomic_add(gelem(cnt, key), next - lane);
  }
  return base;
}

__device__ __forceinline__ uint32_t count_finish(uint32_t base, uint64_t heads) {
  const uint32_t lane = lane_id();
  const uint64_t below_incl = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
  const uint32_t hl = 63u - (uint32_t)__clzll((long long)(heads & below_incl));
  return __shfl(base, (int)hl) + (lane - hl);
}

// Wave-aggregated atomicAdd(&cnt[key], 1) for keys of consecutive lanes:
// one atomic per run of equal keys. Invalid keys are skipped.
__device__ __forceinline__ void count_keys(gptr<uint32_t> cnt, uint32_t key) {
  uint32_t lane = lane_id();
  uint32_t prev = __shfl_up(key, 1);
  bool head = (lane == 0) || (key != prev);
  uint64_t heads = __ballot(head);
  if (head && key != kInvalidKey) {
    uint64_t above = heads & ~((2ull << lane) - 1ull);
    if (lane == 63) above = 0;
    uint32_t next = above ? (uint32_t)__ffsll((unsigned long long)above) - 1u : 64u;
    gatomic_add(gelem(cnt, key), next - lane);
  }
}

}  // namespace

// Work of a block in a launch whose instances need different numbers of
// blocks: {instance, its block}, read from the batch's map (a solver on its
// own has no map). A grid of the largest instance's size for each would be
// mostly blocks that exit (an ensemble of 10k to 500k particles: 213k blocks
// of the scatter, 100 of 150 us).
__device__ __forceinline__ uint2 block_of(const uint2* map) {
  return map ? gload(gmem(map) + blockIdx.x) : make_uint2(0u, blockIdx.x);
}

// ======================================================================= RNG
// InitMersenneTwistersDev (dsmc_kernel.cu:548-562): seed every stream.
__global__ void k_mt_seed(uint32_t* state, const uint32_t* seeds, uint32_t n_streams) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_streams) return;
  Mt m;
  mt_seed(m, seeds[s]);
#pragma unroll
  for (int w = 0; w < kMtN; ++w) state[(uint32_t)w * n_streams + s] = m.st[w];
  state[(uint32_t)kMtN * n_streams + s] = 0u;
}

// Stream outputs for the RNG parity tests (GenerateRandomSamplesUint4,
// mtwister.cu:207-230, with one stream per thread).
__global__ void k_mt_generate(const uint32_t* a, const uint32_t* b, const uint32_t* c, const uint32_t* seeds,
                              uint32_t n_streams, uint32_t n_draws, uint32_t* out) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_streams) return;
  Mt m;
  m.a = a[s];
  m.b = b[s];
  m.c = c[s];
  mt_seed(m, seeds[s]);
  for (uint32_t d = 0; d < n_draws; ++d) out[(size_t)d * n_streams + s] = mt_next(m);
}

// ====================================================================== keys
// CalculateCellIDsDev (dsmc_kernel.cu:1712-1724) on SoA positions.
__global__ void k_cell_ids(InstDesc I, const float* x, const float* y, const float* z, uint32_t n, uint32_t* keys) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  keys[i] = cell_key(I, x[i], y[i], z[i]);
}

// Keys and counts of a freshly loaded state (storage order, buffer `par`).
__global__ void k_keys_count(const InstDesc* __restrict__ Ip, uint32_t par, uint32_t n) {
  const InstDesc& I = *Ip;
  uint32_t base = blockIdx.x * blockDim.x;
  uint32_t i = base + threadIdx.x;
  uint32_t key = kInvalidKey;
  if (i < n) {
    const float x = I.px[par][i], y = I.py[par][i], z = I.pz[par][i];
    key = I.mode == kModePhysics ? cell_key_phys(I, x, y, z) : cell_key(I, x, y, z);
    I.key[par][i] = key;
  }
  count_keys(gmem(I.count), key);
}

// ====================================================================== scan
// Exclusive scan of uint32 counts in three passes (tile sums, scan of the
// tile sums, tile scan); clears the counts and stores the total.
__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(const uint32_t* in, uint32_t n, uint32_t* tile_sums) {
  __shared__ uint32_t red[kScanThreads / 64];
  uint32_t base = blockIdx.x * kScanTile;
  uint32_t sum = 0;
  if (base + kScanTile <= n && (reinterpret_cast<uintptr_t>(in) & 15u) == 0u) {
    // a whole tile of a 16-byte aligned array: vector loads, consecutive lanes on consecutive vectors
    const gptr<const uint4> src = gmem<const uint4>(reinterpret_cast<const uint4*>(in + base));
#pragma unroll
    for (uint32_t k = 0; k < kScanItems / 4u; ++k) {
      const uint4 q = gload(src + k * kScanThreads + threadIdx.x);
      sum += (q.x + q.y) + (q.z + q.w);
    }
  } else {
#pragma unroll
    for (uint32_t k = 0; k < kScanItems; ++k) {
      uint32_t i = base + k * kScanThreads + threadIdx.x;
      if (i < n) sum += in[i];
    }
  }
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off);
  if (lane_id() == 0) red[threadIdx.x / 64] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (uint32_t w = 0; w < kScanThreads / 64; ++w) t += red[w];
    tile_sums[blockIdx.x] = t;
  }
}

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* total, uint32_t* sh) {
  // sh: kScanThreads/64 + 1 words
  uint32_t lane = lane_id(), wid = threadIdx.x / 64;
  uint32_t x = v;
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(x, off);
    if (lane >= (uint32_t)off) x += y;
  }
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (uint32_t w = 0; w < kScanThreads / 64; ++w) {
      uint32_t t = sh[w];
      sh[w] = run;
      run += t;
    }
    sh[kScanThreads / 64] = run;
  }
  __syncthreads();
  uint32_t r = sh[wid] + x - v;
  *total = sh[kScanThreads / 64];
  __syncthreads();
  return r;
}

// Scans tile_sums in place (n_tiles <= kScanTile) and writes the grand total.
__global__ void __launch_bounds__(kScanThreads) k_scan_tiles(uint32_t* tile_sums, uint32_t n_tiles, uint32_t* total_out) {
  __shared__ uint32_t sh[kScanThreads / 64 + 1];
  uint32_t v[kScanItems];
  uint32_t local = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    uint32_t i = threadIdx.x * kScanItems + k;
    v[k] = i < n_tiles ? tile_sums[i] : 0u;
    local += v[k];
  }
  uint32_t total;
  uint32_t off = block_exclusive_scan(local, &total, sh);
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    uint32_t i = threadIdx.x * kScanItems + k;
    if (i < n_tiles) tile_sums[i] = off;
    off += v[k];
  }
  if (threadIdx.x == 0) *total_out = total;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_apply(uint32_t* in, uint32_t n, const uint32_t* tile_sums,
                                                            uint32_t* out, const uint32_t* total) {
  __shared__ uint32_t sh[kScanThreads / 64 + 1];
  uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  uint32_t v[kScanItems];
  uint32_t local = 0;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    uint32_t i = base + k;
    v[k] = i < n ? in[i] : 0u;
    local += v[k];
  }
  uint32_t tot;
  uint32_t off = block_exclusive_scan(local, &tot, sh) + tile_sums[blockIdx.x];
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    uint32_t i = base + k;
    if (i < n) {
      out[i] = off;
      in[i] = 0u;
    }
    off += v[k];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = *total;
}

// Scan of the step over a batch of instances (grid.y = instance): the cell
// counts become cell_start and the scatter's cursors, and the freestream
// faces' inflow of the step is counted beside it (offsets: k_scatter). The
// counts stay: the scatter clears them. Two forms:
//
//  * k_scan_small (instances of at most kScanSmall cells): one launch. Each
//    block of 4096 cells sums the counts before it by itself, so no block
//    waits for another; the last one reads 15 blocks of 16 KB from L2 (of
//    32 KB where the stayers are counted apart).
//  * k_scan_reduce + k_scan_apply_step: block sums first, then each block adds
//    up the sums before it (at most 4096 words).
//
// Blocks: [0, n_cell) cell tiles, [n_cell, n_cell + n_face) face tiles, and
// in the launch that ends the scan one block that folds the wall sums of the
// step before. ts: the batch's tile sums, `stride` words per instance, cells
// first. ctr[4] still holds the step before (the scatter advances it).
constexpr uint32_t kScanSmall = dsmc_launch::kScanSmall;

// Block-wide exclusive scan of v and sum of w over NW waves; sh: 2 NW words.
template <uint32_t NW>
__device__ __forceinline__ uint32_t block_scan_sum(uint32_t v, uint32_t w, uint32_t& total, uint32_t& wsum,
                                                   uint32_t* sh) {
  const uint32_t lane = lane_id(), wid = threadIdx.x / 64u;
  uint32_t x = v;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off);
    if (lane >= (uint32_t)off) x += y;
  }
  for (int off = 32; off > 0; off >>= 1) w += __shfl_xor(w, off);
  if (lane == 63) {
    sh[wid] = x;
    sh[NW + wid] = w;
  }
  __syncthreads();
  uint32_t before = 0u;
  total = wsum = 0u;
#pragma unroll
  for (uint32_t k = 0; k < NW; ++k) {
    before += k < wid ? sh[k] : 0u;
    total += sh[k];
    wsum += sh[NW + k];
  }
  return before + x - v;
}

__device__ __forceinline__ uint32_t face_of(const InstDesc& I, uint32_t g) {
  uint32_t f = 0;
  while (f < 5 && g >= I.face_off[f + 1]) ++f;
  return f;
}

// Injection draws Philox4x32-10 under key (seed, kInjectKey1), so no stream
// state moves and every particle is independent: the count of face cell g
// draws counter (g, step, 0, 0); particle j of g draws (g, step, 1 + j, b)
// for its b-th rejection block (two tries per block) and (g, step, 1 + j,
// 2^31 + k) for its other variates.
constexpr uint32_t kInjectKey1 = 0xBB67AE85u;

__device__ __forceinline__ uint32_t inject_number(const InstDesc& I, uint32_t g, uint32_t stepno) {
  const dsmc_rng::U32x4 c = {{g, stepno, 0u, 0u}};
  const dsmc_rng::U32x4 r = dsmc_rng::philox4x32_10(c, I.wall_key[0], kInjectKey1);
  return dm_f2u_sat(I.inj_lambda[face_of(I, g)] + dsmc_rng::px_unit(r.v[0]));
}

// Inflow numbers of face tile f (kScanTile faces) and their sum; NT threads.
template <uint32_t NT>
__device__ __forceinline__ void count_faces(const InstDesc& I, uint32_t f, uint32_t* ts, uint32_t* sh) {
  const uint32_t stepno = I.ctr[4] + 1u;
  uint32_t sum = 0u;
  for (uint32_t k = threadIdx.x; k < kScanTile; k += NT) {
    const uint32_t g = f * kScanTile + k;
    if (g >= I.n_face_cells) break;
    const uint32_t c = inject_number(I, g, stepno);
    I.face_count[g] = c;
    sum += c;
  }
  uint32_t total, wsum;
  block_scan_sum<NT / 64>(0u, sum, total, wsum, sh);
  if (threadIdx.x == 0) ts[f] = wsum;
}

// The wall pass's per-workgroup sums of one step into the running totals:
// exact 64-bit integer sums (any order gives the same value), converted once
// per step, and cleared, so that a fold without a step between adds nothing.
// NT threads; red: 4 words per wave.
template <uint32_t NT>
__device__ __forceinline__ void fold_walls(const InstDesc& I, long long* red) {
  const uint32_t tid = threadIdx.x, lane = lane_id(), wid = tid / 64u;
  const gptr<long long> part = gmem(I.wall_part);
  long long v[4] = {0, 0, 0, 0};
  for (uint32_t w = tid; w < I.n_wall_part; w += NT)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] += part[w * 4u + k];
      part[w * 4u + k] = 0;
    }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    long long x = v[k];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off);
    if (lane == 0) red[wid * 4 + k] = x;
  }
  __syncthreads();
  if (tid < 4) {
    long long t = 0;
    for (uint32_t q = 0; q < NT / 64; ++q) t += red[q * 4 + tid];
    gmem(I.wall_acc)[tid] += (double)t * I.wall_unit[tid < 3 ? 0 : 1];
  }
}

// What the block with the last cells leaves for the step.
__device__ __forceinline__ void scan_done(const InstDesc& I, uint32_t total) {
  I.cell_start[I.ncells] = total;
  I.ctr[1] = total;
  I.ctr[5] = 0u;  // deferred particles of the step
  for (uint32_t q = 0; q < 8u; ++q) I.ctr[kTileQueueCtr + q] = 0u;  // the tile kernel's queues
}

// Offsets and cursors of N consecutive cells from base: v their counts, off
// the first one's offset. Whole groups move as 16-byte vectors (the engine's
// arrays are 256-byte aligned). Instances without tile-local ranking start
// their cursors at the offsets.
template <uint32_t N>
__device__ __forceinline__ void store_offsets(const InstDesc& I, uint32_t base, const uint32_t (&v)[N], uint32_t off) {
  const uint32_t n = I.ncells;
  if (base + N <= n) {
    uint4 l[N / 4u];
#pragma unroll
    for (uint32_t k = 0; k < N / 4u; ++k)
      l[k] = I.tile_dyn ? gload(gmem<const uint4>(reinterpret_cast<const uint4*>(I.local_cnt + base)) + k)
                        : make_uint4(0u, 0u, 0u, 0u);
    const gptr<uint4> dst = gmem(reinterpret_cast<uint4*>(I.cell_start + base));
    const gptr<uint4> cur = gmem(reinterpret_cast<uint4*>(I.cursor + base));
#pragma unroll
    for (uint32_t k = 0; k < N / 4u; ++k) {
      const uint32_t o0 = off, o1 = o0 + v[4 * k], o2 = o1 + v[4 * k + 1], o3 = o2 + v[4 * k + 2];
      off = o3 + v[4 * k + 3];
      gstore(dst + k, make_uint4(o0, o1, o2, o3));
      gstore(cur + k, make_uint4(o0 + l[k].x, o1 + l[k].y, o2 + l[k].z, o3 + l[k].w));
    }
    return;
  }
  for (uint32_t k = 0; k < N && base + k < n; ++k) {
    I.cell_start[base + k] = off;
    I.cursor[base + k] = off + (I.tile_dyn ? I.local_cnt[base + k] : 0u);
    off += v[k];
  }
}

// Whether the particles that stay in their tile are counted in local_cnt
// alone, and `count` holds the others: asked by the tile kernel, which counts,
// and by the scan, which adds them up. It saves the tile kernel most of its
// global atomics (33.5 million particles, 16 per cell: 695 -> 678 us, of which the scan takes 3 more).
// REFERENCE tiles count all of them in `count` (its benchmark case: 176 us,
// apart 187).
template <uint32_t MODE>
__device__ __forceinline__ bool stayers_apart(const InstDesc& I) {
  return MODE == kModePhysics && I.tile_dyn;
}

__device__ __forceinline__ bool add_stayers(const InstDesc& I) {
  return I.mode == kModePhysics && stayers_apart<kModePhysics>(I);
}

// Particles of a cell.
__device__ __forceinline__ uint32_t cell_count(const InstDesc& I, uint32_t c) {
  return I.count[c] + (add_stayers(I) ? I.local_cnt[c] : 0u);
}
__device__ __forceinline__ uint4 cell_counts4(const InstDesc& I, uint32_t q) {  // cells [4 q, 4 q + 4)
  uint4 v = gload(gmem<const uint4>(reinterpret_cast<const uint4*>(I.count)) + q);
  if (add_stayers(I)) {
    const uint4 l = gload(gmem<const uint4>(reinterpret_cast<const uint4*>(I.local_cnt)) + q);
    v = make_uint4(v.x + l.x, v.y + l.y, v.z + l.z, v.w + l.w);
  }
  return v;
}

template <uint32_t N>
__device__ __forceinline__ void load_counts(const InstDesc& I, uint32_t base, uint32_t (&v)[N]) {
  if (base + N <= I.ncells) {
#pragma unroll
    for (uint32_t k = 0; k < N / 4u; ++k) {
      const uint4 q = cell_counts4(I, base / 4u + k);
      v[4 * k] = q.x;
      v[4 * k + 1] = q.y;
      v[4 * k + 2] = q.z;
      v[4 * k + 3] = q.w;
    }
  } else {
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) v[k] = base + k < I.ncells ? cell_count(I, base + k) : 0u;
  }
}

constexpr uint32_t kSmallThreads = 1024;

__global__ void __launch_bounds__(kSmallThreads) k_scan_small(const InstDesc* __restrict__ D, uint32_t n_cell,
                                                              uint32_t n_face, uint32_t* ts, uint32_t stride) {
  const InstDesc& I = D[blockIdx.y];
  __shared__ __align__(8) uint32_t sh[4 * 2 * kSmallThreads / 64];
  const uint32_t b = blockIdx.x, tid = threadIdx.x;
  if (b >= n_cell + n_face) {
    if (I.defer_bits) fold_walls<kSmallThreads>(I, reinterpret_cast<long long*>(sh));
    return;
  }
  if (b >= n_cell) {
    if ((b - n_cell) * kScanTile < I.n_face_cells)
      count_faces<kSmallThreads>(I, b - n_cell, ts + blockIdx.y * stride + n_cell, sh);
    return;
  }
  const uint32_t n = I.ncells;
  if (b * kScanTile >= n) return;
  // the counts of the tiles before this one, all of whose cells exist
  uint32_t pre = 0u;
#pragma unroll 5
  for (uint32_t k = 0; k < b; ++k) {
    const uint4 q = cell_counts4(I, k * kSmallThreads + tid);
    pre += (q.x + q.y) + (q.z + q.w);
  }
  const uint32_t base = b * kScanTile + tid * 4u;
  uint32_t v[4];
  load_counts<4>(I, base, v);
  uint32_t total, before;
  const uint32_t off = block_scan_sum<kSmallThreads / 64>((v[0] + v[1]) + (v[2] + v[3]), pre, total, before, sh);
  store_offsets<4>(I, base, v, before + off);
  if ((b + 1u) * kScanTile >= n && tid == 0) scan_done(I, before + total);
}

__global__ void __launch_bounds__(kScanThreads) k_scan_reduce_step(const InstDesc* __restrict__ D, uint32_t n_cell,
                                                                  uint32_t* ts, uint32_t stride) {
  const InstDesc& I = D[blockIdx.y];
  __shared__ uint32_t sh[2 * kScanThreads / 64];
  const uint32_t b = blockIdx.x;
  uint32_t* const t = ts + blockIdx.y * stride;
  if (b >= n_cell) {
    if ((b - n_cell) * kScanTile < I.n_face_cells) count_faces<kScanThreads>(I, b - n_cell, t + n_cell, sh);
    return;
  }
  const uint32_t n = I.ncells, base = b * kScanTile;
  if (base >= n) return;
  uint32_t sum = 0u;
  if (base + kScanTile <= n) {  // consecutive lanes on consecutive vectors
#pragma unroll
    for (uint32_t k = 0; k < kScanItems / 4u; ++k) {
      const uint4 q = cell_counts4(I, base / 4u + k * kScanThreads + threadIdx.x);
      sum += (q.x + q.y) + (q.z + q.w);
    }
  } else {
    for (uint32_t i = base + threadIdx.x; i < n; i += kScanThreads) sum += cell_count(I, i);
  }
  uint32_t total, wsum;
  block_scan_sum<kScanThreads / 64>(0u, sum, total, wsum, sh);
  if (threadIdx.x == 0) t[b] = wsum;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_apply_step(const InstDesc* __restrict__ D, uint32_t n_cell,
                                                                 const uint32_t* ts, uint32_t stride) {
  const InstDesc& I = D[blockIdx.y];
  __shared__ __align__(8) uint32_t sh[4 * 2 * kScanThreads / 64];
  const uint32_t b = blockIdx.x;
  if (b >= n_cell) {
    if (I.defer_bits) fold_walls<kScanThreads>(I, reinterpret_cast<long long*>(sh));
    return;
  }
  if (b * kScanTile >= I.ncells) return;
  const gptr<const uint32_t> t = gmem<const uint32_t>(ts + blockIdx.y * stride);
  uint32_t pre = 0u;
  for (uint32_t k = threadIdx.x; k < b; k += kScanThreads) pre += t[k];
  // each thread scans kScanItems consecutive cells
  const uint32_t base = b * kScanTile + threadIdx.x * kScanItems;
  uint32_t v[kScanItems];
  load_counts<kScanItems>(I, base, v);
  uint32_t local = 0u;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) local += v[k];
  uint32_t total, before;
  const uint32_t off = block_scan_sum<kScanThreads / 64>(local, pre, total, before, sh);
  store_offsets<kScanItems>(I, base, v, before + off);
  if ((b + 1u) * kScanTile >= I.ncells && threadIdx.x == 0) scan_done(I, before + total);
}

// Face tile f: inflow numbers to offsets, in place (total in face_count[n]).
__device__ __forceinline__ void offset_faces(const InstDesc& I, uint32_t f, const uint32_t* ts, uint32_t* sh) {
  const uint32_t n = I.n_face_cells;
  if (f * kScanTile >= n) return;
  uint32_t pre = 0u;
  for (uint32_t k = threadIdx.x; k < f; k += kScanThreads) pre += ts[k];
  const uint32_t base = f * kScanTile + threadIdx.x * kScanItems;
  uint32_t v[kScanItems], local = 0u;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    v[k] = base + k < n ? I.face_count[base + k] : 0u;
    local += v[k];
  }
  uint32_t total, before;
  uint32_t off = block_scan_sum<kScanThreads / 64>(local, pre, total, before, sh) + before;
#pragma unroll
  for (uint32_t k = 0; k < kScanItems; ++k) {
    if (base + k < n) I.face_count[base + k] = off;
    off += v[k];
  }
  if ((f + 1u) * kScanTile >= n && threadIdx.x == 0) I.face_count[n] = before + total;
}

// =================================================================== scatter
// Places every stored particle i in the sorted order: perm[dst] = i, dst in
// its cell's segment. The tile kernel stored the particles of each tile in
// one run of slots (tile_p0) and counted per cell how many of them stayed
// in the tile's own cells (local_cnt); the scan set cursor = cell_start +
// local_cnt. A workgroup takes up to kScatterSpan consecutive cells (whole
// tiles) and the slots of their tiles: the particles that stayed in their
// tile are ranked with LDS atomics into the first local_cnt places of their
// cells; the others (they left their tile, went through the wall pass, or
// were injected after the tile-ordered slots) take the places from the
// cursor on, with one wave-aggregated global atomic per run of equal keys
// and the atomics of kScatterRounds rounds of 256 slots in flight together
// (one atomic per particle is far slower: runs are common, e.g. a cell's
// particles after the wall pass).
// The order within a cell is the order in which the atomics landed; the
// tile kernel sorts each cell's segment by storage index.
constexpr uint32_t kScatterRounds = 4;
constexpr uint32_t kScatterSpan = 1024;  // cells per workgroup pass (a multiple of every tile size)

//
// Beside that the launch clears the counts for the next step (the scan has
// read them), advances the step number and, in the blocks after the instance's n_scatter_wg,
// turns the face tiles' inflow numbers into offsets.
__global__ void __launch_bounds__(256) k_scatter(const InstDesc* __restrict__ Ip, uint32_t par, const uint2* map,
                                                 const uint32_t* face_ts, uint32_t stride) {
  const uint2 blk = block_of(map);
  const InstDesc& I = Ip[blk.x];
  const uint32_t bx = blk.y, grid = I.n_scatter_wg;
  __shared__ uint32_t s_cnt[kScatterSpan];
  __shared__ uint32_t s_tp[kScatterSpan / 32u + 1u];
  const uint32_t tid = threadIdx.x;
  if (bx >= grid) {
    offset_faces(I, bx - grid, face_ts + blk.x * stride, s_cnt);
    return;
  }
  if (bx == 0 && tid == 0) I.ctr[4] += 1u;  // step number (counter of the draws)
  {
    const gptr<uint4> cnt4 = gmem(reinterpret_cast<uint4*>(I.count));
    const uint32_t n4 = I.ncells / 4u;
    for (uint32_t i = bx * 256u + tid; i < n4; i += grid * 256u) gstore(cnt4 + i, make_uint4(0u, 0u, 0u, 0u));
    if (bx == 0 && tid < I.ncells % 4u) I.count[4u * n4 + tid] = 0u;
  }
  const uint32_t n = I.ctr[0];
  const gptr<const uint32_t> keys = gmem<const uint32_t>(I.key[par]);
  const gptr<const uint32_t> start = gmem<const uint32_t>(I.cell_start);
  const gptr<const uint32_t> tp0 = gmem<const uint32_t>(I.tile_p0);
  const gptr<uint32_t> perm = gmem(I.perm);
  const gptr<uint32_t> cursor = gmem(I.cursor);
  const uint32_t cap = I.cap, tile_cells = I.tile_cells;
  // end of the tile-ordered slots; instances with small tiles place every
  // particle through the cursors (their tile kernel counts none as stayed)
  const uint32_t S = I.tile_dyn ? min(tp0[I.ntiles], n) : 0u;
  // tiles per pass: up to kScatterSpan cells, fewer when the instance has
  // too few tiles to give every workgroup a pass
  const uint32_t K = max(1u, min(kScatterSpan / tile_cells, I.ntiles / grid));
  // Slots of the pass's tiles [t0, t0 + K) (runs starting at s_tp[]), in
  // rounds of 256 slots from q0 (below q1). Each lane keeps the tile of its
  // last slot in t (its slots only grow). A particle that stayed in its
  // tile takes the next LDS place of its cell (s_cnt, seeded with the cell
  // starts); any other takes its cell's cursor, with one wave-aggregated
  // atomic per run of equal keys (particles of one cell that leave together,
  // or a cell's particles after the wall pass), the atomics of
  // kScatterRounds rounds issued before any result is used. kk holds the
  // keys of slots q0...; the keys of the next kScatterRounds rounds are
  // requested before these atomics, so both latencies overlap.
  auto load_keys = [&](uint32_t q0, uint32_t q1, uint32_t (&kk)[kScatterRounds]) {
#pragma unroll
    for (uint32_t r = 0; r < kScatterRounds; ++r) {
      const uint32_t i = q0 + r * 256u + tid;
      kk[r] = i < q1 ? *gelem(keys, i) : kInvalidKey;
    }
  };
  auto place_tiled = [&](uint32_t q0, uint32_t q1, uint32_t c0, uint32_t K, uint32_t& t,
                         uint32_t (&kk)[kScatterRounds]) {
    uint32_t kc[kScatterRounds], loc[kScatterRounds], g[kScatterRounds], base[kScatterRounds], lds[kScatterRounds];
    uint64_t heads[kScatterRounds];
#pragma unroll
    for (uint32_t r = 0; r < kScatterRounds; ++r) kc[r] = kk[r];
    if (q0 + 256u * kScatterRounds < q1) load_keys(q0 + 256u * kScatterRounds, q1, kk);  // uniform
#pragma unroll
    for (uint32_t r = 0; r < kScatterRounds; ++r) {
      const uint32_t i = q0 + r * 256u + tid;
      const uint32_t key = kc[r];
      while (t + 1u < K && s_tp[t + 1u] <= i) ++t;
      const uint32_t rel = key - c0;
      const bool stayed = rel - t * tile_cells < tile_cells;  // its cell lies in the tile that holds its slot
      loc[r] = stayed ? rel : kInvalidKey;
      g[r] = stayed ? kInvalidKey : key_cell(key);
      base[r] = count_issue(cursor, g[r], heads[r]);
      if (stayed) lds[r] = atomicAdd(&s_cnt[rel], 1u);
    }
#pragma unroll
    for (uint32_t r = 0; r < kScatterRounds; ++r) {
      const uint32_t i = q0 + r * 256u + tid;
      uint32_t dst = count_finish(base[r], heads[r]);
      if (loc[r] != kInvalidKey) dst = lds[r];
      if ((loc[r] != kInvalidKey || g[r] != kInvalidKey) && dst < cap) *gelem(perm, dst) = i;
    }
  };
  // slots after the tile-ordered ones (or all of them before the first
  // step): through the cursors, one wave-aggregated atomic per run of
  // equal keys
  auto place_rest = [&](uint32_t q0, uint32_t q1) {
    uint32_t key[kScatterRounds], base[kScatterRounds];
    uint64_t heads[kScatterRounds];
#pragma unroll
    for (uint32_t r = 0; r < kScatterRounds; ++r) {
      const uint32_t i = q0 + r * 256u + tid;
      key[r] = i < q1 ? key_cell(*gelem(keys, i)) : kInvalidKey;
      base[r] = count_issue(cursor, key[r], heads[r]);
    }
#pragma unroll
    for (uint32_t r = 0; r < kScatterRounds; ++r) {
      const uint32_t i = q0 + r * 256u + tid;
      const uint32_t dst = count_finish(base[r], heads[r]);
      if (key[r] != kInvalidKey && dst < cap) *gelem(perm, dst) = i;
    }
  };
  const uint32_t passes = S ? (I.ntiles + K - 1u) / K : 0u;
  for (uint32_t g = bx; g < passes; g += grid) {  // uniform over the workgroup
    const uint32_t t0 = g * K;
    const uint32_t c0 = t0 * I.tile_cells;
    for (uint32_t c = tid; c < K * tile_cells; c += 256u) s_cnt[c] = c0 + c < I.ncells ? start[c0 + c] : 0u;
    if (tid <= K) s_tp[tid] = t0 + tid <= I.ntiles ? min(tp0[t0 + tid], S) : S;
    __syncthreads();
    const uint32_t p0 = s_tp[0], p1 = max(s_tp[K], p0);
    uint32_t t = 0;
    uint32_t kk[kScatterRounds];
    if (p0 < p1) load_keys(p0, p1, kk);
    __builtin_amdgcn_s_waitcnt(0);  // the loop starts with no load pending, so its top waits for none
    for (uint32_t q0 = p0; q0 < p1; q0 += 256u * kScatterRounds) place_tiled(q0, p1, c0, K, t, kk);
    __syncthreads();  // s_cnt and s_tp are set again for the next pass
  }
  for (uint32_t q0 = S + bx * 256u * kScatterRounds; q0 < n; q0 += grid * 256u * kScatterRounds)
    place_rest(q0, n);
}

// ============================================================ sort operator
// Stable LSD radix sort of (key, storage index) pairs: the permutation of
// SortParticlesIndices' thrust::sort_by_key (dsmc_kernel.cu:2033-2051). Keys
// >= n_cells (dropped particles) sort as n_cells, after every valid key.
//
// A pass takes up to 10 bits (2^20 keys of 2^19 cells: two passes) in three
// launches: each block counts its keys' digits (table[digit * nblocks +
// block]), k_rs_scan turns each digit's row into offsets and leaves the row's
// total, and k_rs_scatter ranks its keys and moves them. Latency bounds it at
// this size, so a block has 16 waves, of which each ranks a run of consecutive
// keys by itself (peers of equal digit found with a ballot per bit, counts of
// the earlier rounds in LDS of its own), and the block sorts its keys in LDS
// first, so that its stores are runs. The cell offsets come from the sorted
// keys (k_rs_cells). 2^20 keys, 128x64x64 cells: 55 us; with 8 bits per
// pass, four waves per block and barriers in each of 16 rounds, a scan of three
// launches over the table, and offsets from atomic counts 128 us.
constexpr uint32_t kRsThreads = 1024, kRsWaves = kRsThreads / 64;
constexpr uint32_t kRsMaxBits = 10, kRsMaxDigits = 1u << kRsMaxBits;
constexpr uint32_t kRsCells = 1024;   // cells per block of k_rs_cells
constexpr uint32_t kRsStage = 4096;   // keys of them that it takes into LDS
static_assert(kRsMaxDigits <= kRsThreads, "a thread per digit");

__device__ __forceinline__ uint32_t rs_key(const uint32_t* keys, uint32_t i, uint32_t n_cells, bool raw) {
  const uint32_t k = keys[i];
  return raw ? (k < n_cells ? k : n_cells) : k;
}

// R: keys per thread
template <uint32_t R>
__global__ void __launch_bounds__(kRsThreads) k_rs_hist(const uint32_t* keys, uint32_t n, uint32_t n_cells,
                                                        uint32_t raw, uint32_t shift, uint32_t digits,
                                                        uint32_t nblocks, uint32_t* table) {
  __shared__ uint32_t s_h[kRsMaxDigits];
  const uint32_t tid = threadIdx.x, base = blockIdx.x * (kRsThreads * R);
  uint32_t k[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t i = base + r * kRsThreads + tid;
    k[r] = i < n ? rs_key(keys, i, n_cells, raw != 0u) : 0u;
  }
  s_h[tid] = 0u;
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < R; ++r)
    if (base + r * kRsThreads + tid < n) atomicAdd(&s_h[(k[r] >> shift) & (digits - 1u)], 1u);
  __syncthreads();
  if (tid < digits) table[(size_t)tid * nblocks + blockIdx.x] = s_h[tid];
}

// Block d: row d of the table to exclusive offsets, in place, its total to tot[d].
__global__ void __launch_bounds__(kScanThreads) k_rs_scan(uint32_t* table, uint32_t nblocks, uint32_t* tot) {
  __shared__ __align__(8) uint32_t sh[4 * 2 * kScanThreads / 64];
  uint32_t* row = table + (size_t)blockIdx.x * nblocks;
  uint32_t carry = 0u;
  for (uint32_t b0 = 0; b0 < nblocks; b0 += 4u * kScanThreads) {
    const uint32_t base = b0 + 4u * threadIdx.x;
    uint32_t v[4], sum = 0u;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      v[k] = base + k < nblocks ? row[base + k] : 0u;
      sum += v[k];
    }
    uint32_t total, none;
    uint32_t off = carry + block_scan_sum<kScanThreads / 64>(sum, 0u, total, none, sh);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      if (base + k < nblocks) row[base + k] = off;
      off += v[k];
    }
    carry += total;
    __syncthreads();  // sh is used again
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

template <uint32_t R>
__global__ void __launch_bounds__(kRsThreads) k_rs_scatter(const uint32_t* keys, const uint32_t* vals, uint32_t n,
                                                           uint32_t n_cells, uint32_t raw, uint32_t shift,
                                                           uint32_t bits, uint32_t nblocks, const uint32_t* table,
                                                           const uint32_t* tot, uint32_t* keys_out,
                                                           uint32_t* vals_out) {
  __shared__ uint16_t s_wc[kRsWaves][kRsMaxDigits];  // a wave's keys of each digit, then the earlier waves'
  __shared__ uint32_t s_k[kRsThreads * R], s_v[kRsThreads * R];
  __shared__ uint32_t s_first[kRsMaxDigits];  // first place of the digit in the block
  __shared__ uint32_t s_dst[kRsMaxDigits];    // its first place in the result, less s_first
  __shared__ uint32_t s_part[2][kRsWaves];
  const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / 64u;
  const uint32_t base = blockIdx.x * (kRsThreads * R), digits = 1u << bits, mask = digits - 1u;
  uint32_t k[R], v[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t i = base + w * (64u * R) + r * 64u + lane;
    k[r] = i < n ? rs_key(keys, i, n_cells, raw != 0u) : 0u;
    v[r] = i < n ? (vals ? vals[i] : i) : 0u;
  }
  const uint32_t g_tot = tid < digits ? tot[tid] : 0u;
  const uint32_t g_row = tid < digits ? table[(size_t)tid * nblocks + blockIdx.x] : 0u;
  for (uint32_t d = lane; d < digits; d += 64u) s_wc[w][d] = 0u;
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t rank[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const bool valid = base + w * (64u * R) + r * 64u + lane < n;
    const uint32_t d = (k[r] >> shift) & mask;
    uint64_t peers = __ballot(valid);
    for (uint32_t bit = 0; bit < bits; ++bit) {
      const bool one = (d >> bit) & 1u;
      const uint64_t m = __ballot(one);
      peers &= one ? m : ~m;
    }
    wave_sync();  // the round before has stored its counts
    const uint32_t at = (uint32_t)__popcll(peers & below), had = s_wc[w][d];
    wave_sync();
    if (valid && at == 0u) s_wc[w][d] = (uint16_t)(had + (uint32_t)__popcll(peers));
    rank[r] = had + at;
  }
  __syncthreads();
  uint32_t cnt = 0u;
  if (tid < digits) {
#pragma unroll
    for (uint32_t q = 0; q < kRsWaves; ++q) {
      const uint32_t c = s_wc[q][tid];
      s_wc[q][tid] = (uint16_t)cnt;
      cnt += c;
    }
  }
  // exclusive scans over the digits, of the block's counts and of all keys'
  uint32_t x = cnt, y = g_tot;
#pragma unroll
  for (uint32_t o = 1; o < 64u; o <<= 1) {
    const uint32_t xo = __shfl_up(x, o), yo = __shfl_up(y, o);
    if (lane >= o) x += xo, y += yo;
  }
  if (lane == 63u) s_part[0][w] = x, s_part[1][w] = y;
  __syncthreads();
  uint32_t px = 0u, py = 0u;
#pragma unroll
  for (uint32_t q = 0; q < kRsWaves; ++q) {
    px += q < w ? s_part[0][q] : 0u;
    py += q < w ? s_part[1][q] : 0u;
  }
  if (tid < digits) {
    const uint32_t first = px + x - cnt;
    s_first[tid] = first;
    s_dst[tid] = py + y - g_tot + g_row - first;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    if (base + w * (64u * R) + r * 64u + lane >= n) continue;
    const uint32_t d = (k[r] >> shift) & mask;
    const uint32_t at = s_first[d] + s_wc[w][d] + rank[r];
    s_k[at] = k[r];
    s_v[at] = v[r];
  }
  __syncthreads();
  const uint32_t m = min(n - base, kRsThreads * R);
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) {
    const uint32_t i = r * kRsThreads + tid;
    if (i >= m) continue;
    const uint32_t kk = s_k[i], dst = s_dst[(kk >> shift) & mask] + i;
    keys_out[dst] = kk;
    vals_out[dst] = s_v[i];
  }
}

// First place in the sorted keys whose key is not below v, found by a wave in
// steps of 64 places (2^20 keys: four rounds of loads).
__device__ __forceinline__ uint32_t rs_lower_bound(const uint32_t* keys, uint32_t n, uint32_t v) {
  uint32_t lo = 0u, len = n;  // the place is in [lo, lo + len]
  while (len) {
    const uint32_t step = (len + 63u) / 64u;
    const uint32_t at = (lane_id() + 1u) * step;
    const uint32_t hit = (uint32_t)__popcll(__ballot(at <= len && keys[lo + at - 1u] < v)) * step;
    lo += hit;
    len = min(step - 1u, len - hit);
  }
  return lo;
}

// cell_start[c] = keys below c, for c in [0, n_cells], kRsCells cells per
// block: their stretch of the keys, then a search in it per cell, in LDS where
// the stretch is short.
__global__ void __launch_bounds__(256) k_rs_cells(const uint32_t* keys, uint32_t n, uint32_t n_cells,
                                                  uint32_t* cell_start) {
  __shared__ uint32_t s_k[kRsStage];
  __shared__ uint32_t s_end[2];
  constexpr uint32_t kPer = kRsCells / 256u;
  const uint32_t tid = threadIdx.x, c0 = blockIdx.x * kRsCells, w = tid / 64u;
  if (w < 2u) {
    const uint32_t at = rs_lower_bound(keys, n, c0 + w * kRsCells);
    if (lane_id() == 0u) s_end[w] = at;
  }
  __syncthreads();
  const uint32_t lo = s_end[0], len = s_end[1] - lo;
  uint32_t at[kPer];
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) at[k] = 0u;
  // at[k]: keys of the stretch below the cell, the largest power of two first
  const uint32_t top = len ? 1u << (31u - (uint32_t)__clz((int)len)) : 0u;
  auto search = [&](auto key) {
    for (uint32_t step = top; step; step >>= 1) {
#pragma unroll
      for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t q = at[k] + step;
        if (q <= len && key(q - 1u) < c0 + k * 256u + tid) at[k] = q;
      }
    }
  };
  if (len <= kRsStage) {
    for (uint32_t q = tid; q < len; q += 256u) s_k[q] = keys[lo + q];
    __syncthreads();
    search([&](uint32_t q) { return s_k[q]; });
  } else {
    search([&](uint32_t q) { return keys[lo + q]; });
  }
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t c = c0 + k * 256u + tid;
    if (c <= n_cells) cell_start[c] = lo + at[k];
  }
}

// ====================================================================== tile
using dsmc_launch::kFlagSample;
using dsmc_launch::kFlagKeepPerm;
using dsmc_launch::kFlagHits;

// A tile is worked by NT threads: a workgroup (wide), or one wave of it
// (narrow: tiles of few particles, see k_tile).
template <uint32_t NT>
struct TileShape {
  static constexpr bool kWide = NT == kTileThreads;
  static constexpr uint32_t kCap = kWide ? kLdsCap : kNarrowCap;  // particles staged in LDS
  static constexpr uint32_t kMoveBatch = kWide ? 6 : 4;  // rounds of NT positions whose loads are issued together
  // PHYSICS: rounds of NT permutation entries of the next tile loaded into
  // registers during this tile's move (the next tile's first phase then only
  // stores them to LDS)
  static constexpr uint32_t kPermPrefetch = kWide ? 6 : 4;
};

// Pops a tile from a queue. The address comes from a vector register that the
// compiler cannot see through: an atomic that it knows to be uniform it makes
// for the whole wave, with a wait for the result right behind it (the wide
// kernel was 1.4 % slower at 33.5 million particles).
__device__ __forceinline__ uint32_t queue_pop(gptr<uint32_t> queue) {
  uint32_t at = 0u;
  asm volatile("" : "+v"(at));
  return gatomic_add(gelem(queue, at), 1u);
}

// Cells of at least this many particles are ranked in steps of 16: the launch
// waits for such a cell's tile, whose ranks take n^2 comparisons (REFERENCE
// benchmark case, which gathers 1100 of its 557k particles in one cell: 174 ->
// 124 us, without such a cell 75 us as before).
constexpr uint32_t kFullCell = 64;

// Thread of the tile.
template <uint32_t NT>
__device__ __forceinline__ uint32_t tile_tid() {
  return TileShape<NT>::kWide ? threadIdx.x : lane_id();
}

// Between the phases of a tile.
template <uint32_t NT>
__device__ __forceinline__ void tile_sync() {
  if (TileShape<NT>::kWide) {
    __syncthreads();
  } else {
    wave_sync();
  }
}

// LDS of the PHYSICS NTC rounds.
struct NtcLds {
  uint32_t* off;   // [cells] each cell's first item of the round
  uint32_t* nmax;  // [cells] (sigma c_r)max at the round's start (float bits)
  uint32_t* rmax;  // [cells] largest sigma c_r seen so far (float bits)
  uint8_t* icell;  // [NT] cell of each of the round's first NT items
  uint32_t* red;   // [8] wave totals of the scan, then the waves' largest round counts
};

// PHYSICS NTC of one tile in rounds of disjoint pairs (common/pairing.h).
// Lane l < nc computes cell l's candidate count M; round r holds
// min(floor(n / 2), M - r floor(n / 2)) pairs of each cell, and the pairs of
// all cells of a round are dealt to every thread of the workgroup (item t of
// the round: its cell from the scanned pair counts). The pairs of a round
// share no particle, so each is tested against the round's starting
// (sigma c_r)max and collided independently; the maximum then takes the
// round's largest sigma c_r. Draws: Philox4x32-10 under key
// (seed, kNtcKey1) at counter (cell, step, round, item).
template <uint32_t NT>
__device__ __forceinline__ void tile_ntc_rounds(const InstDesc& I, uint32_t c0, uint32_t nc, uint32_t p0,
                                                const uint32_t* s_start, float* vx, float* vy, float* vz,
                                                float2& nt, float frac, uint32_t stepno, const NtcLds& L,
                                                CollAcc& acc) {
  using namespace dsmc_pairing;
  const uint32_t tid = tile_tid<NT>(), lane = lane_id(), wid = tid / 64u;
  uint32_t n = 0u, M = 0u;
  if (tid < nc) {
    n = s_start[tid + 1] - s_start[tid];
    if (n >= 2u) {
      const float vol = I.cell_volume * (I.fluid_frac ? fmaxf(frac, kMinFluidFrac) : 1.0f);
      const float fpc = (float)(0.5 * (double)n * (double)(n - 1u) * (double)I.fnum * (double)nt.x *
                                    (double)I.dt / (double)vol +
                                (double)nt.y);
      M = dm_f2u_sat(fpc);
      nt.y = fpc - (float)M;
      if (M > kMaxPairsPerCell) {
        M = kMaxPairsPerCell;
        atomicOr(&I.ctr[3], kStatusPairs);
      }
      acc.sel += M;
    }
    L.nmax[tid] = __float_as_uint(nt.x);
    L.rmax[tid] = __float_as_uint(nt.x);
  }
  // rounds of the tile (the most over its cells), found with the first
  // round's scan
  uint32_t R = rounds_of(n, M);
  for (int o = 32; o > 0; o >>= 1) R = max(R, (uint32_t)__shfl_xor((int)R, o));
  uint32_t rounds = 1u;
  for (uint32_t r = 0; r < rounds; ++r) {
    const uint32_t m = round_pairs(n, M, r);
    // exclusive scan of the round's pair counts over the cells
    uint32_t x = m;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= (uint32_t)o) x += y;
    }
    if (lane == 63) L.red[wid] = x;
    if (r == 0u && lane == 0) L.red[4 + wid] = R;
    tile_sync<NT>();
    uint32_t base = 0u, total = 0u;
#pragma unroll
    for (uint32_t w = 0; w < NT / 64; ++w) {
      const uint32_t t = L.red[w];
      base += w < wid ? t : 0u;
      total += t;
      if (r == 0u) rounds = max(rounds, L.red[4 + w]);
    }
    if (total == 0u) break;  // uniform: round 0 without pairs means a tile without candidates
    const uint32_t off = base + x - m;
    if (tid < nc) {
      L.off[tid] = off;
      for (uint32_t q = off; q < off + m && q < NT; ++q) L.icell[q] = (uint8_t)tid;
    }
    tile_sync<NT>();
    for (uint32_t it = tid; it < total; it += NT) {
      uint32_t c;
      if (it < NT) {
        c = L.icell[it];
      } else {  // the last cell whose first item is at or before it
        uint32_t lo = 0u, hi = nc - 1u;
        while (lo < hi) {
          const uint32_t mid = (lo + hi + 1u) >> 1;
          if (L.off[mid] <= it) lo = mid;
          else hi = mid - 1u;
        }
        c = lo;
      }
      const uint32_t oc = L.off[c];
      const uint32_t mc = (c + 1u < nc ? L.off[c + 1u] : total) - oc;
      const uint32_t k = it - oc;
      const uint32_t a = s_start[c] - p0, nn = s_start[c + 1u] - s_start[c];
      const dsmc_rng::U32x4 rk = dsmc_rng::philox4x32_10({{c0 + c, stepno, r, kRoundItem}}, I.wall_key[0], kNtcKey1);
      const dsmc_rng::U32x4 d = dsmc_rng::philox4x32_10({{c0 + c, stepno, r, k}}, I.wall_key[0], kNtcKey1);
      uint32_t i, j;
      pair_members(nn, mc, k, rk, i, j);
      i += a;
      j += a;
      const float dx = vx[i] - vx[j], dy = vy[i] - vy[j], dz = vz[i] - vz[j];
      const float mag = sqrtf(dx * dx + dy * dy + dz * dz);
      const float sc =
          (I.vhs_exp == 1.0f) ? I.vhs_k * mag : (mag > 0.0f ? I.vhs_k * dm_powf(mag, I.vhs_exp) : 0.0f);
      atomicMax(&L.rmax[c], __float_as_uint(sc));
      const float max0 = __uint_as_float(L.nmax[c]);
      if (sc > dsmc_rng::px_unit(d.v[0]) * max0) {
        acc.coll += 1u;
        acc.cr += __double2ll_rn((double)mag * kCrScale);
        scatter_uv(vx, vy, vz, i, j, mag, dsmc_rng::px_unit(d.v[1]), dsmc_rng::px_unit(d.v[2]));
      }
    }
    tile_sync<NT>();
    if (tid < nc) L.nmax[tid] = L.rmax[tid];
  }
  if (tid < nc) nt.x = __uint_as_float(L.rmax[tid]);
}

template <uint32_t MODE, bool LDS, uint32_t NT>
__device__ __forceinline__ void tile_body(const InstDesc& I, uint32_t par, uint32_t flags, uint32_t tile,
                                          uint32_t c0, uint32_t nc, uint32_t p0, uint32_t np,
                                          const uint32_t* s_start, const uint8_t* s_nearc, uint32_t& tile_n,
                                          gptr<uint32_t> queue, uint32_t qx, bool per_xcd, uint32_t e_static,
                                          uint32_t* s_pop,
                                          uint32_t* sn_start, uint8_t* sn_nearc,
                                          uint32_t (&pf)[TileShape<NT>::kPermPrefetch],
                                          uint32_t* s_raw,
                                          uint32_t* s_perm, uint8_t* s_owner, float* s_vx, float* s_vy,
                                          float* s_vz, uint32_t stepno, const NtcLds& ntl, CollAcc& cacc) {
  const uint32_t tid = tile_tid<NT>();
  constexpr uint32_t kBatch = TileShape<NT>::kMoveBatch, kPf = TileShape<NT>::kPermPrefetch;
  constexpr uint32_t kCap = TileShape<NT>::kCap;
  const uint32_t opar = par ^ 1u;
  const gptr<const float> ipx = gmem<const float>(I.px[par]);
  const gptr<const float> ipy = gmem<const float>(I.py[par]);
  const gptr<const float> ipz = gmem<const float>(I.pz[par]);
  const gptr<const float> ivx = gmem<const float>(I.vx[par]);
  const gptr<const float> ivy = gmem<const float>(I.vy[par]);
  const gptr<const float> ivz = gmem<const float>(I.vz[par]);
  const gptr<float> opx = gmem(I.px[opar] + p0);
  const gptr<float> opy = gmem(I.py[opar] + p0);
  const gptr<float> opz = gmem(I.pz[opar] + p0);
  const gptr<float> ovx = gmem(I.vx[opar] + p0);
  const gptr<float> ovy = gmem(I.vy[opar] + p0);
  const gptr<float> ovz = gmem(I.vz[opar] + p0);
  const gptr<uint32_t> okey = gmem(I.key[opar] + p0);
  uint32_t* raw = LDS ? s_raw : (I.perm + p0);
  uint32_t* srt = LDS ? s_perm : (I.perm_tmp + p0);
  uint8_t* own = LDS ? s_owner : (I.owner_tmp + p0);
  float* vx = LDS ? s_vx : I.vx[opar] + p0;
  float* vy = LDS ? s_vy : I.vy[opar] + p0;
  float* vz = LDS ? s_vz : I.vz[opar] + p0;

  // the workgroup's next tile: taken from its queue now (dynamic
  // schedule; the atomic's latency is covered by phases 1 and 2), or the
  // next element of its fixed sequence
  const bool dyn = I.tile_dyn != 0u;
  uint32_t popped = 0u;
  if (dyn && tid == 0) popped = queue_pop(queue);
  // (1) raw permutation of the tile and the owning cell of each position
  if (LDS) {
    if (MODE == kModePhysics) {
#pragma unroll
      for (uint32_t k = 0; k < kPf; ++k)
        if (tid + k * NT < np) raw[tid + k * NT] = pf[k];
      for (uint32_t q = tid + kPf * NT; q < np; q += NT) raw[q] = *gelem(gmem(I.perm), p0 + q);
    } else {
      for (uint32_t q = tid; q < np; q += NT) raw[q] = *gelem(gmem(I.perm), p0 + q);
    }
  }
  if (tid < nc) {
    uint32_t a = s_start[tid] - p0, b = s_start[tid + 1] - p0;
    for (uint32_t q = a; q < b; ++q) own[q] = (uint8_t)tid;
  }
  tile_sync<NT>();
  // (2) rank of each entry among its cell's entries -> stable order
  for (uint32_t q = tid; q < np; q += NT) {
    uint32_t c = own[q];
    uint32_t a = s_start[c] - p0, b = s_start[c + 1] - p0;
    uint32_t v = raw[q];
    // four independent reads per iteration: dense cells are long loops
    uint32_t r0 = 0, r1 = 0, r2 = 0, r3 = 0;
    uint32_t j = a;
    if (LDS && TileShape<NT>::kWide && __builtin_expect(b - a >= kFullCell, 0)) {  // 16 reads
      for (; j & 3u; ++j) r0 += raw[j] < v ? 1u : 0u;
      for (; j + 16u <= b; j += 16u) {
        const uint4* const w = reinterpret_cast<const uint4*>(raw + j);
        const uint4 w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
        r0 += (w0.x < v ? 1u : 0u) + (w1.x < v ? 1u : 0u) + (w2.x < v ? 1u : 0u) + (w3.x < v ? 1u : 0u);
        r1 += (w0.y < v ? 1u : 0u) + (w1.y < v ? 1u : 0u) + (w2.y < v ? 1u : 0u) + (w3.y < v ? 1u : 0u);
        r2 += (w0.z < v ? 1u : 0u) + (w1.z < v ? 1u : 0u) + (w2.z < v ? 1u : 0u) + (w3.z < v ? 1u : 0u);
        r3 += (w0.w < v ? 1u : 0u) + (w1.w < v ? 1u : 0u) + (w2.w < v ? 1u : 0u) + (w3.w < v ? 1u : 0u);
      }
    }
    for (; j + 4u <= b; j += 4u) {
      r0 += raw[j] < v ? 1u : 0u;
      r1 += raw[j + 1u] < v ? 1u : 0u;
      r2 += raw[j + 2u] < v ? 1u : 0u;
      r3 += raw[j + 3u] < v ? 1u : 0u;
    }
    for (; j < b; ++j) r0 += raw[j] < v ? 1u : 0u;
    srt[a + r0 + r1 + r2 + r3] = v;
  }
  if (dyn && tid == 0) *s_pop = popped;
  tile_sync<NT>();
  {
    const uint32_t jn = tile_queue_pos(dyn ? *s_pop : e_static, qx, per_xcd);
    tile_n = jn < I.ntiles ? (I.tile_order ? gmem(I.tile_order)[jn] : jn) : kInvalidKey;
  }
  // the collision lane's cell state, requested with the first velocity
  // gathers so that the latencies overlap (lanes without a gather request it
  // before the loop)
  float2 nt_pf = make_float2(0.0f, 0.0f);
  float frac_pf = 1.0f;
  float4 st_pf = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  auto load_cell_state = [&]() {
    if (tid < nc && s_start[tid + 1] - s_start[tid] >= 2u) {
      nt_pf = gload(gmem<const float2>(I.ntc) + c0 + tid);
      if (MODE == kModeReference) st_pf = gload(gmem<const float4>(I.cstat) + c0 + tid);
      else if (I.fluid_frac) frac_pf = gmem(I.fluid_frac)[c0 + tid];
    }
  };
  if (tid >= np) load_cell_state();
  // (3) gather velocities in sorted order; the loads of kBatch positions
  // are issued before any store so that their latencies overlap
  for (uint32_t q0 = tid; q0 < np; q0 += kBatch * NT) {
    float gx[kBatch], gy[kBatch], gz[kBatch];
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
      const uint32_t q = q0 + k * NT;
      gx[k] = gy[k] = gz[k] = 0.0f;
      if (q < np) {
        const uint32_t src = srt[q];
        gx[k] = *gelem(ivx, src);
        gy[k] = *gelem(ivy, src);
        gz[k] = *gelem(ivz, src);
      }
    }
    if (q0 == tid) load_cell_state();
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
      const uint32_t q = q0 + k * NT;
      if (q < np) {
        vx[q] = gx[k];
        vy[q] = gy[k];
        vz[q] = gz[k];
      }
    }
  }
  tile_sync<NT>();
  // Every load issued so far has arrived (the velocity gather waited for
  // them); saying so here keeps the compiler from waiting for the next
  // tile's loads below at the first use of an older one in the NTC phase.
  wait_vmem();
  // the next tile's cell offsets and near flags, stored to the other LDS
  // buffer at the end of this phase: the next tile starts without a load
  uint32_t nx_start = 0u, nx_end = 0u, ncn = 0u;
  uint8_t nx_near = 255u;
  if (tile_n != kInvalidKey) {
    const uint32_t c0n = tile_n * I.tile_cells;
    ncn = min(I.tile_cells, I.ncells - c0n);
    nx_start = gmem(I.cell_start)[c0n + min(tid, ncn)];
    if (tid == 0) nx_end = gmem(I.cell_start)[c0n + ncn];
    if (MODE == kModePhysics) nx_near = (I.near_cell && tid < ncn) ? gmem(I.near_cell)[c0n + tid] : (uint8_t)255;
  }
  // (4) NTC collisions: REFERENCE one lane per cell (the reference's loop),
  // PHYSICS in rounds of disjoint pairs over the whole workgroup
  if (MODE == kModeReference) {
    if (tid < nc) {
      const uint32_t c = c0 + tid;
      const uint32_t a = s_start[tid] - p0, n = s_start[tid + 1] - s_start[tid];
      if (n >= 2u) {
        float2 nt = nt_pf;
        float4 st = st_pf;
        if (I.taus) {
          uint4 q = gload(gmem<const uint4>(reinterpret_cast<const uint4*>(I.taus)) + c);
          Taus t = {q.x, q.y, q.z, q.w};
          ntc_reference(I, vx + a, vy + a, vz + a, n, nt, st, t);
          gstore(gmem(reinterpret_cast<uint4*>(I.taus)) + c, make_uint4(t.x, t.y, t.z, t.w));
        } else {
          // ComputeBirdCollisionsDev draws from the cell's own stream
          // (ds_mtState[cellid], dsmc_kernel.cu:1030-1031)
          Mt cr;
          mt_load(I, c, cr);
          ntc_reference(I, vx + a, vy + a, vz + a, n, nt, st, cr);
          mt_store(I, c, cr);
        }
        gstore(gmem(I.cstat) + c, st);
        gstore(gmem(I.ntc) + c, nt);
      }
    }
  }
  float2 ntc_state = nt_pf;
  if (MODE == kModePhysics) {
    // frac_pf is first used here: without this marker the compiler applies
    // the NTC's clamp of it right after its load, whose wait then comes
    // before the velocity gather instead of after it
    asm volatile("" : "+v"(frac_pf));
    tile_ntc_rounds<NT>(I, c0, nc, p0, s_start, vx, vy, vz, ntc_state, frac_pf, stepno, ntl, cacc);
  }
  if (tile_n != kInvalidKey) {
    sn_start[tid] = nx_start;
    if (tid == 0) sn_start[ncn] = nx_end;
    if (MODE == kModePhysics) sn_nearc[tid] = nx_near;
  }
  if (MODE == kModePhysics) {  // after the next tile's offsets, so that their wait is not a wait for this store
    if (tid < nc && s_start[tid + 1] - s_start[tid] >= 2u) gstore(gmem(I.ntc) + c0 + tid, ntc_state);
  }
  // per-cell counts of the particles that stay in the tile (the NTC is done
  // with the offsets that share this LDS)
  ntl.off[tid] = 0u;
  if (tid == 0) gmem(I.tile_p0)[tile] = p0;
  tile_sync<NT>();
  // the next tile's first permutation entries (its offsets are in LDS now),
  // requested with the first batch of position gathers and waited for with
  // them, so that no later wait (the next tile's first use of pf comes after
  // this tile's stores) has to wait for the stores
  auto load_pf = [&]() {
    if (MODE == kModePhysics && tile_n != kInvalidKey) {
      const uint32_t p0n = sn_start[0];
      const uint32_t npn = sn_start[ncn] - p0n;
#pragma unroll
      for (uint32_t k = 0; k < kPf; ++k) {
        const uint32_t q = tid + k * NT;
        pf[k] = (npn <= kCap && q < npn) ? *gelem(gmem(I.perm), p0n + q) : 0u;
      }
    }
  };
  // (5) move, walls, box faces, next key; rounds keep waves converged for
  // the aggregated counting
  const uint32_t rounds = (np + NT - 1u) / NT;
  if (rounds == 0u) {
    load_pf();
    wait_vmem();
  }
  for (uint32_t r0 = 0; r0 < rounds; r0 += kBatch) {
    if (r0 == 0u) load_pf();
    // positions of up to kBatch rounds in flight before the first store
    float bx[kBatch], by[kBatch], bz[kBatch];
    uint32_t bsrc[kBatch];
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
      const uint32_t q = (r0 + k) * NT + tid;
      bsrc[k] = 0u;
      bx[k] = by[k] = bz[k] = 0.0f;
      if (q < np) {
        const uint32_t src = srt[q];
        bsrc[k] = src;
        bx[k] = *gelem(ipx, src);
        by[k] = *gelem(ipy, src);
        bz[k] = *gelem(ipz, src);
      }
    }
    wait_vmem();
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
    if (r0 + k >= rounds) break;  // uniform over the workgroup
    uint32_t q = (r0 + k) * NT + tid;
    uint32_t key = kInvalidKey;
    // REFERENCE: the wall flights of the wavefront run together (every lane
    // takes part, with or without a particle)
    float rx = 0.0f, ry = 0.0f, rz = 0.0f, rux = 0.0f, ruy = 0.0f, ruz = 0.0f;
    uint32_t rhits = 0;
    if (MODE == kModeReference) {
      if (q < np) {
        rx = bx[k], ry = by[k], rz = bz[k];
        rux = vx[q], ruy = vy[q], ruz = vz[q];
      }
      rhits = move_reference_wave(I, q < np, rx, ry, rz, rux, ruy, ruz, I.dt, ntl.rmax + (tid & ~63u));
    }
    if (q < np) {
      const uint32_t src = bsrc[k];
      float x = bx[k], y = by[k], z = bz[k];
      float ux = vx[q], uy = vy[q], uz = vz[q];
      uint32_t hits = 0;
      if (MODE == kModeReference) {
        x = rx, y = ry, z = rz, ux = rux, uy = ruy, uz = ruz;
        hits = rhits;
        key = cell_key(I, x, y, z);
      } else if (phys_near(I, s_nearc[own[q]], ux, uy, uz, I.dt)) {
        key = kDeferredKey;  // stored as is; k_walls moves it and counts its key
      } else {
        key = move_free(I, x, y, z, ux, uy, uz, I.dt);
      }
      opx[q] = x;
      opy[q] = y;
      opz[q] = z;
      okey[q] = key;
      if (LDS) {
        ovx[q] = ux;
        ovy[q] = uy;
        ovz[q] = uz;
      }
      if (!LDS || (flags & kFlagSample)) {  // post-move velocities: output (global path) or sampled
        vx[q] = ux;
        vy[q] = uy;
        vz[q] = uz;
      }
      if (flags & kFlagHits) gmem(I.hits)[p0 + q] = hits;
      if (flags & kFlagKeepPerm) *gelem(gmem(I.perm), p0 + q) = src;
    }
    const bool stayed = I.tile_dyn && key - c0 < nc;  // in the tile's cells
    if (stayed) atomicAdd(&ntl.off[key - c0], 1u);
    count_keys(gmem(I.count), key == kDeferredKey || (stayed && stayers_apart<MODE>(I)) ? kInvalidKey : key);
    if (MODE == kModePhysics) {
      // mark the wave's deferred slots in the bitmask the wall pass reads
      const uint64_t m = __ballot(key == kDeferredKey);
      if (m && lane_id() == 0) {
        const uint32_t s0 = p0 + (r0 + k) * NT + (tid & ~63u);
        const uint32_t sh = s0 & 63u;
        const gptr<unsigned long long> wb = gmem(I.defer_bits) + s0 / 64u;
        __hip_atomic_fetch_or(wb, (unsigned long long)(m << sh), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (sh)
          __hip_atomic_fetch_or(wb + 1, (unsigned long long)(m >> (64u - sh)), __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    }
  }

  // (6) sampling of the post-move velocities, one lane per cell
  if ((flags & kFlagSample) && I.sample_on) {
    tile_sync<NT>();
    if (tid < nc) {
      uint32_t c = c0 + tid;
      uint32_t a = s_start[tid] - p0, b = s_start[tid + 1] - p0;
      if (b > a) {
        if (MODE == kModeReference) {
          // SampleCellStatisticsDev (dsmc_kernel.cu:856-890), FP32 sums
          const gptr<float> S = gmem(reinterpret_cast<float*>(I.samp));
          const uint32_t C = I.ncells;
          float sn = S[c], sx = S[C + c], sy = S[2 * C + c], sz = S[3 * C + c], s2 = S[4 * C + c];
          for (uint32_t q = a; q < b; ++q) {
            float ux = vx[q], uy = vy[q], uz = vz[q];
            sn += 1.0f;
            sx += ux;
            sy += uy;
            sz += uz;
            s2 += ux * ux + uy * uy + uz * uz;
          }
          S[c] = sn; S[C + c] = sx; S[2 * C + c] = sy; S[3 * C + c] = sz; S[4 * C + c] = s2;
        } else {
          const gptr<double> S = gmem(I.samp);
          const uint32_t C = I.ncells;
          double sn = S[c], sx = S[C + c], sy = S[2 * C + c], sz = S[3 * C + c], s2 = S[4 * C + c];
          for (uint32_t q = a; q < b; ++q) {
            double ux = vx[q], uy = vy[q], uz = vz[q];
            sn += 1.0;
            sx += ux;
            sy += uy;
            sz += uz;
            s2 += ux * ux + uy * uy + uz * uz;
          }
          S[c] = sn; S[C + c] = sx; S[2 * C + c] = sy; S[3 * C + c] = sz; S[4 * C + c] = s2;
        }
      }
    }
  }
}

// LDS of one tile. The raw permutation is dead once the rank sort has run
// (phase 2), so the z velocities reuse its space.
struct TileLds {
  static constexpr uint32_t kStart = kTileCells + 4;
  uint32_t* start;  // [cells + 1] cell offsets of the current tile, and kStart further of the next one
  uint8_t* near;    // [cells] PHYSICS: near flags, likewise (kTileCells further)
  uint32_t* raw;    // [kCap] and so are the others
  uint32_t* perm;
  uint8_t* owner;
  float* vx;
  float* vy;
  NtcLds ntc;
};

// Walk over tiles: `tile` first, then the positions that tile_body finds next
// (queue, or e_stride further along the fixed sequence; single: none).
template <uint32_t MODE, uint32_t NT>
__device__ __forceinline__ void tile_walk(const InstDesc& I, uint32_t par, uint32_t flags, uint32_t tile, uint32_t e,
                                          uint32_t e_stride, uint32_t qx, bool per_xcd, gptr<uint32_t> queue,
                                          uint32_t* s_pop, uint32_t stepno, const TileLds& L, CollAcc& cacc,
                                          uint32_t* over) {
  using S = TileShape<NT>;
  const uint32_t tid = tile_tid<NT>();
  float* const vz = reinterpret_cast<float*>(L.raw);
  {
    const uint32_t c0 = tile * I.tile_cells;
    const uint32_t nc = min(I.tile_cells, I.ncells - c0);
    L.start[tid] = gmem(I.cell_start)[c0 + min(tid, nc)];
    if (tid == 0) L.start[nc] = gmem(I.cell_start)[c0 + nc];
    if (MODE == kModePhysics) L.near[tid] = (I.near_cell && tid < nc) ? gmem(I.near_cell)[c0 + tid] : (uint8_t)255;
  }
  tile_sync<NT>();
  uint32_t pf[S::kPermPrefetch];
  if (MODE == kModePhysics) {
    const uint32_t nc = min(I.tile_cells, I.ncells - tile * I.tile_cells);
    const uint32_t p0 = L.start[0], np = L.start[nc] - p0;
#pragma unroll
    for (uint32_t k = 0; k < S::kPermPrefetch; ++k) {
      const uint32_t q = tid + k * NT;
      pf[k] = (np <= S::kCap && q < np) ? *gelem(gmem(I.perm), p0 + q) : 0u;
    }
  }
  wait_vmem();  // the first tile needs them now; later tiles find theirs arrived
  for (uint32_t b = 0; tile != kInvalidKey; b ^= 1u) {
    uint32_t tile_n = kInvalidKey;  // set by tile_body
    e += e_stride;                  // the next element of the fixed sequence
    const uint32_t c0 = tile * I.tile_cells;
    const uint32_t nc = min(I.tile_cells, I.ncells - c0);
    uint32_t *const start = L.start + b * L.kStart, *const start_n = L.start + (b ^ 1u) * L.kStart;
    uint8_t *const near = L.near + b * kTileCells, *const near_n = L.near + (b ^ 1u) * kTileCells;
    const uint32_t p0 = start[0], np = start[nc] - p0;
    // a narrow tile above its capacity is left to the whole workgroup: the
    // wave takes it as empty and only finds the next one
    const bool fits = np <= S::kCap;
    if (!S::kWide && !fits && tid == 0) over[atomicAdd(over, 1u) + 1u] = tile;
    if (fits || !S::kWide)
      tile_body<MODE, true, NT>(I, par, flags, tile, c0, fits ? nc : 0u, p0, fits ? np : 0u, start, near, tile_n,
                                queue, qx, per_xcd, e, s_pop, start_n, near_n, pf, L.raw, L.perm, L.owner, L.vx, L.vy, vz,
                                stepno, L.ntc, cacc);
    else
      tile_body<MODE, false, NT>(I, par, flags, tile, c0, nc, p0, np, start, near, tile_n, queue, qx,
                                 per_xcd, e, s_pop, start_n, near_n, pf, L.raw, L.perm, L.owner, L.vx,
                                 L.vy, vz, stepno, L.ntc, cacc);
    tile_sync<NT>();
    if (I.tile_dyn && tid < nc) gmem(I.local_cnt)[c0 + tid] = L.ntc.off[tid];
    tile = tile_n;
  }
}

// A workgroup takes one tile after the other; where tiles hold few particles
// (NARROW, instances with tile_narrow), each of its waves takes its own:
// the phases of such a tile are too short to feed 256 threads, and what bounds
// it is the latency of its chain of loads, of which four times as many are in
// flight this way, without a barrier between the phases. Tiles that turn out
// too full for a wave's LDS are done by the workgroup at the end.
template <uint32_t MODE, bool NARROW>
__global__ void __launch_bounds__(kTileThreads, 4) k_tile(const InstDesc* __restrict__ Ip, uint32_t par, uint32_t flags,
                                                      const uint2* map) {
  const uint2 blk = block_of(map);
  const InstDesc& I = Ip[blk.x];
  // 40.7 KB, four workgroups per CU. Arrays of their own, so that the compiler
  // can tell them apart (one struct of them: 1.5 % slower); a wave's share
  // where tiles are narrow.
  __shared__ uint32_t s_start[2 * TileLds::kStart];
  __shared__ uint8_t s_nearc[2 * kTileCells];
  __shared__ __align__(16) uint32_t s_raw[kLdsCap];
  __shared__ uint32_t s_perm[kLdsCap];
  __shared__ uint8_t s_owner[kLdsCap];
  __shared__ float s_vx[kLdsCap];
  __shared__ float s_vy[kLdsCap];
  __shared__ uint32_t s_ntc_off[kTileCells];
  __shared__ uint32_t s_ntc_nmax[kTileCells];
  __shared__ uint32_t s_ntc_rmax[kTileCells];
  __shared__ uint32_t s_ntc_red[NARROW ? 8 * (kTileThreads / 64) : 8];
  // the NTC rounds' item-cell table, and the counters' sums at the end
  __shared__ long long s_red[kTileThreads / 8];
  static_assert(4u * kNarrowCap <= kLdsCap && 4u * kNarrowCells <= kTileCells && 4u * (kNarrowCells + 1u) <= TileLds::kStart,
                "four narrow tiles share a wide tile's LDS");
  const auto lds_of = [&](uint32_t cells, uint32_t cap, uint32_t k) {  // the k-th of tiles of this size
    TileLds L;
    L.start = s_start + k * (cells + 1u);
    L.near = s_nearc + k * cells;
    L.raw = s_raw + k * cap;
    L.perm = s_perm + k * cap;
    L.owner = s_owner + k * cap;
    L.vx = s_vx + k * cap;
    L.vy = s_vy + k * cap;
    L.ntc.off = s_ntc_off + k * cells;
    L.ntc.nmax = s_ntc_nmax + k * cells;
    L.ntc.rmax = s_ntc_rmax + k * cells;
    L.ntc.icell = reinterpret_cast<uint8_t*>(s_red) + k * cells;
    L.ntc.red = s_ntc_red + k * 8u;
    return L;
  };
  __shared__ uint32_t s_pop;
  const uint32_t tid = threadIdx.x;
  const uint32_t vw = blk.y;
  const uint32_t stepno = gmem(I.ctr)[4];  // this step's number (counter of the PHYSICS draws)
  if (vw == 0 && tid == 0) {
    I.ctr[0] = I.ctr[1];
    I.tile_p0[I.ntiles] = I.ctr[1];  // the slots this launch stores in tile order
  }
  // tiles come from the XCD's queue (dynamic schedule) or, for instances
  // whose tiles are small, as the fixed sequence of elements vw / 8,
  // vw / 8 + G / 8, ... of that queue (no atomic per tile); narrow: with a
  // walker per wave
  const bool per_xcd = I.n_tile_wg % 8u == 0u;
  const uint32_t qx = per_xcd ? vw % 8u : 0u;
  const uint32_t wgs = per_xcd ? I.n_tile_wg / 8u : I.n_tile_wg;
  const gptr<uint32_t> queue = gmem(I.ctr) + kTileQueueCtr + qx;
  uint32_t e = per_xcd ? vw / 8u : vw;
  CollAcc cacc = {0ull, 0ull, 0ll};
  auto tile_at = [&](uint32_t el) {
    const uint32_t j = tile_queue_pos(el, qx, per_xcd);
    return j >= I.ntiles ? kInvalidKey : I.tile_order ? gmem(I.tile_order)[j] : j;
  };
  if constexpr (NARROW) {
    constexpr uint32_t kW = kTileThreads / 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64u);
    __shared__ uint32_t s_over[kNarrowWalk * kW + 1u];  // count, tiles
    if (tid == 0) s_over[0] = 0u;
    __syncthreads();
    e = e * kW + wave;
    const uint32_t tile = tile_at(e);
    if (tile != kInvalidKey)
      tile_walk<MODE, 64>(I, par, flags, tile, e, wgs * kW, qx, per_xcd, queue, &s_pop, stepno,
                          lds_of(kNarrowCells, kNarrowCap, wave), cacc, s_over);
    __syncthreads();
    for (uint32_t k = 0; k < s_over[0]; ++k) {
      tile_walk<MODE, kTileThreads>(I, par, flags, s_over[k + 1u], kInvalidKey / 2u, 0u, 0u, false, queue, &s_pop, stepno,
                                    lds_of(kTileCells, kLdsCap, 0u), cacc, nullptr);
      __syncthreads();
    }
  } else {
    if (I.tile_dyn) {
      if (tid == 0) s_pop = queue_pop(queue);
      __syncthreads();
      e = s_pop;
    }
    const uint32_t tile = tile_at(e);
    if (tile == kInvalidKey) return;  // no tile: this workgroup's counters stay as they are
    tile_walk<MODE, kTileThreads>(I, par, flags, tile, e, wgs, qx, per_xcd, queue, &s_pop, stepno,
                                  lds_of(kTileCells, kLdsCap, 0u), cacc, nullptr);
  }

  // per-workgroup collision counters (integers: exact in any order)
  if (MODE == kModePhysics) {
    __syncthreads();
    long long v[3] = {(long long)cacc.sel, (long long)cacc.coll, cacc.cr};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      long long x = v[k];
      for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off);
      if (lane_id() == 0) s_red[(tid / 64) * 3 + k] = x;
    }
    __syncthreads();
    if (tid < 3) {
      long long t = 0;
      for (uint32_t w = 0; w < kTileThreads / 64; ++w) t += s_red[w * 3 + tid];
      gmem(I.wg_acc)[vw * kAccSlots + tid] += t;
    }
  }
}


// =============================================================== wall pass
// PHYSICS: the particles the tile kernel deferred (key kDeferredKey, state
// after collisions, before the move; one bit per slot in defer_bits) fly
// with walls and faces here, in two launches.
//
// k_defer_list (large instances) compacts the marked slots: each wave takes chunks of 64
// bitmask words (4096 slots) and finds their set bits with one coalesced
// load; the workgroup reserves room for its waves' chunks in defer_list with
// one atomic; each word's slots are written as one contiguous run (lane l
// tests bit l) and the words cleared.
__global__ void __launch_bounds__(kTileThreads) k_defer_list(const InstDesc* __restrict__ Ip) {
  const InstDesc& I = Ip[blockIdx.y];
  if (!I.defer_bits || I.wall_direct || blockIdx.x >= I.n_wall_wg) return;
  __shared__ uint32_t s_tot[kTileThreads / 64u + 1u];
  const uint32_t lane = lane_id(), wave = threadIdx.x / 64u;
  const uint32_t nwords = (I.ctr[1] + 63u) / 64u;  // deferred slots lie below the sorted count
  const uint32_t nchunks = (nwords + 63u) / 64u;
  const gptr<unsigned long long> bits = gmem(I.defer_bits);
  const gptr<uint32_t> list = gmem(I.defer_list);
  constexpr uint32_t kWaves = kTileThreads / 64u;
  // the workgroup takes kWaves chunks per round (one per wave) and reserves
  // room for all of them with one atomic
  for (uint32_t c0 = blockIdx.x * kWaves; c0 < nchunks; c0 += I.n_wall_wg * kWaves) {
    const uint32_t ch = c0 + wave;
    const uint32_t w = ch * 64u + lane;
    const unsigned long long word = (ch < nchunks && w < nwords) ? bits[w] : 0ull;
    const uint32_t pc = (uint32_t)__popcll(word);
    uint32_t incl = pc;
    for (uint32_t off = 1; off < 64u; off <<= 1) {
      const uint32_t t = __shfl_up(incl, off);
      if (lane >= off) incl += t;
    }
    if (lane == 63u) s_tot[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t sum = 0;
      for (uint32_t q = 0; q < kWaves; ++q) {
        const uint32_t x = s_tot[q];
        s_tot[q] = sum;
        sum += x;
      }
      s_tot[kWaves] = sum ? gatomic_add(gmem(I.ctr) + 5, sum) : 0u;
    }
    __syncthreads();
    const uint32_t base = s_tot[kWaves] + s_tot[wave];
    const bool any = __shfl(incl, 63) != 0u;
    __syncthreads();  // s_tot is rewritten in the next round
    if (!any) continue;  // uniform over the wave
    // word r of the chunk (read from lane r): each lane tests its own bit,
    // so the word's set slots are written as one contiguous run
    const uint32_t ex = incl - pc;
    const unsigned long long below = (1ull << lane) - 1ull;
    for (uint32_t r = 0; r < 64u; ++r) {
      const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)word, r);
      const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(word >> 32), r);
      const unsigned long long wr = ((unsigned long long)hi << 32) | lo;
      if (wr == 0ull) continue;  // uniform over the wave
      const uint32_t off = __builtin_amdgcn_readlane(ex, r);
      if ((wr >> lane) & 1ull) list[base + off + (uint32_t)__popcll(wr & below)] = (ch * 64u + r) * 64u + lane;
    }
    if (word) bits[w] = 0ull;
  }
}

// ================================================================= injection
// Freestream inflow through open faces (PHYSICS): face cell g of face f
// injects floor(lambda_f + R) particles with the flux-weighted half-range
// Maxwellian normal velocity (acceptance-rejection on the speed-ratio
// density z exp(-(z - s)^2), Bird 1994 sec. 12.1) and Gaussian tangential
// components, placed on the face and advanced a random fraction of dt.
//
// One thread per injected particle t (workgroup ib of nib, grid-stride): its
// face cell is the last g with face_count[g] <= t (face_count holds the
// exclusive offsets), it is particle t - face_count[g] of that cell, and it
// goes to slot sorted count + t.
__device__ __forceinline__ void inject_generate(const InstDesc& I, uint32_t opar, uint32_t ib, uint32_t nib) {
  const uint32_t F = I.n_face_cells;
  if (F == 0) return;
  const uint32_t t0 = ib * kTileThreads + threadIdx.x;
  const uint32_t base = I.ctr[1];
  const uint32_t tot = I.face_count[F];
  if (t0 == 0) {
    uint32_t end = base + tot;
    if (end > I.cap || end < base) {  // capacity exceeded: drop the excess, flag it
      end = I.cap;
      atomicOr(&I.ctr[3], kStatusCapacity);
    }
    I.ctr[0] = end;
    I.ctr[2] += end - base;
  }
  const uint32_t stepno = I.ctr[4];
  const uint32_t k0 = I.wall_key[0];
  const gptr<const uint32_t> fc = gmem<const uint32_t>(I.face_count);
  const float twopi = 6.28318530717958647692f;
  const float vm = I.vm_inf;
  const float sd = vm * 0.70710678118654752f;  // sqrt(kT/m)
  for (uint32_t t = t0; t < tot; t += nib * kTileThreads) {
    const uint32_t idx = base + t;
    if (idx >= I.cap || idx < base) break;  // later t only go further
    uint32_t lo = 0u, hi = F;  // fc[lo] <= t < fc[hi]
    while (hi - lo > 1u) {
      const uint32_t mid = lo + (hi - lo) / 2u;
      if (fc[mid] <= t) lo = mid;
      else hi = mid;
    }
    const uint32_t g = lo, j = t - fc[g];
    const uint32_t f = face_of(I, g);
    const uint32_t local = g - I.face_off[f];
    const uint32_t axis = f >> 1;           // normal axis
    const uint32_t ta = axis == 0 ? 1u : 0u;  // first tangential axis
    const uint32_t tb = axis == 2 ? 1u : 2u;  // second tangential axis
    const uint32_t na = I.dim[ta];
    const uint32_t ia = local % na, ib = local / na;
    const float sign = (f & 1u) ? -1.0f : 1.0f;  // inward normal direction
    const float un = sign * I.U[axis];           // inward stream component
    const float sr = un / vm;                    // speed ratio of the inflow
    float zlo = sr - 5.0f;
    zlo = zlo > 0.0f ? zlo : 0.0f;
    float zhi = sr + 5.0f;
    zhi = zhi > 1.0e-3f ? zhi : 1.0e-3f;
    float zs = 0.5f * (sr + sqrtf(sr * sr + 2.0f));  // mode of z exp(-(z-s)^2)
    zs = zs < zlo ? zlo : (zs > zhi ? zhi : zs);
    const float gmax = zs * dm_expf(-(zs - sr) * (zs - sr));
    float z = zlo;
    bool ok = false;
    for (uint32_t b = 0; b < 500u && !ok; ++b) {
      const dsmc_rng::U32x4 c = {{g, stepno, 1u + j, b}};
      const dsmc_rng::U32x4 r = dsmc_rng::philox4x32_10(c, k0, kInjectKey1);
      for (int h = 0; h < 2 && !ok; ++h) {
        z = zlo + (zhi - zlo) * dsmc_rng::px_unit(r.v[2 * h]);
        const float gz = z * dm_expf(-(z - sr) * (z - sr));
        ok = gz > gmax * dsmc_rng::px_unit(r.v[2 * h + 1]);
      }
    }
    const dsmc_rng::U32x4 ca = {{g, stepno, 1u + j, 0x80000000u}};
    const dsmc_rng::U32x4 ra = dsmc_rng::philox4x32_10(ca, k0, kInjectKey1);
    const dsmc_rng::U32x4 cb = {{g, stepno, 1u + j, 0x80000001u}};
    const dsmc_rng::U32x4 rb = dsmc_rng::philox4x32_10(cb, k0, kInjectKey1);
    const float vn = z * vm;
    const float a1 = sqrtf(-2.0f * dm_logf(dsmc_rng::px_unit(ra.v[0])));
    float s1, c1;
    dm_sincosf(twopi * dsmc_rng::px_unit(ra.v[1]), &s1, &c1);
    float p[3], v[3];
    v[axis] = sign * vn;
    v[ta] = I.U[ta] + sd * a1 * c1;
    v[tb] = I.U[tb] + sd * a1 * s1;
    p[axis] = (f & 1u) ? I.gmax[axis] : I.gmin[axis];
    p[ta] = I.gmin[ta] + ((float)ia + dsmc_rng::px_unit(ra.v[2])) * I.cell[ta];
    p[tb] = I.gmin[tb] + ((float)ib + dsmc_rng::px_unit(ra.v[3])) * I.cell[tb];
    const float fr = dsmc_rng::px_unit(rb.v[0]) * I.dt;
    float x = p[0] + v[0] * fr, y = p[1] + v[1] * fr, zz = p[2] + v[2] * fr;
    x = x < I.gmin[0] ? I.gmin[0] : (x > I.gmax[0] ? I.gmax[0] : x);
    y = y < I.gmin[1] ? I.gmin[1] : (y > I.gmax[1] ? I.gmax[1] : y);
    zz = zz < I.gmin[2] ? I.gmin[2] : (zz > I.gmax[2] ? I.gmax[2] : zz);
    I.px[opar][idx] = x; I.py[opar][idx] = y; I.pz[opar][idx] = zz;
    I.vx[opar][idx] = v[0]; I.vy[opar][idx] = v[1]; I.vz[opar][idx] = v[2];
    const uint32_t key = cell_key_phys(I, x, y, zz);
    I.key[opar][idx] = key;
    gatomic_add(gmem(I.count) + key, 1u);
  }
}

// k_walls moves the deferred particles, one per thread; the 64 lanes of a
// wavefront fly their particles together, testing the triangle entries of all
// their cells as one pool. They come from the compacted list (a grid-stride
// loop over it), or, where one small instance has the GPU to itself
// (wall_direct), from the bitmask: each wave takes whole words, 64 slots, and
// moves the marked lanes - the compaction's launch and round trip take longer
// than the idle lanes (100k particles: list, walls and sum 6 + 22 + 4 us, 15
// direct; 64 such instances together: 53 us against 154).
// The pass holds no RNG state (Philox draws keyed by slot and step). Wall
// forces and heat are summed in 64-bit fixed point, so the order in which
// particles are taken does not change the sums; each workgroup stores its
// sums in its own slot of wall_part, which the next step's scan (or the host,
// before it reads the totals) folds into wall_acc.
//
// The workgroups after the instance's n_wall_wg inject the inflow beside
// that: both only add to the cell counts, injection writes the slots after
// the sorted ones and the wall pass deferred slots below them.
__global__ void __launch_bounds__(kTileThreads, 4) k_walls(const InstDesc* __restrict__ Ip, uint32_t opar,
                                                       uint32_t flags, const uint2* map) {
  const uint2 blk = block_of(map);
  const InstDesc& I = Ip[blk.x];
  const uint32_t bx = blk.y, n_wg = I.defer_bits ? I.n_wall_wg : 0u;
  if (bx >= n_wg) {
    inject_generate(I, opar, bx - n_wg, I.n_inj_wg);
    return;
  }
  __shared__ long long s_red[kTileThreads / 64][4];
  __shared__ unsigned long long s_hit[kTileThreads / 64][64];
  const uint32_t stepno = I.ctr[4];
  const uint32_t tid = threadIdx.x, lane = lane_id(), wid = tid / 64;
  const gptr<float> px = gmem(I.px[opar]);
  const gptr<float> py = gmem(I.py[opar]);
  const gptr<float> pz = gmem(I.pz[opar]);
  const gptr<float> vx = gmem(I.vx[opar]);
  const gptr<float> vy = gmem(I.vy[opar]);
  const gptr<float> vz = gmem(I.vz[opar]);
  const gptr<uint32_t> key = gmem(I.key[opar]);
  WallAcc acc = {0, 0, 0, 0};
  const WaveHitLds hl = {s_hit[wid]};
  // called by whole wavefronts: the wall flights run their lanes together,
  // and the counting is wave-aggregated (neighbouring slots mostly land in
  // the same cell)
  auto fly = [&](bool act, uint32_t slot) {
    float x = 0.0f, y = 0.0f, z = 0.0f, ux = 0.0f, uy = 0.0f, uz = 0.0f;
    if (act) {
      x = px[slot], y = py[slot], z = pz[slot];
      ux = vx[slot], uy = vy[slot], uz = vz[slot];
    }
    uint32_t hits;
    const uint32_t k = move_walls(I, act, x, y, z, ux, uy, uz, I.dt, slot, stepno, hits, acc, hl);
    if (act) {
      px[slot] = x;
      py[slot] = y;
      pz[slot] = z;
      vx[slot] = ux;
      vy[slot] = uy;
      vz[slot] = uz;
      key[slot] = k == kInvalidKey ? k : (k | kWallKeyBit);
      if (flags & kFlagHits) gmem(I.hits)[slot] = hits;
    }
    count_keys(gmem(I.count), k);
  };
  if (I.wall_direct) {
    const gptr<unsigned long long> bits = gmem(I.defer_bits);
    const uint32_t nwords = (I.ctr[1] + 63u) / 64u;  // deferred slots lie below the sorted count
    for (uint32_t w = bx * (kTileThreads / 64u) + wid; w < nwords; w += n_wg * (kTileThreads / 64u)) {
      const unsigned long long word = bits[w];
      if (word == 0ull) continue;  // uniform over the wave
      fly((word >> lane) & 1ull, w * 64u + lane);
      if (lane == 0) bits[w] = 0ull;
    }
  } else {
    const gptr<const uint32_t> list = gmem<const uint32_t>(I.defer_list);
    const uint32_t cnt = I.ctr[5];
    for (uint32_t b = bx * kTileThreads; b < cnt; b += n_wg * kTileThreads) {
      const bool act = b + tid < cnt;
      fly(act, act ? list[b + tid] : 0u);
    }
  }
  long long v[4] = {acc.fx, acc.fy, acc.fz, acc.heat};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    long long x = v[k];
    for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off);
    if (lane == 0) s_red[wid][k] = x;
  }
  __syncthreads();
  if (tid < 4) {  // the workgroup's own slot: plain stores, no contention
    long long t = 0;
    for (uint32_t q = 0; q < kTileThreads / 64; ++q) t += s_red[q][tid];
    gmem(I.wall_part)[bx * 4u + tid] = t;
  }
}

// The totals that the host reads: the wall sums that no step has folded yet
// into wall_acc, and the sums over the workgroups' collision counters, as
// 64-bit sums of their low and high halves (out[2 k], out[2 k + 1] of slot k:
// exact, the host puts them together in 128 bits). n_acc: the tile kernel's
// workgroups so far.
__global__ void __launch_bounds__(kTileThreads) k_totals(const InstDesc* __restrict__ Ip, uint32_t n_acc, long long* out) {
  const InstDesc& I = *Ip;
  __shared__ long long s_red[kTileThreads / 64 * 4];
  __shared__ long long s_sum[kTileThreads / kAccSlots][2 * kAccSlots];
  if (I.wall_part) fold_walls<kTileThreads>(I, s_red);
  const uint32_t k = threadIdx.x % kAccSlots, r = threadIdx.x / kAccSlots;
  long long lo = 0, hi = 0;
#pragma unroll 8
  for (uint32_t w = r; w < n_acc; w += kTileThreads / kAccSlots) {
    const long long v = gmem(I.wg_acc)[w * kAccSlots + k];
    lo += (long long)((unsigned long long)v & 0xFFFFFFFFull);
    hi += v >> 32;
  }
  s_sum[r][2 * k] = lo;
  s_sum[r][2 * k + 1] = hi;
  __syncthreads();
  if (threadIdx.x < 2 * kAccSlots) {
    long long t = 0;
    for (uint32_t q = 0; q < kTileThreads / kAccSlots; ++q) t += s_sum[q][threadIdx.x];
    out[threadIdx.x] = t;
  }
}

// Fields of the samples (ProcessAndOutputStatistics, dsmc_base.cu:104-163), one
// lane per cell: n, u, v, w, T in double from the sums, stored as float
// [5][ncells], so that 20 bytes per cell travel to the host and not 40.
template <class T>
__global__ void __launch_bounds__(256) k_fields(const InstDesc* __restrict__ Ip, double samples, double kb, float* out) {
  const InstDesc& I = *Ip;
  const uint32_t c = blockIdx.x * 256u + threadIdx.x, C = I.ncells;
  if (c >= C) return;
  const gptr<const T> S = gmem<const T>(reinterpret_cast<const T*>(I.samp));
  const double N = S[c], sx = S[(size_t)C + c], sy = S[2 * (size_t)C + c], sz = S[3 * (size_t)C + c],
               s2 = S[4 * (size_t)C + c];
  const double fr = I.fluid_frac ? (double)I.fluid_frac[c] : 1.0;
  const double vol = (double)I.cell_volume * fr;
  const double dens = vol > 0.0 ? (double)I.fnum * N / (vol * samples) : 0.0;
  double ux = 0.0, uy = 0.0, uz = 0.0, tt = 0.0;
  if (N > 0.0) {
    ux = sx / N;
    uy = sy / N;
    uz = sz / N;
    tt = (double)I.mass * (s2 / N - (ux * ux + uy * uy + uz * uz)) / (3.0 * kb);
  }
  out[c] = (float)dens;
  out[(size_t)C + c] = (float)ux;
  out[2 * (size_t)C + c] = (float)uy;
  out[3 * (size_t)C + c] = (float)uz;
  out[4 * (size_t)C + c] = (float)tt;
}

// =================================================================== loading
// GenerateInitialVelocitiesDevBlocks / GenerateUniformVelocitiesDevBlocks
// (dsmc_kernel.cu:574-680): one thread per (x, y, i) column, i < ppc, walking
// z; stream X*Y*i + y*X + x; particle index = cell*ppc + i. Cells with a
// flagged collision-grid corner get parked particles (pos = vel = 0).
__device__ __forceinline__ bool geometry_in_cell(const InstDesc& I, float cx, float cy, float cz, float sx, float sy,
                                                 float sz) {
  // IsGeometryInCell (dsmc_kernel.cu:479-546), corners in the reference's order
  float px = cx, py = cy, pz = cz;
  uint32_t c;
#define DSMC_CORNER()                                                  \
  if ((c = cg_cell(I, px, py, pz)) != kInvalidKey && I.cg_flag[c] != 0u) \
    return true;
  DSMC_CORNER();
  px = px + sx;
  DSMC_CORNER();
  py = py + sy;
  DSMC_CORNER();
  pz = pz + sz;
  DSMC_CORNER();
  px = cx; py = cy; pz = cz;
  py = py + sy;
  DSMC_CORNER();
  pz = pz + sz;
  DSMC_CORNER();
  py = cy;
  DSMC_CORNER();
  px = px + sx;
  DSMC_CORNER();
#undef DSMC_CORNER
  return false;
}

__global__ void k_load_reference(const InstDesc* __restrict__ Ip, uint32_t par, uint32_t ppc, float sux, float suy,
                                 float suz, float temp) {
  const InstDesc& I = *Ip;
  const uint32_t X = I.dim[0], Y = I.dim[1], Z = I.dim[2];
  uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= X * Y * ppc) return;
  const uint32_t i = t / (X * Y);
  const uint32_t xy = t - i * X * Y;
  const uint32_t cy = xy / X, cx = xy - cy * X;
  const uint32_t stream = t;  // = X*Y*i + y*X + x
  Mt rng;
  mt_load(I, stream, rng);
  float cellx = I.gmin[0] + (float)cx * I.cell[0];
  float celly = I.gmin[1] + (float)cy * I.cell[1];
  const float twopi = 2.0f * kPiRef;
  for (uint32_t z = 0; z < Z; ++z) {
    uint32_t idx = (X * Y * z + cy * X + cx) * ppc + i;
    float cellz = I.gmin[2] + (float)z * I.cell[2];
    bool geom = I.has_geom && geometry_in_cell(I, cellx, celly, cellz, I.cell[0], I.cell[1], I.cell[2]);
    if (!geom) {
      // GetRandomVelocity / SampleDensityFunction (dsmc_kernel.cu:394-415)
      float vv = sqrtf(2.0f * kBoltzRef * temp / I.mass * (-dm_logf(mt_float(rng))));
      float vx = vv * dm_sinf(mt_float(rng) * twopi) + sux;
      float vy = vv * dm_sinf(mt_float(rng) * twopi) + suy;
      float vz = vv * dm_sinf(mt_float(rng) * twopi) + suz;
      // GetRandomPosition (dsmc_kernel.cu:417-427)
      float px = cellx + mt_float(rng) * I.cell[0];
      float py = celly + mt_float(rng) * I.cell[1];
      float pz = cellz + mt_float(rng) * I.cell[2];
      I.px[par][idx] = px; I.py[par][idx] = py; I.pz[par][idx] = pz;
      I.vx[par][idx] = vx; I.vy[par][idx] = vy; I.vz[par][idx] = vz;
    } else {
      I.px[par][idx] = 0.0f; I.py[par][idx] = 0.0f; I.pz[par][idx] = 0.0f;
      I.vx[par][idx] = 0.0f; I.vy[par][idx] = 0.0f; I.vz[par][idx] = 0.0f;
    }
  }
  mt_store(I, stream, rng);
}

// Move with dt = 0 after loading (include/gpu_dsmc.inl:79): box functor and
// walls on the loaded state, in place.
__global__ void k_move_zero(const InstDesc* __restrict__ Ip, uint32_t par, uint32_t n) {
  const InstDesc& I = *Ip;
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float x = I.px[par][i], y = I.py[par][i], z = I.pz[par][i];
  float ux = I.vx[par][i], uy = I.vy[par][i], uz = I.vz[par][i];
  move_reference(I, x, y, z, ux, uy, uz, 0.0f);
  I.px[par][i] = x; I.py[par][i] = y; I.pz[par][i] = z;
  I.vx[par][i] = ux; I.vy[par][i] = uy; I.vz[par][i] = uz;
}

// PHYSICS loading, pass 1: particles per cell by stochastic rounding of
// n * V_fluid / Fn (per-cell density when fields are given), plus a uniform
// random NTC remainder. Stream = cell mod n_streams, cells in increasing order.
__global__ void k_load_count(const InstDesc* __restrict__ Ip, const float* __restrict__ fn) {
  const InstDesc& I = *Ip;
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= I.n_streams) return;
  Mt rng;
  mt_load(I, s, rng);
  for (uint32_t c = s; c < I.ncells; c += I.n_streams) {
    float dens = fn ? fn[c] : I.n_inf;
    float frac = I.fluid_frac ? I.fluid_frac[c] : 1.0f;
    float lam = (float)((double)dens * (double)I.cell_volume * (double)frac / (double)I.fnum);
    float r = mt_float(rng);
    uint32_t k = frac > 0.0f ? dm_f2u_sat(lam + r) : 0u;
    I.count[c] = k;
    float2 nt = I.ntc[c];
    nt.y = mt_float(rng);
    I.ntc[c] = nt;
  }
  mt_store(I, s, rng);
}

// PHYSICS loading, pass 2: positions uniform in the cell (rejecting points in
// the body), velocities Maxwellian (Box-Muller) about the stream velocity.
__global__ void k_load_generate(const InstDesc* __restrict__ Ip, uint32_t par, const float* __restrict__ fu,
                                const float* __restrict__ fv, const float* __restrict__ fw,
                                const float* __restrict__ fT) {
  const InstDesc& I = *Ip;
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= I.n_streams) return;
  Mt rng;
  mt_load(I, s, rng);
  const float twopi = 6.28318530717958647692f;
  const uint32_t X = I.dim[0], Y = I.dim[1];
  for (uint32_t c = s; c < I.ncells; c += I.n_streams) {
    uint32_t off = I.cell_start[c], k = I.cell_start[c + 1] - off;
    if (k == 0) continue;
    uint32_t cz = c / (X * Y), rem = c - cz * X * Y, cy = rem / X, cx = rem - cy * X;
    float bx = I.gmin[0] + (float)cx * I.cell[0];
    float by = I.gmin[1] + (float)cy * I.cell[1];
    float bz = I.gmin[2] + (float)cz * I.cell[2];
    float ux = fu ? fu[c] : I.U[0], uy = fv ? fv[c] : I.U[1], uz = fw ? fw[c] : I.U[2];
    float T = fT ? fT[c] : I.T_inf;
    float sd = sqrtf((float)(kBoltz * (double)T / (double)I.mass));
    bool cut = I.fluid_frac && I.fluid_frac[c] < 1.0f;
    for (uint32_t j = 0; j < k; ++j) {
      float px, py, pz;
      int tries = 0;
      do {
        px = bx + mt_float(rng) * I.cell[0];
        py = by + mt_float(rng) * I.cell[1];
        pz = bz + mt_float(rng) * I.cell[2];
        ++tries;
      } while (cut && tries < 64 && inside_body(I, px, py, pz));
      float r1 = mt_float(rng), r2 = mt_float(rng), r3 = mt_float(rng), r4 = mt_float(rng);
      float a1 = sqrtf(-2.0f * dm_logf(r1)), a2 = sqrtf(-2.0f * dm_logf(r3));
      float s1, c1, s2, c2;
      dm_sincosf(twopi * r2, &s1, &c1);
      dm_sincosf(twopi * r4, &s2, &c2);
      uint32_t idx = off + j;
      I.px[par][idx] = px; I.py[par][idx] = py; I.pz[par][idx] = pz;
      I.vx[par][idx] = ux + sd * a1 * c1;
      I.vy[par][idx] = uy + sd * a1 * s1;
      I.vz[par][idx] = uz + sd * a2 * c2;
      I.key[par][idx] = c;
    }
  }
  mt_store(I, s, rng);
}

// ================================================================== utility
// Count particles with non-finite state or outside the box.
__global__ void k_validate(const InstDesc* __restrict__ Ip, uint32_t par, uint32_t n, uint32_t* bad) {
  const InstDesc& I = *Ip;
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (I.key[par][i] == kInvalidKey) return;
  float x = I.px[par][i], y = I.py[par][i], z = I.pz[par][i];
  float a = I.vx[par][i], b = I.vy[par][i], c = I.vz[par][i];
  bool ok = (x - x == 0.0f) && (y - y == 0.0f) && (z - z == 0.0f) && (a - a == 0.0f) && (b - b == 0.0f) &&
            (c - c == 0.0f);
  if (I.mode == kModePhysics)
    ok = ok && x >= I.gmin[0] && x <= I.gmax[0] && y >= I.gmin[1] && y <= I.gmax[1] && z >= I.gmin[2] &&
         z <= I.gmax[2];
  if (!ok) atomicAdd(bad, 1u);
}

// One extra sample of the current state (SampleCellStatistics outside the
// step, dsmc_kernel.cu:892-910): cells of the last ordering, current velocities.
__global__ void k_sample_cells(const InstDesc* __restrict__ Ip, uint32_t par, uint32_t mode) {
  const InstDesc& I = *Ip;
  uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= I.ncells) return;
  uint32_t a = I.cell_start[c], b = I.cell_start[c + 1];
  if (b <= a) return;
  const uint32_t C = I.ncells;
  const float* vx = I.vx[par];
  const float* vy = I.vy[par];
  const float* vz = I.vz[par];
  if (mode == kModeReference) {
    float* S = reinterpret_cast<float*>(I.samp);
    float sn = S[c], sx = S[C + c], sy = S[2 * C + c], sz = S[3 * C + c], s2 = S[4 * C + c];
    for (uint32_t q = a; q < b; ++q) {
      float ux = vx[q], uy = vy[q], uz = vz[q];
      sn += 1.0f; sx += ux; sy += uy; sz += uz;
      s2 += ux * ux + uy * uy + uz * uz;
    }
    S[c] = sn; S[C + c] = sx; S[2 * C + c] = sy; S[3 * C + c] = sz; S[4 * C + c] = s2;
  } else {
    double* S = I.samp;
    double sn = S[c], sx = S[C + c], sy = S[2 * C + c], sz = S[3 * C + c], s2 = S[4 * C + c];
    for (uint32_t q = a; q < b; ++q) {
      double ux = vx[q], uy = vy[q], uz = vz[q];
      sn += 1.0; sx += ux; sy += uy; sz += uz;
      s2 += ux * ux + uy * uy + uz * uz;
    }
    S[c] = sn; S[C + c] = sx; S[2 * C + c] = sy; S[3 * C + c] = sz; S[4 * C + c] = s2;
  }
}

// ================================================================ launchers
namespace dsmc_launch {

static inline uint32_t blocks_for(uint32_t n, uint32_t t) { return (n + t - 1u) / t; }

void mt_seed(uint32_t* state, const uint32_t* seeds, uint32_t n_streams, hipStream_t st) {
  if (!n_streams) return;
  hipLaunchKernelGGL(k_mt_seed, dim3(blocks_for(n_streams, 256)), dim3(256), 0, st, state, seeds, n_streams);
}

void mt_generate(const uint32_t* a, const uint32_t* b, const uint32_t* c, const uint32_t* seeds, uint32_t n_streams,
                 uint32_t n_draws, uint32_t* out, hipStream_t st) {
  if (!n_streams) return;
  hipLaunchKernelGGL(k_mt_generate, dim3(blocks_for(n_streams, 256)), dim3(256), 0, st, a, b, c, seeds, n_streams,
                     n_draws, out);
}

void cell_ids(const InstDesc& I, const float* x, const float* y, const float* z, uint32_t n, uint32_t* keys,
              hipStream_t st) {
  if (!n) return;
  hipLaunchKernelGGL(k_cell_ids, dim3(blocks_for(n, 256)), dim3(256), 0, st, I, x, y, z, n, keys);
}

void keys_count(const InstDesc* d, uint32_t par, uint32_t n, hipStream_t st) {
  if (!n) return;
  hipLaunchKernelGGL(k_keys_count, dim3(blocks_for(n, 256)), dim3(256), 0, st, d, par, n);
}

int scan(uint32_t* in, uint32_t n, uint32_t* out, uint32_t* scratch, uint32_t* total_out, hipStream_t st) {
  uint32_t tiles = blocks_for(n > 0 ? n : 1u, kScanTile);
  if (tiles > kScanMaxTiles) return -1;
  hipLaunchKernelGGL(k_scan_reduce, dim3(tiles), dim3(kScanThreads), 0, st, in, n, scratch);
  hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(kScanThreads), 0, st, scratch, tiles, total_out);
  hipLaunchKernelGGL(k_scan_apply, dim3(tiles), dim3(kScanThreads), 0, st, in, n, scratch, out, total_out);
  return 0;
}

StepScan step_scan_plan(uint32_t max_cells, uint32_t max_faces) {
  StepScan p;
  p.n_cell = blocks_for(max_cells > 0 ? max_cells : 1u, kScanTile);
  p.n_face = blocks_for(max_faces, kScanTile);
  p.small = max_cells <= kScanSmall;
  return p;
}

void step_scan(const InstDesc* d, const StepScan& p, uint32_t* ts, hipStream_t st, uint32_t n_inst) {
  if (p.small) {
    hipLaunchKernelGGL(k_scan_small, dim3(p.n_cell + p.n_face + 1, n_inst), dim3(kSmallThreads), 0, st, d, p.n_cell,
                       p.n_face, ts, p.words());
    return;
  }
  hipLaunchKernelGGL(k_scan_reduce_step, dim3(p.n_cell + p.n_face, n_inst), dim3(kScanThreads), 0, st, d, p.n_cell, ts,
                     p.words());
  hipLaunchKernelGGL(k_scan_apply_step, dim3(p.n_cell + 1, n_inst), dim3(kScanThreads), 0, st, d, p.n_cell, ts,
                     p.words());
}

uint32_t scatter_blocks(const InstDesc& I) { return I.n_scatter_wg + blocks_for(I.n_face_cells, kScanTile); }

void scatter(const InstDesc* d, uint32_t par, uint32_t blocks, const uint2* map, const StepScan& p, const uint32_t* ts,
             hipStream_t st) {
  hipLaunchKernelGGL(k_scatter, dim3(blocks), dim3(256), 0, st, d, par, map, ts + p.n_cell, p.words());
}

uint64_t op_sort_work_words(uint32_t n, uint32_t n_cells) {
  const uint64_t nb = blocks_for(n > 0 ? n : 1u, 4096u);
  return (uint64_t)n_cells + 2ull * (256ull * nb + 1ull) + (kScanMaxTiles + 1ull) + 3ull * n;
}

int op_sort(const uint32_t* keys, uint32_t n, uint32_t n_cells, uint32_t* perm, uint32_t* cell_start,
            uint32_t* work, hipStream_t st) {
  constexpr uint64_t kMost = (uint64_t)kScanMaxTiles * kScanTile;
  if ((uint64_t)n_cells > kMost || (n + 4095ull) / 4096ull * 256ull > kMost) return -1;
  // radix passes over the bits of n_cells (the largest mapped key)
  uint32_t bits = 1;
  while (bits < 32 && (n_cells >> bits) != 0u) ++bits;
  const uint32_t passes = blocks_for(bits, kRsMaxBits), per = blocks_for(bits, passes), digits = 1u << per;
  // 4096 keys per block (2^18, 2^20 and 2^25 keys of 65536 cells: 43, 56 and
  // 626 us, with 8192 54, 71 and 750), 8192 where the table does not fit the
  // workspace (at most 2^10 digits, so that of 8192 always does).
  const uint64_t words = op_sort_work_words(n, n_cells) - 3ull * n;
  const auto table_words = [&](uint32_t r) { return (uint64_t)digits * (blocks_for(n, kRsThreads * r) + 1u); };
  const bool small = table_words(4u) <= words;
  const uint32_t nb = blocks_for(n, kRsThreads * (small ? 4u : 8u));
  uint32_t* ka = work;
  uint32_t* kb = ka + n;
  uint32_t* vt = kb + n;
  uint32_t* tot = vt + n;
  uint32_t* table = tot + digits;
  const uint32_t* kin = keys;
  const uint32_t* vin = nullptr;
  for (uint32_t p = 0; p < (n ? passes : 0u); ++p) {
    const uint32_t raw = p == 0 ? 1u : 0u;
    uint32_t* kout = (p & 1u) ? kb : ka;
    uint32_t* vout = ((passes - 1u - p) & 1u) ? vt : perm;  // the last pass writes perm
    hipLaunchKernelGGL((small ? k_rs_hist<4> : k_rs_hist<8>), dim3(nb), dim3(kRsThreads), 0, st, kin, n, n_cells, raw,
                       per * p, digits, nb, table);
    hipLaunchKernelGGL(k_rs_scan, dim3(digits), dim3(kScanThreads), 0, st, table, nb, tot);
    hipLaunchKernelGGL((small ? k_rs_scatter<4> : k_rs_scatter<8>), dim3(nb), dim3(kRsThreads), 0, st, kin, vin, n,
                       n_cells, raw, per * p, per, nb, table, tot, kout, vout);
    kin = kout;
    vin = vout;
  }
  hipLaunchKernelGGL(k_rs_cells, dim3(n_cells / kRsCells + 1u), dim3(256), 0, st, kin, n, n_cells, cell_start);
  return 0;
}

uint32_t wall_blocks(const InstDesc& I) {
  return (I.defer_bits ? I.n_wall_wg : 0u) + (I.n_face_cells ? I.n_inj_wg : 0u);
}

void defer_list(const InstDesc* d, uint32_t grid, hipStream_t st, uint32_t n_inst) {
  if (grid) hipLaunchKernelGGL(k_defer_list, dim3(grid, n_inst), dim3(kTileThreads), 0, st, d);
}

void walls(const InstDesc* d, uint32_t opar, uint32_t flags, uint32_t blocks, const uint2* map, hipStream_t st) {
  if (blocks) hipLaunchKernelGGL(k_walls, dim3(blocks), dim3(kTileThreads), 0, st, d, opar, flags, map);
}

void totals(const InstDesc* d, uint32_t n_acc, long long* out, hipStream_t st) {
  hipLaunchKernelGGL(k_totals, dim3(1), dim3(kTileThreads), 0, st, d, n_acc, out);
}

void fields(const InstDesc* d, uint32_t mode, uint32_t ncells, double samples, double kb, float* out, hipStream_t st) {
  if (mode == kModePhysics)
    hipLaunchKernelGGL(k_fields<double>, dim3(blocks_for(ncells, 256)), dim3(256), 0, st, d, samples, kb, out);
  else
    hipLaunchKernelGGL(k_fields<float>, dim3(blocks_for(ncells, 256)), dim3(256), 0, st, d, samples, kb, out);
}

void tile(uint32_t mode, bool narrow, const InstDesc* d, uint32_t par, uint32_t flags, uint32_t blocks,
          const uint2* map, hipStream_t st) {
  if (!blocks) return;
  const auto k = mode == kModeReference ? (narrow ? k_tile<kModeReference, true> : k_tile<kModeReference, false>)
                                        : (narrow ? k_tile<kModePhysics, true> : k_tile<kModePhysics, false>);
  hipLaunchKernelGGL(k, dim3(blocks), dim3(kTileThreads), 0, st, d, par, flags, map);
}

void load_reference(const InstDesc* d, uint32_t par, uint32_t ppc, uint32_t n_threads, float sux, float suy,
                    float suz, float temp, hipStream_t st) {
  if (!n_threads) return;
  hipLaunchKernelGGL(k_load_reference, dim3(blocks_for(n_threads, 128)), dim3(128), 0, st, d, par, ppc, sux, suy,
                     suz, temp);
}

void move_zero(const InstDesc* d, uint32_t par, uint32_t n, hipStream_t st) {
  if (!n) return;
  hipLaunchKernelGGL(k_move_zero, dim3(blocks_for(n, 256)), dim3(256), 0, st, d, par, n);
}

void load_count(const InstDesc* d, uint32_t n_streams, const float* fn, hipStream_t st) {
  hipLaunchKernelGGL(k_load_count, dim3(blocks_for(n_streams, 256)), dim3(256), 0, st, d, fn);
}

void load_generate(const InstDesc* d, uint32_t par, uint32_t n_streams, const float* fu, const float* fv,
                   const float* fw, const float* fT, hipStream_t st) {
  hipLaunchKernelGGL(k_load_generate, dim3(blocks_for(n_streams, 256)), dim3(256), 0, st, d, par, fu, fv, fw, fT);
}

void sample_cells(const InstDesc* d, uint32_t par, uint32_t mode, uint32_t ncells, hipStream_t st) {
  if (!ncells) return;
  hipLaunchKernelGGL(k_sample_cells, dim3(blocks_for(ncells, 256)), dim3(256), 0, st, d, par, mode);
}

void validate(const InstDesc* d, uint32_t par, uint32_t n, uint32_t* bad, hipStream_t st) {
  if (!n) return;
  hipLaunchKernelGGL(k_validate, dim3(blocks_for(n, 256)), dim3(256), 0, st, d, par, n, bad);
}

}  // namespace dsmc_launch
