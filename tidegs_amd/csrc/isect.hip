// Gaussian-tile intersection: per-Gaussian tile counts, key/id emission and
// per-(camera, tile) offset encoding.
//
// Reference: gsplat/cuda/csrc/isect_tiles.cu:14-98 (kernel), :100-232 (host),
// :234-301 (offset encode).
//   tile rect  [floor(x/ts - r/ts), ceil(x/ts + r/ts)) clamped to the grid
//   key        cam << (32 + tile_bits) | tile << 32 | int32 bits of depth
//              (sign-extended to 64 bits, as the reference does)
//   flatten id index into [C*N] (non-packed) or [nnz] (packed)
//   offsets    offsets[c, tile] = first isect index of that (camera, tile) run;
//              empty tiles take the next run's start; trailing tiles take n.
#include "tgs_common.cuh"

#include <algorithm>

// scan_sort.hip
extern "C" size_t tgs_scan_workspace_size(uint64_t n);
extern "C" int tgs_exclusive_scan_u32(const uint32_t* in, uint32_t* out, uint64_t n,
                                      void* workspace, size_t workspace_bytes,
                                      hipStream_t stream);
extern "C" size_t tgs_segmented_sort_workspace_size(uint64_t n, uint32_t n_segments);
extern "C" int tgs_segmented_sort_pairs_u32(uint32_t* keys, void* vals, uint32_t* keys_alt,
                                            void* vals_alt, uint32_t value_bytes, uint64_t n,
                                            uint32_t n_segments, const uint32_t* seg_offsets,
                                            int begin_bit, int end_bit, void* workspace,
                                            size_t workspace_bytes, int* selector,
                                            hipStream_t stream);
extern "C" int tgs_segmented_sort_pairs_u32_range(uint32_t* keys, void* vals, uint32_t* keys_alt,
                                                  void* vals_alt, uint32_t value_bytes, uint64_t n,
                                                  uint32_t n_segments,
                                                  const uint32_t* seg_offsets, uint32_t key_base,
                                                  int key_bits, void* workspace,
                                                  size_t workspace_bytes, int* selector,
                                                  hipStream_t stream);
// tide_step.hip
extern "C" uint32_t tgs_tide_isect_fused_digit_bits(uint32_t tile_n_bits);
extern "C" uint64_t tgs_tide_isect_fused_hist_words(uint32_t C, const uint32_t* cam_offsets,
                                                    uint32_t tile_n_bits);
extern "C" uint64_t tgs_tide_isect_fused_used_words(uint32_t C, const uint32_t* cam_offsets,
                                                    uint32_t tile_n_bits);
extern "C" int tgs_tide_isect_fused_count(uint32_t C, const uint32_t* cam_offsets,
                                          const uint64_t* entry_rects, uint32_t tile_width,
                                          uint32_t tile_n_bits, uint32_t* hist,
                                          uint64_t hist_words, hipStream_t stream);
extern "C" int tgs_tide_isect_fused_scatter(uint32_t C, const uint32_t* cam_offsets,
                                            const uint64_t* entry_rects, uint32_t tile_width,
                                            uint32_t tile_n_bits, const uint32_t* hist_scan,
                                            uint64_t hist_words, uint32_t n_isects,
                                            uint32_t* keys, int32_t* flatten_ids,
                                            hipStream_t stream);

struct TileRect {
  uint32_t x0, y0, x1, y1;
};

// Clamp a floor/ceil value into [0, limit] the way the reference's unsigned
// conversion followed by min/max does for finite inputs.
__device__ __forceinline__ uint32_t clamp_tile(float v, uint32_t limit) {
  if (!(v > 0.f)) return 0u;  // negatives (and NaN) saturate to 0
  if (v >= (float)limit) return limit;
  return (uint32_t)v;
}

__device__ __forceinline__ TileRect tile_rect(float mx, float my, int32_t radius, uint32_t tile_size,
                                              uint32_t tw, uint32_t th) {
  const float ts = (float)tile_size;
  const float tr = (float)radius / ts;
  const float tx = mx / ts;
  const float ty = my / ts;
  TileRect r;
  r.x0 = clamp_tile(floorf(tx - tr), tw);
  r.y0 = clamp_tile(floorf(ty - tr), th);
  r.x1 = clamp_tile(ceilf(tx + tr), tw);
  r.y1 = clamp_tile(ceilf(ty + tr), th);
  return r;
}

__device__ __forceinline__ uint32_t tile_count(const TileRect& r) {
  return (r.x1 > r.x0 ? r.x1 - r.x0 : 0u) * (r.y1 > r.y0 ? r.y1 - r.y0 : 0u);
}

__global__ void __launch_bounds__(256) isect_count_kernel(
    uint64_t total, const float* __restrict__ means2d, const int32_t* __restrict__ radii,
    uint32_t tile_size, uint32_t tw, uint32_t th, int32_t* __restrict__ tiles_per_gauss) {
  const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int32_t radius = radii[idx];
  if (radius <= 0) {
    tiles_per_gauss[idx] = 0;
    return;
  }
  const TileRect r = tile_rect(means2d[idx * 2], means2d[idx * 2 + 1], radius, tile_size, tw, th);
  tiles_per_gauss[idx] = (int32_t)tile_count(r);
}

// One Gaussian's keys and ids, rows of its rectangle in order, from `cur` on.
__device__ __forceinline__ void emit_keys(int64_t cur, uint64_t idx, const TileRect& r, int64_t cid,
                                          float depth, uint32_t tw, uint32_t tile_n_bits,
                                          int64_t* __restrict__ isect_ids,
                                          int32_t* __restrict__ flatten_ids) {
  const int64_t cam_enc = cid << (32 + tile_n_bits);
  const int64_t depth_enc = (int64_t)__float_as_int(depth);  // sign-extended
  for (uint32_t y = r.y0; y < r.y1; ++y) {
    for (uint32_t x = r.x0; x < r.x1; ++x) {
      const int64_t tile = (int64_t)y * tw + x;
      isect_ids[cur] = cam_enc | (tile << 32) | depth_enc;
      flatten_ids[cur] = (int32_t)idx;
      ++cur;
    }
  }
}

__global__ void __launch_bounds__(256) isect_emit_kernel(
    uint64_t total, uint32_t N, const int64_t* __restrict__ camera_ids,
    const float* __restrict__ means2d, const int32_t* __restrict__ radii,
    const float* __restrict__ depths, const int64_t* __restrict__ cum_tiles, uint32_t tile_size,
    uint32_t tw, uint32_t th, uint32_t tile_n_bits, int64_t* __restrict__ isect_ids,
    int32_t* __restrict__ flatten_ids) {
  const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int32_t radius = radii[idx];
  if (radius <= 0) return;
  emit_keys(idx == 0 ? 0 : cum_tiles[idx - 1], idx,
            tile_rect(means2d[idx * 2], means2d[idx * 2 + 1], radius, tile_size, tw, th),
            camera_ids ? camera_ids[idx] : (int64_t)(idx / N), depths[idx], tw, tile_n_bits,
            isect_ids, flatten_ids);
}

// Offsets by search: bucket b = (camera, tile) gets the index of the first sorted
// key of its own or a later bucket, i.e. an empty bucket takes the next occupied
// one's start and buckets after the last key take n_isects, as the reference's
// scatter from the run starts writes them.  A key's bucket is computed from its
// signed high word as there: a negative depth's sign fills the word, and such a
// key counts where the formula puts it, not past the last bucket.  One thread per
// bucket, a branch-free binary search with a uniform trip count.  One thread per
// key, writing the run of empty buckets before its own, took 9 us for 2.7M keys of
// 4293 tiles and 31 us for 1.4M where one thread met a long run (the empty rows
// above a scene): 6 us in both here.
// Word: int32_t where the tile bits leave the camera some of the signed word (any
// bucket of such a word then fits it too), else int64_t.
template <typename Word>
__global__ void __launch_bounds__(256) isect_offset_search_kernel(
    uint64_t n_isects, const int64_t* __restrict__ isect_ids, uint64_t n_buckets, uint32_t n_tiles,
    uint32_t tile_n_bits, uint64_t top, int32_t* __restrict__ offsets) {
  const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_buckets) return;
  const Word tmask = (Word)(((int64_t)1 << tile_n_bits) - 1), tiles = (Word)n_tiles;
  uint64_t pos = 0;  // keys [0, pos) lie in buckets before b
  for (uint64_t step = top; step != 0u; step >>= 1) {
    const uint64_t p = pos + step;
    if (p > n_isects) continue;
    const Word hi = (Word)(isect_ids[p - 1] >> 32);
    if ((int64_t)((hi >> tile_n_bits) * tiles + (hi & tmask)) < (int64_t)b) pos = p;
  }
  offsets[b] = (int32_t)pos;
}

// ---------------------------------------------------------------------------
// Counts and offsets by block.  The reference scans every Gaussian's tile count
// into a 64-bit array that the emission reads back (16 bytes per Gaussian
// moved, three launches: 20 of the 300 us of 1.2M Gaussians and 2.7M
// intersections).  Here a block of IB_ENTRIES Gaussians keeps one sum: the plan
// writes the counts the caller asks for and the block's sum and depth range,
// one workgroup scans the sums, and the emission recovers each Gaussian's offset
// from its block's.
// ---------------------------------------------------------------------------
#define IB_ENTRIES 256

struct IsectBlock {
  int64_t sum;       // intersections; after the scan, those of the blocks before
  uint32_t entries;  // Gaussians with any; after the scan, those of the blocks before
  uint32_t kmin;     // their depth bits: the least ...
  uint32_t kmax;     // ... and greatest, as unsigned (0xffffffff, 0 where none)
  uint32_t pad;
};

// The Gaussian of this thread: each camera takes blocks_per_cam blocks, so that no block spans
// two cameras.  False past the camera's last.
__device__ __forceinline__ bool isect_block_entry(uint64_t N, uint32_t blocks_per_cam,
                                                  uint64_t& idx) {
  const uint32_t cam = blockIdx.x / blocks_per_cam;
  const uint64_t local = (uint64_t)(blockIdx.x - cam * blocks_per_cam) * IB_ENTRIES + threadIdx.x;
  idx = (uint64_t)cam * N + local;
  return local < N;
}

__global__ void __launch_bounds__(IB_ENTRIES) isect_plan_kernel(
    uint64_t N, uint32_t blocks_per_cam, const float* __restrict__ means2d,
    const int32_t* __restrict__ radii, const float* __restrict__ depths, uint32_t tile_size,
    uint32_t tw, uint32_t th, int32_t* __restrict__ tiles_per_gauss,
    IsectBlock* __restrict__ blocks) {
  __shared__ IsectBlock s_w[IB_ENTRIES / 64];
  uint64_t idx;
  uint32_t n = 0u, key = 0u;
  if (isect_block_entry(N, blocks_per_cam, idx)) {
    const int32_t radius = radii[idx];
    if (radius > 0) {
      n = tile_count(
          tile_rect(means2d[idx * 2], means2d[idx * 2 + 1], radius, tile_size, tw, th));
      if (n) key = (uint32_t)__float_as_int(depths[idx]);
    }
    tiles_per_gauss[idx] = (int32_t)n;
  }
  int64_t sum = (int32_t)n;
  uint32_t kmin = n ? key : 0xffffffffu, kmax = n ? key : 0u;
  const uint32_t any = (uint32_t)__popcll(tgs_ballot(n != 0u));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
    kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, off, 64));
    kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, off, 64));
  }
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = IsectBlock{sum, any, kmin, kmax, 0u};
  __syncthreads();
  if (threadIdx.x == 0) {
    IsectBlock b = s_w[0];
#pragma unroll
    for (int w = 1; w < IB_ENTRIES / 64; ++w) {
      b.sum += s_w[w].sum;
      b.entries += s_w[w].entries;
      b.kmin = min(b.kmin, s_w[w].kmin);
      b.kmax = max(b.kmax, s_w[w].kmax);
    }
    blocks[blockIdx.x] = b;
  }
}

// Exclusive scan of the blocks' sums in place by one workgroup, and the whole:
// summary = {intersections, kmin | kmax << 32} and, for every camera, {entries,
// intersections} up to its end.
#define IB_SCAN_THREADS 1024
#define IB_SCAN_ITEMS 4
__global__ void __launch_bounds__(IB_SCAN_THREADS) isect_plan_scan_kernel(
    uint32_t n_blocks, uint32_t blocks_per_cam, IsectBlock* __restrict__ blocks,
    uint64_t* __restrict__ summary) {
  constexpr int WAVES = IB_SCAN_THREADS / 64;
  __shared__ int64_t s_sum[WAVES];
  __shared__ uint32_t s_ent[WAVES], s_min[WAVES], s_max[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t sum_carry = 0;
  uint32_t ent_carry = 0u, kmin = 0xffffffffu, kmax = 0u;
  for (uint32_t base = 0; base < n_blocks; base += IB_SCAN_THREADS * IB_SCAN_ITEMS) {
    const uint32_t i0 = base + threadIdx.x * IB_SCAN_ITEMS;
    IsectBlock b[IB_SCAN_ITEMS];
    int64_t sum = 0;
    uint32_t ent = 0u;
#pragma unroll
    for (int k = 0; k < IB_SCAN_ITEMS; ++k) {
      b[k] = i0 + k < n_blocks ? blocks[i0 + k] : IsectBlock{0, 0u, 0xffffffffu, 0u, 0u};
      kmin = min(kmin, b[k].kmin);
      kmax = max(kmax, b[k].kmax);
      sum += b[k].sum;
      ent += b[k].entries;
    }
    int64_t sum_inc = sum;
    uint32_t ent_inc = ent;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int64_t o = __shfl_up(sum_inc, off, 64);
      const uint32_t e = __shfl_up(ent_inc, off, 64);
      if (lane >= off) {
        sum_inc += o;
        ent_inc += e;
      }
    }
    if (lane == 63) {
      s_sum[wave] = sum_inc;
      s_ent[wave] = ent_inc;
    }
    __syncthreads();
    int64_t sum_run = sum_carry + sum_inc - sum;
    uint32_t ent_run = ent_carry + ent_inc - ent;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      if (w < wave) {
        sum_run += s_sum[w];
        ent_run += s_ent[w];
      }
      sum_carry += s_sum[w];
      ent_carry += s_ent[w];
    }
#pragma unroll
    for (int k = 0; k < IB_SCAN_ITEMS; ++k) {
      if (i0 + k >= n_blocks) break;
      blocks[i0 + k].sum = sum_run;
      blocks[i0 + k].entries = ent_run;
      sum_run += b[k].sum;
      ent_run += b[k].entries;
      const uint32_t cam = (i0 + k) / blocks_per_cam;
      if (i0 + k + 1 == (cam + 1) * blocks_per_cam) {
        summary[2 + 2 * cam] = ent_run;
        summary[3 + 2 * cam] = (uint64_t)sum_run;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, off, 64));
    kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, off, 64));
  }
  if (lane == 0) {
    s_min[wave] = kmin;
    s_max[wave] = kmax;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      kmin = min(kmin, s_min[w]);
      kmax = max(kmax, s_max[w]);
    }
    summary[0] = (uint64_t)sum_carry;
    summary[1] = (uint64_t)kmin | ((uint64_t)kmax << 32);
  }
}

__global__ void __launch_bounds__(IB_ENTRIES) isect_emit_blocks_kernel(
    uint64_t plan_n, uint32_t blocks_per_cam, uint64_t N, const int64_t* __restrict__ camera_ids,
    const float* __restrict__ means2d, const int32_t* __restrict__ radii,
    const float* __restrict__ depths, const int32_t* __restrict__ tiles_per_gauss,
    const IsectBlock* __restrict__ blocks, uint32_t tile_size, uint32_t tw, uint32_t th,
    uint32_t tile_n_bits, int64_t* __restrict__ isect_ids, int32_t* __restrict__ flatten_ids) {
  __shared__ int64_t s_w[IB_ENTRIES / 64];
  uint64_t idx;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int32_t n = isect_block_entry(plan_n, blocks_per_cam, idx) ? tiles_per_gauss[idx] : 0;
  int64_t inc = n;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t o = __shfl_up(inc, off, 64);
    if (lane >= off) inc += o;
  }
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  int64_t cur = blocks[blockIdx.x].sum + inc - n;
  for (int w = 0; w < wave; ++w) cur += s_w[w];
  if (n == 0) return;
  emit_keys(cur, idx, tile_rect(means2d[idx * 2], means2d[idx * 2 + 1], radii[idx], tile_size, tw, th),
            camera_ids ? camera_ids[idx] : (int64_t)(idx / N), depths[idx], tw, tile_n_bits,
            isect_ids, flatten_ids);
}

// The cameras the two sorts take (one segment of the sorts and of the fused
// emission each); a plan for more is laid out as one camera of them all, so that
// many small cameras still fill their blocks.
#define IB_MAX_CAMS 32

struct IsectGrid {
  uint32_t cams, per_cam;
  uint64_t n;
};

static IsectGrid isect_grid(uint32_t C, uint64_t N) {
  const uint32_t cams = C <= IB_MAX_CAMS ? C : 1u;
  const uint64_t n = C <= IB_MAX_CAMS ? N : (uint64_t)C * N;
  return IsectGrid{cams, tgs_blocks(n, IB_ENTRIES), n};
}

static int isect_plan_check(const char* who, uint32_t C, uint64_t N) {
  TGS_CHECK_ARG(C > 0 && N > 0, "%s: nothing to plan", who);
  TGS_CHECK_ARG((uint64_t)C * N < (1ull << 31),
                "isect_tiles: C*N (or nnz) must fit int32 flatten ids");
  return TGS_OK;
}

// No less than for fewer cameras or Gaussians (up to IB_MAX_CAMS cameras each end on
// a block of their own).
extern "C" uint64_t tgs_isect_tiles_plan_size(uint32_t C, uint64_t N) {
  const IsectGrid g = isect_grid(C, N);
  const uint64_t own = (uint64_t)std::min(C, (uint32_t)IB_MAX_CAMS) * tgs_blocks(N, IB_ENTRIES);
  return std::max((uint64_t)g.cams * g.per_cam, own) * sizeof(IsectBlock);
}

extern "C" int tgs_isect_tiles_plan(uint32_t C, uint64_t N, const float* means2d,
                                    const int32_t* radii, const float* depths, uint32_t tile_size,
                                    uint32_t tile_width, uint32_t tile_height,
                                    int32_t* tiles_per_gauss, void* plan, size_t plan_bytes,
                                    uint64_t* summary, hipStream_t stream) {
  int rc = isect_plan_check("isect_tiles_plan", C, N);
  if (rc) return rc;
  TGS_CHECK_ARG(means2d && radii && depths && tiles_per_gauss && plan && summary &&
                    ((uintptr_t)plan & 7u) == 0,
                "isect_tiles_plan: null pointer (or a plan not 8-byte aligned)");
  TGS_CHECK_ARG(tile_size > 0, "tile_size must be > 0");
  if (plan_bytes < tgs_isect_tiles_plan_size(C, N)) {
    tgs_set_error("isect_tiles_plan: plan buffer too small");
    return TGS_ERR_WORKSPACE;
  }
  const IsectGrid g = isect_grid(C, N);
  hipLaunchKernelGGL(isect_plan_kernel, dim3(g.cams * g.per_cam), dim3(IB_ENTRIES), 0, stream, g.n,
                     g.per_cam, means2d, radii, depths, tile_size, tile_width, tile_height, tiles_per_gauss,
                     (IsectBlock*)plan);
  TGS_LAUNCH_CHECK("isect_plan");
  hipLaunchKernelGGL(isect_plan_scan_kernel, dim3(1), dim3(IB_SCAN_THREADS), 0, stream,
                     g.cams * g.per_cam, g.per_cam, (IsectBlock*)plan, summary);
  TGS_RETURN_LAUNCH("tgs_isect_tiles_plan");
}

extern "C" int tgs_isect_tiles_emit_plan(uint32_t C, uint64_t N, const int64_t* camera_ids,
                                         const float* means2d, const int32_t* radii,
                                         const float* depths, const int32_t* tiles_per_gauss,
                                         const void* plan, uint32_t tile_size,
                                         uint32_t tile_width, uint32_t tile_height,
                                         uint32_t tile_n_bits, int64_t* isect_ids,
                                         int32_t* flatten_ids, hipStream_t stream) {
  int rc = isect_plan_check("isect_tiles_emit_plan", C, N);
  if (rc) return rc;
  TGS_CHECK_ARG(means2d && radii && depths && tiles_per_gauss && plan && isect_ids && flatten_ids,
                "isect_tiles_emit_plan: null pointer");
  TGS_CHECK_ARG(tile_size > 0, "tile_size must be > 0");
  const IsectGrid g = isect_grid(C, N);
  hipLaunchKernelGGL(isect_emit_blocks_kernel, dim3(g.cams * g.per_cam), dim3(IB_ENTRIES), 0, stream, g.n,
                     g.per_cam, N, camera_ids, means2d, radii, depths, tiles_per_gauss,
                     (const IsectBlock*)plan, tile_size, tile_width, tile_height, tile_n_bits,
                     isect_ids, flatten_ids);
  TGS_RETURN_LAUNCH("tgs_isect_tiles_emit_plan");
}

extern "C" uint32_t tgs_bit_width(uint32_t v) {
  uint32_t b = 0;
  while (v) {
    ++b;
    v >>= 1;
  }
  return b;
}

// ---------------------------------------------------------------------------
// The reference's order in two sorts: Gaussians by depth (32-bit keys), then the
// intersections they emit in that order by tile, stably, gives (camera, tile,
// depth, Gaussian) with two 8-byte moves per intersection instead of the single
// sort's five 12-byte ones (both measured at the rule below).  The single sort takes
// what this does not: packed camera ids (in any order), grids past 255 tiles a side
// (8-bit rectangles), more cameras than the emission's segments, negative depths
// (their sign fills the id).
// ---------------------------------------------------------------------------
// Depth keys and tile rectangles (x0 | x1 << 8 | y0 << 16 | y1 << 24, above the
// index) of the Gaussians that meet any tile, in order.
__global__ void __launch_bounds__(IB_ENTRIES) isect_entries_kernel(
    uint64_t N, uint32_t blocks_per_cam, const float* __restrict__ means2d,
    const int32_t* __restrict__ radii, const float* __restrict__ depths, uint32_t tile_size,
    uint32_t tw, uint32_t th, const IsectBlock* __restrict__ blocks, uint32_t* __restrict__ keys,
    uint64_t* __restrict__ rects) {
  __shared__ uint32_t s_w[IB_ENTRIES / 64];
  uint64_t idx;
  TileRect r{0u, 0u, 0u, 0u};
  if (isect_block_entry(N, blocks_per_cam, idx)) {
    const int32_t radius = radii[idx];
    if (radius > 0)
      r = tile_rect(means2d[idx * 2], means2d[idx * 2 + 1], radius, tile_size, tw, th);
  }
  const bool any = tile_count(r) != 0u;
  const uint64_t m = tgs_ballot(any);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) s_w[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  if (!any) return;
  uint32_t pos = blocks[blockIdx.x].entries + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
  for (int w = 0; w < wave; ++w) pos += s_w[w];
  keys[pos] = (uint32_t)__float_as_int(depths[idx]);
  rects[pos] = (uint64_t)(r.x0 | (r.x1 << 8) | (r.y0 << 16) | (r.y1 << 24)) << 32 | (uint32_t)idx;
}

// The 64-bit ids of sorted camera | tile keys; the flatten ids too where the sort
// left them in scratch.
__global__ void __launch_bounds__(256) isect_rebuild_ids_kernel(
    uint32_t n, const uint32_t* __restrict__ keys, const int32_t* fids,
    const float* __restrict__ depths, int64_t* __restrict__ isect_ids, int32_t* flatten_ids) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t f = fids[i];
  isect_ids[i] = ((int64_t)keys[i] << 32) | (int64_t)__float_as_int(depths[f]);
  if (flatten_ids != fids) flatten_ids[i] = f;
}

struct IsectSorted {
  uint32_t V, n, tile_bits;  // entries, intersections, bit width of the tile count
  uint32_t ent[IB_MAX_CAMS + 1], isect[IB_MAX_CAMS + 1];
  uint64_t hist_words, dkeys, dkeys2, rects, hist, scan, keys, keys2, fids2, sort_ws, scan_ws, end;
  size_t sort_bytes, scan_bytes;
};

// False where the two sorts do not apply.
static bool isect_sorted_layout(uint32_t C, const uint64_t* summary, uint32_t tile_width,
                                uint32_t tile_height, IsectSorted& o) {
  if (!summary || C == 0 || C > IB_MAX_CAMS || tile_width == 0 || tile_height == 0 || tile_width > 255 ||
      tile_height > 255 || summary[0] == 0 || summary[0] >= (1ull << 31) || summary[1] >> 63)
    return false;
  o = IsectSorted{};
  o.tile_bits = tgs_bit_width(tile_width * tile_height);
  for (uint32_t c = 0; c < C; ++c) {
    o.ent[c + 1] = (uint32_t)summary[2 + 2 * c];
    o.isect[c + 1] = (uint32_t)summary[3 + 2 * c];
  }
  o.V = o.ent[C];
  o.n = o.isect[C];
  // Two sorts move each Gaussian once per depth pass and each intersection twice,
  // one sort every intersection five times (six with several cameras' bits): two win
  // where the intersections outnumber the Gaussians by enough, and past the sizes at
  // which either is launches only (one sort of few keys has fewer).  Few Gaussians of
  // many tiles are few blocks of the fused emission, each a serial chain.
  // isect_tiles in two sorts and in one, in us, by Gaussians and tiles of each:
  //   1 camera
  //   3000     1.6 88 77, 3.2 88 80, 5 89 82      2000 of 16 99 113, of 61 196 138
  //   12k      1.6 91 85, 3.2 97 99, 5 97 99      10k of 16 109 124, of 61 200 169
  //   40k      1.6 110 101, 3.2 112 103, 5 113 107       40k of 61 239 255
  //   130k     1.6 124 117, 2.5 126 126, 3.2 128 131, 5 131 146
  //   500k     1.3 153 150, 1.6 153 154, 2 156 168, 3.2 167 186, 5 177 223
  //   1.5M     1.3 238 208, 1.6 248 229, 2 255 238, 2.5 269 326, 5 321 455
  //   4M       1.3 448 390, 1.6 475 427, 2 511 495, 2.5 566 605, 5 805 1199
  //   4 cameras, Gaussians of all
  //   5000     1.6 88 81, 3.2 89 85, 5 89 92
  //   12k      1.3 89 85, 2 89 91, 3.2 90 104
  //   40k      1.3 96 107, 3.2 98 112             500k 1.3 147 166, 3.2 161 194
  //   4M       1.3 392 396, 2 432 501, 5 670 1210
  const bool few = o.V < (1u << 15);
  if (few && (o.V < 2048u || o.n > 32ull * o.V)) return false;
  if (C > 1 ? o.n < (3u << 13) : few ? o.n < 8ull * o.V : o.n < (3u << 17) || o.n < 2ull * o.V)
    return false;
  o.hist_words = tgs_tide_isect_fused_used_words(C, o.ent, o.tile_bits);
  if (o.hist_words == 0 || o.n != summary[0]) return false;
  o.sort_bytes = std::max(tgs_segmented_sort_workspace_size(o.V, C),
                          tgs_segmented_sort_workspace_size(o.n, C));
  // (buffers that also hold every smaller call's)
  const uint64_t hist_most = tgs_tide_isect_fused_hist_words(C, o.ent, o.tile_bits);
  o.scan_bytes = tgs_scan_workspace_size(hist_most);
  uint64_t at = 0;
  auto take = [&](uint64_t bytes) {
    const uint64_t a = at;
    at += (bytes + 255) & ~255ull;
    return a;
  };
  o.dkeys = take(4ull * o.V);
  o.dkeys2 = take(4ull * o.V);
  o.rects = take(8ull * o.V);
  o.hist = take(4 * hist_most);
  o.scan = take(4 * hist_most);
  o.keys = take(4ull * o.n);
  o.keys2 = take(4ull * o.n);
  o.fids2 = take(4ull * o.n);
  o.sort_ws = take(o.sort_bytes);
  o.scan_ws = take(o.scan_bytes);
  o.end = at;
  return true;
}

extern "C" uint64_t tgs_isect_tiles_sorted_workspace_size(uint32_t C, const uint64_t* summary,
                                                          uint32_t tile_width,
                                                          uint32_t tile_height) {
  IsectSorted o;
  return isect_sorted_layout(C, summary, tile_width, tile_height, o) ? o.end : 0;
}

extern "C" int tgs_isect_tiles_sorted(uint32_t C, uint64_t N, const float* means2d,
                                      const int32_t* radii, const float* depths, const void* plan,
                                      const uint64_t* summary, uint32_t tile_size,
                                      uint32_t tile_width, uint32_t tile_height,
                                      int64_t* isect_ids, int32_t* flatten_ids, void* workspace,
                                      size_t workspace_bytes, hipStream_t stream) {
  int rc = isect_plan_check("isect_tiles_sorted", C, N);
  if (rc) return rc;
  IsectSorted o;
  TGS_CHECK_ARG(isect_sorted_layout(C, summary, tile_width, tile_height, o),
                "isect_tiles_sorted: not for these cameras, tiles or depths");
  TGS_CHECK_ARG(means2d && radii && depths && plan && isect_ids && flatten_ids && workspace,
                "isect_tiles_sorted: null pointer");
  TGS_CHECK_ARG(tile_size > 0, "tile_size must be > 0");
  TGS_CHECK_ARG((uint64_t)o.V <= (uint64_t)C * N, "isect_tiles_sorted: not this plan's summary");
  if (workspace_bytes < o.end) {
    tgs_set_error("isect_tiles_sorted: workspace %zu < %llu", workspace_bytes,
                  (unsigned long long)o.end);
    return TGS_ERR_WORKSPACE;
  }
  char* w = (char*)workspace;
  uint32_t *dkeys = (uint32_t*)(w + o.dkeys), *dkeys2 = (uint32_t*)(w + o.dkeys2);
  uint64_t *rects = (uint64_t*)(w + o.rects), *rects2 = (uint64_t*)isect_ids;  // V <= n
  uint32_t *hist = (uint32_t*)(w + o.hist), *scan = (uint32_t*)(w + o.scan);
  uint32_t *keys = (uint32_t*)(w + o.keys), *keys2 = (uint32_t*)(w + o.keys2);
  int32_t *fids = (int32_t*)(w + o.fids2), *fids2 = flatten_ids;
  const IsectGrid g = isect_grid(C, N);
  hipLaunchKernelGGL(isect_entries_kernel, dim3(g.cams * g.per_cam), dim3(IB_ENTRIES), 0, stream, g.n,
                     g.per_cam, means2d, radii, depths, tile_size, tile_width, tile_height,
                     (const IsectBlock*)plan, dkeys, rects);
  TGS_LAUNCH_CHECK("isect_entries");
  const uint32_t kmin = (uint32_t)summary[1], kmax = (uint32_t)(summary[1] >> 32);
  int sel = 0;
  rc = tgs_segmented_sort_pairs_u32_range(dkeys, rects, dkeys2, rects2, 8, o.V, C, o.ent, kmin,
                                          (int)std::max(1u, tgs_bit_width(kmax - kmin)),
                                          w + o.sort_ws, o.sort_bytes, &sel, stream);
  if (rc) return rc;
  if (sel) rects = rects2;
  if ((rc = tgs_tide_isect_fused_count(C, o.ent, rects, tile_width, o.tile_bits, hist,
                                       o.hist_words, stream)))
    return rc;
  if ((rc = tgs_exclusive_scan_u32(hist, scan, o.hist_words, w + o.scan_ws, o.scan_bytes, stream)))
    return rc;
  if ((rc = tgs_tide_isect_fused_scatter(C, o.ent, rects, tile_width, o.tile_bits, scan,
                                         o.hist_words, o.n, keys, fids, stream)))
    return rc;
  const int first = (int)tgs_tide_isect_fused_digit_bits(o.tile_bits);
  if ((int)o.tile_bits > first) {
    sel = 0;
    rc = tgs_segmented_sort_pairs_u32(keys, fids, keys2, fids2, 4, o.n, C, o.isect, first,
                                      (int)o.tile_bits, w + o.sort_ws, o.sort_bytes, &sel, stream);
    if (rc) return rc;
    if (sel) {
      keys = keys2;
      fids = fids2;
    }
  }
  hipLaunchKernelGGL(isect_rebuild_ids_kernel, dim3(tgs_blocks(o.n, 256)), dim3(256), 0, stream,
                     o.n, keys, fids, depths, isect_ids, flatten_ids);
  TGS_RETURN_LAUNCH("tgs_isect_tiles_sorted");
}

extern "C" int tgs_isect_tiles_count(uint64_t total, const float* means2d, const int32_t* radii,
                                     uint32_t tile_size, uint32_t tile_width,
                                     uint32_t tile_height, int32_t* tiles_per_gauss,
                                     hipStream_t stream) {
  if (total == 0) return TGS_OK;
  TGS_CHECK_ARG(means2d && radii && tiles_per_gauss, "isect_tiles_count: null pointer");
  TGS_CHECK_ARG(tile_size > 0, "tile_size must be > 0");
  TGS_CHECK_ARG(total < (1ull << 31), "isect_tiles: C*N (or nnz) must fit int32 flatten ids");
  hipLaunchKernelGGL(isect_count_kernel, dim3(tgs_blocks(total, 256)), dim3(256), 0, stream,
                     total, means2d, radii, tile_size, tile_width, tile_height, tiles_per_gauss);
  TGS_RETURN_LAUNCH("tgs_isect_tiles_count");
}

// camera_ids: [total] int64 for packed inputs, or null with N = Gaussians per
// camera for [C, N] inputs.
extern "C" int tgs_isect_tiles_emit(uint64_t total, uint32_t N, const int64_t* camera_ids,
                                    const float* means2d, const int32_t* radii,
                                    const float* depths, const int64_t* cum_tiles_per_gauss,
                                    uint32_t tile_size, uint32_t tile_width, uint32_t tile_height,
                                    uint32_t tile_n_bits, int64_t* isect_ids,
                                    int32_t* flatten_ids, hipStream_t stream) {
  if (total == 0) return TGS_OK;
  TGS_CHECK_ARG(means2d && radii && depths && cum_tiles_per_gauss && isect_ids && flatten_ids,
                "isect_tiles_emit: null pointer");
  TGS_CHECK_ARG(camera_ids || N > 0, "isect_tiles_emit: need camera_ids or N");
  hipLaunchKernelGGL(isect_emit_kernel, dim3(tgs_blocks(total, 256)), dim3(256), 0, stream, total,
                     N, camera_ids, means2d, radii, depths, cum_tiles_per_gauss, tile_size,
                     tile_width, tile_height, tile_n_bits, isect_ids, flatten_ids);
  TGS_RETURN_LAUNCH("tgs_isect_tiles_emit");
}

extern "C" int tgs_isect_offset_encode(uint64_t n_isects, const int64_t* isect_ids, uint32_t C,
                                       uint32_t tile_width, uint32_t tile_height,
                                       int32_t* offsets, hipStream_t stream) {
  const uint64_t total = (uint64_t)C * tile_width * tile_height;
  if (total == 0) return TGS_OK;
  TGS_CHECK_ARG(offsets != nullptr, "isect_offset_encode: null offsets");
  if (n_isects == 0) {
    // reference: offsets.fill_(0) (isect_tiles.cu:298)
    return tgs_fill_u32(offsets, total, 0u, stream);
  }
  TGS_CHECK_ARG(isect_ids != nullptr, "isect_offset_encode: null isect_ids");
  const uint32_t n_tiles = tile_width * tile_height;
  const uint32_t tile_n_bits = tgs_bit_width(n_tiles);
  uint64_t top = 1;
  while (top <= n_isects / 2) top <<= 1;
  hipLaunchKernelGGL(tile_n_bits < 31 ? isect_offset_search_kernel<int32_t>
                                      : isect_offset_search_kernel<int64_t>,
                     dim3(tgs_blocks(total, 256)), dim3(256), 0, stream, n_isects, isect_ids, total,
                     n_tiles, tile_n_bits, top, offsets);
  TGS_RETURN_LAUNCH("tgs_isect_offset_encode");
}
