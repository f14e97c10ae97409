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
// key whose high word is >= its own (camera << tile_n_bits | tile), i.e. an empty
// bucket takes the next occupied one's start and buckets after the last key take
// n_isects, as the reference's scatter from the run starts writes them.  One
// thread per bucket, a branch-free binary search with a uniform trip count.  One
// thread per key, writing the run of empty buckets before its own, took 9 us for
// 2.7M keys of 4293 tiles and 31 us for 1.4M where one thread met a long run
// (the empty rows above a scene): 6 us in both here.
__global__ void __launch_bounds__(256) isect_offset_search_kernel(
    uint64_t n_isects, const uint64_t* __restrict__ isect_ids, uint64_t n_buckets, uint32_t n_tiles,
    uint32_t tile_n_bits, uint64_t top, int32_t* __restrict__ offsets) {
  const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n_buckets) return;
  const uint64_t cam = b / n_tiles;
  const uint64_t kb = (cam << tile_n_bits) | (b - cam * n_tiles);
  uint64_t pos = 0;  // keys [0, pos) lie in buckets before b
  for (uint64_t step = top; step != 0u; step >>= 1) {
    const uint64_t p = pos + step;
    if (p <= n_isects && (isect_ids[p - 1] >> 32) < kb) pos = p;
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
  int64_t sum;    // intersections; after the scan, those of the blocks before
  uint32_t kmin;  // depth bits of the Gaussians with any: the least ...
  uint32_t kmax;  // ... and greatest, as unsigned (0xffffffff, 0 where none)
};

__global__ void __launch_bounds__(IB_ENTRIES) isect_plan_kernel(
    uint64_t total, const float* __restrict__ means2d, const int32_t* __restrict__ radii,
    const float* __restrict__ depths, uint32_t tile_size, uint32_t tw, uint32_t th,
    int32_t* __restrict__ tiles_per_gauss, IsectBlock* __restrict__ blocks) {
  __shared__ IsectBlock s_w[IB_ENTRIES / 64];
  const uint64_t idx = (uint64_t)blockIdx.x * IB_ENTRIES + threadIdx.x;
  uint32_t n = 0u, key = 0u;
  if (idx < total) {
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
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
    kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, off, 64));
    kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, off, 64));
  }
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = IsectBlock{sum, kmin, kmax};
  __syncthreads();
  if (threadIdx.x == 0) {
    IsectBlock b = s_w[0];
#pragma unroll
    for (int w = 1; w < IB_ENTRIES / 64; ++w) {
      b.sum += s_w[w].sum;
      b.kmin = min(b.kmin, s_w[w].kmin);
      b.kmax = max(b.kmax, s_w[w].kmax);
    }
    blocks[blockIdx.x] = b;
  }
}

// Exclusive scan of the blocks' sums in place by one workgroup, and the whole
// range: summary = {intersections, kmin | kmax << 32}.
#define IB_SCAN_THREADS 1024
__global__ void __launch_bounds__(IB_SCAN_THREADS) isect_plan_scan_kernel(
    uint32_t n_blocks, IsectBlock* __restrict__ blocks, uint64_t* __restrict__ summary) {
  constexpr int WAVES = IB_SCAN_THREADS / 64;
  __shared__ int64_t s_sum[WAVES];
  __shared__ uint32_t s_min[WAVES], s_max[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t carry = 0;
  uint32_t kmin = 0xffffffffu, kmax = 0u;
  for (uint32_t base = 0; base < n_blocks; base += IB_SCAN_THREADS) {
    const uint32_t i = base + threadIdx.x;
    const IsectBlock b = i < n_blocks ? blocks[i] : IsectBlock{0, 0xffffffffu, 0u};
    kmin = min(kmin, b.kmin);
    kmax = max(kmax, b.kmax);
    int64_t inc = b.sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int64_t o = __shfl_up(inc, off, 64);
      if (lane >= off) inc += o;
    }
    if (lane == 63) s_sum[wave] = inc;
    __syncthreads();
    int64_t before = carry;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      if (w < wave) before += s_sum[w];
      carry += s_sum[w];
    }
    if (i < n_blocks) blocks[i].sum = before + inc - b.sum;
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
    summary[0] = (uint64_t)carry;
    summary[1] = (uint64_t)kmin | ((uint64_t)kmax << 32);
  }
}

__global__ void __launch_bounds__(IB_ENTRIES) isect_emit_blocks_kernel(
    uint64_t total, uint32_t N, const int64_t* __restrict__ camera_ids,
    const float* __restrict__ means2d, const int32_t* __restrict__ radii,
    const float* __restrict__ depths, const int32_t* __restrict__ tiles_per_gauss,
    const IsectBlock* __restrict__ blocks, uint32_t tile_size, uint32_t tw, uint32_t th,
    uint32_t tile_n_bits, int64_t* __restrict__ isect_ids, int32_t* __restrict__ flatten_ids) {
  __shared__ int64_t s_w[IB_ENTRIES / 64];
  const uint64_t idx = (uint64_t)blockIdx.x * IB_ENTRIES + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int32_t n = idx < total ? tiles_per_gauss[idx] : 0;
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

extern "C" uint64_t tgs_isect_tiles_plan_size(uint64_t total) {
  return (total + IB_ENTRIES - 1) / IB_ENTRIES * sizeof(IsectBlock);
}

extern "C" int tgs_isect_tiles_plan(uint64_t total, const float* means2d, const int32_t* radii,
                                    const float* depths, uint32_t tile_size, uint32_t tile_width,
                                    uint32_t tile_height, int32_t* tiles_per_gauss, void* plan,
                                    size_t plan_bytes, uint64_t* summary, hipStream_t stream) {
  TGS_CHECK_ARG(total > 0, "isect_tiles_plan: nothing to plan");
  TGS_CHECK_ARG(means2d && radii && depths && tiles_per_gauss && plan && summary &&
                    ((uintptr_t)plan & 15u) == 0,
                "isect_tiles_plan: null pointer (or a plan not 16-byte aligned)");
  TGS_CHECK_ARG(tile_size > 0, "tile_size must be > 0");
  TGS_CHECK_ARG(total < (1ull << 31), "isect_tiles: C*N (or nnz) must fit int32 flatten ids");
  if (plan_bytes < tgs_isect_tiles_plan_size(total)) {
    tgs_set_error("isect_tiles_plan: plan buffer too small");
    return TGS_ERR_WORKSPACE;
  }
  const uint32_t nb = tgs_blocks(total, IB_ENTRIES);
  hipLaunchKernelGGL(isect_plan_kernel, dim3(nb), dim3(IB_ENTRIES), 0, stream, total, means2d,
                     radii, depths, tile_size, tile_width, tile_height, tiles_per_gauss,
                     (IsectBlock*)plan);
  TGS_LAUNCH_CHECK("isect_plan");
  hipLaunchKernelGGL(isect_plan_scan_kernel, dim3(1), dim3(IB_SCAN_THREADS), 0, stream, nb,
                     (IsectBlock*)plan, summary);
  TGS_RETURN_LAUNCH("tgs_isect_tiles_plan");
}

extern "C" int tgs_isect_tiles_emit_plan(uint64_t total, uint32_t N, const int64_t* camera_ids,
                                         const float* means2d, const int32_t* radii,
                                         const float* depths, const int32_t* tiles_per_gauss,
                                         const void* plan, uint32_t tile_size,
                                         uint32_t tile_width, uint32_t tile_height,
                                         uint32_t tile_n_bits, int64_t* isect_ids,
                                         int32_t* flatten_ids, hipStream_t stream) {
  if (total == 0) return TGS_OK;
  TGS_CHECK_ARG(means2d && radii && depths && tiles_per_gauss && plan && isect_ids && flatten_ids,
                "isect_tiles_emit_plan: null pointer");
  TGS_CHECK_ARG(camera_ids || N > 0, "isect_tiles_emit_plan: need camera_ids or N");
  hipLaunchKernelGGL(isect_emit_blocks_kernel, dim3(tgs_blocks(total, IB_ENTRIES)),
                     dim3(IB_ENTRIES), 0, stream, total, N, camera_ids, means2d, radii, depths,
                     tiles_per_gauss, (const IsectBlock*)plan, tile_size, tile_width, tile_height,
                     tile_n_bits, isect_ids, flatten_ids);
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
  hipLaunchKernelGGL(isect_offset_search_kernel, dim3(tgs_blocks(total, 256)), dim3(256), 0, stream,
                     n_isects, (const uint64_t*)isect_ids, total, n_tiles, tile_n_bits, top,
                     offsets);
  TGS_RETURN_LAUNCH("tgs_isect_offset_encode");
}
