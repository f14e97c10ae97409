// Device-wide scan and stable LSD radix sort of (uint64 key, uint32 value)
// pairs, written for wave64.
//
// The tile-intersection sort (gsplat isect_tiles.cu:189-227 calls
// cub::DeviceRadixSort::SortPairs on bits [0, 32+tile_bits+cam_bits)) needs a
// stable ascending sort on a bit range of the key.  Because every flatten id
// appears at most once per (camera, tile) key prefix, "stable on the key bits"
// equals "ascending in (key bits, input position)", a total order, so any
// correct stable sort reproduces the reference output bit for bit.
//
// Scan: up to SCAN_ONE_BLOCK_MAX values in one workgroup; above, reduce-then-
// scan in three kernels (block sums, one-block scan of the sums, per-block
// rescan), no inter-block spin-waits.
// Radix pass (<= 8-bit digit, tiles of 256 threads x ITEMS keys):
//   hist      per-tile digit histogram
//   scan      exclusive scan of the histogram (large sorts only: a small
//             sort's scatter adds up the counts before its tile by itself)
//   scatter   per-tile stable ranking (ballot matching + per-wave counters),
//             LDS reorder, coalesced write of each digit run.
#include <mutex>

#include "tgs_common.cuh"

#define SCAN_THREADS 256
#define SCAN_ITEMS 16
#define SCAN_CHUNK (SCAN_THREADS * SCAN_ITEMS)

#define SORT_THREADS 256
#define SORT_ITEMS 16  // keys per thread of a large sort
#define SORT_TILE (SORT_THREADS * SORT_ITEMS)
#define SORT_BINS 256
#define RADIX_MAX_SEGS 64

// ---------------------------------------------------------------------------
// Block-level exclusive scan of one value per thread (256 threads, 4 waves).
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* s_wave, T& total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  T inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    T o = __shfl_up(inc, off, 64);
    if (lane >= off) inc += o;
  }
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  T wave_base = 0;
  T tot = 0;
#pragma unroll
  for (int w = 0; w < SCAN_THREADS / 64; ++w) {
    const T s = s_wave[w];
    if (w < wave) wave_base += s;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return wave_base + inc - v;
}

template <typename InT, typename OutT>
__global__ void __launch_bounds__(SCAN_THREADS) scan_reduce_kernel(const InT* __restrict__ in,
                                                                   uint64_t n,
                                                                   OutT* __restrict__ sums) {
  __shared__ OutT s_wave[SCAN_THREADS / 64];
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_CHUNK;
  OutT acc = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint64_t i = base + (uint64_t)k * SCAN_THREADS + threadIdx.x;
    if (i < n) acc += (OutT)in[i];
  }
  OutT total;
  (void)block_exclusive_scan<OutT>(acc, s_wave, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// In-place exclusive scan of `n` block sums by one block: each thread scans a
// contiguous run of the sums, one block-wide scan joins the runs.
template <typename OutT>
__global__ void __launch_bounds__(SCAN_THREADS) scan_sums_kernel(OutT* __restrict__ sums,
                                                                 uint64_t n) {
  __shared__ OutT s_wave[SCAN_THREADS / 64];
  const uint64_t per = (n + SCAN_THREADS - 1) / SCAN_THREADS;
  const uint64_t b0 = (uint64_t)threadIdx.x * per;
  const uint64_t b1 = b0 + per < n ? b0 + per : n;
  OutT run = 0;
  for (uint64_t i = b0; i < b1; ++i) run += sums[i];
  OutT total;
  OutT carry = block_exclusive_scan<OutT>(run, s_wave, total);
  for (uint64_t i = b0; i < b1; ++i) {
    const OutT v = sums[i];
    sums[i] = carry;
    carry += v;
  }
}

// Wave-level inclusive scan (wave64, shuffles).
template <typename T>
__device__ __forceinline__ T wave_inclusive_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const T o = __shfl_up(v, off, 64);
    if (lane >= off) v += o;
  }
  return v;
}

// Striped arrangement: wave w of the block owns items [w*64*ITEMS, (w+1)*64*ITEMS)
// of the chunk in rounds of 64 consecutive items, so every load and store of
// a round is one contiguous span.
template <typename InT, typename OutT, bool INCLUSIVE>
__global__ void __launch_bounds__(SCAN_THREADS) scan_apply_kernel(const InT* __restrict__ in,
                                                                  uint64_t n,
                                                                  const OutT* __restrict__ sums,
                                                                  OutT* __restrict__ out) {
  __shared__ OutT s_wtot[SCAN_THREADS / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t wbase = (uint64_t)blockIdx.x * SCAN_CHUNK + (uint64_t)wave * 64 * SCAN_ITEMS;
  OutT vals[SCAN_ITEMS];
  OutT acc = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint64_t i = wbase + (uint64_t)k * 64 + lane;
    vals[k] = i < n ? (OutT)in[i] : (OutT)0;
    acc += vals[k];
  }
  // wave total -> exclusive prefix of the waves before this one
  OutT wt = acc;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) wt += __shfl_xor(wt, off, 64);
  if (lane == 0) s_wtot[wave] = wt;
  __syncthreads();
  OutT carry = sums[blockIdx.x];
  for (int w = 0; w < wave; ++w) carry += s_wtot[w];
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const OutT inc = wave_inclusive_scan<OutT>(vals[k]);
    const uint64_t i = wbase + (uint64_t)k * 64 + lane;
    if (i < n) out[i] = carry + (INCLUSIVE ? inc : inc - vals[k]);
    carry += __shfl(inc, 63, 64);
  }
}

// The whole scan in one 1024-thread workgroup, SCAN_ONE_ITEMS consecutive
// values per thread.  The three-kernel form spends its time in launches when the
// array is short (a pass's histogram, the per-block counts of a few hundred
// thousand rows): 1000 values 9.0 us in three launches and 3.5 in one, 4096 10.3
// and 5.3, 8192 10.5 and 8.7.  A second round of the one workgroup costs what
// three launches do: 10k values 10.7 and 10.7, 16k 10.8 and 16.1.
#define SCAN_ONE_THREADS 1024
#define SCAN_ONE_ITEMS 8
#define SCAN_ONE_BLOCK_MAX (SCAN_ONE_THREADS * SCAN_ONE_ITEMS)

template <typename InT, typename OutT, bool INCLUSIVE>
__global__ void __launch_bounds__(SCAN_ONE_THREADS) scan_one_block_kernel(
    const InT* __restrict__ in, uint32_t n, OutT* __restrict__ out) {
  __shared__ OutT s_wave[SCAN_ONE_THREADS / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t i0 = threadIdx.x * SCAN_ONE_ITEMS;
  OutT vals[SCAN_ONE_ITEMS];
  OutT sum = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ONE_ITEMS; ++k) {
    vals[k] = i0 + k < n ? (OutT)in[i0 + k] : (OutT)0;
    sum += vals[k];
  }
  const OutT inc = wave_inclusive_scan<OutT>(sum);
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  OutT run = inc - sum;
#pragma unroll
  for (int w = 0; w < SCAN_ONE_THREADS / 64; ++w) {
    const OutT t = s_wave[w];
    if (w < wave) run += t;
  }
#pragma unroll
  for (int k = 0; k < SCAN_ONE_ITEMS; ++k) {
    if (INCLUSIVE) run += vals[k];
    if (i0 + k < n) out[i0 + k] = run;
    if (!INCLUSIVE) run += vals[k];
  }
}

static uint64_t scan_blocks(uint64_t n) { return (n + SCAN_CHUNK - 1) / SCAN_CHUNK; }

template <typename InT, typename OutT, bool INCLUSIVE>
static int launch_scan(const InT* in, OutT* out, uint64_t n, OutT* sums, hipStream_t stream) {
  if (n == 0) return TGS_OK;
  if (n <= SCAN_ONE_BLOCK_MAX) {
    hipLaunchKernelGGL((scan_one_block_kernel<InT, OutT, INCLUSIVE>), dim3(1),
                       dim3(SCAN_ONE_THREADS), 0, stream, in, (uint32_t)n, out);
    TGS_RETURN_LAUNCH("scan");
  }
  const uint64_t nb = scan_blocks(n);
  hipLaunchKernelGGL((scan_reduce_kernel<InT, OutT>), dim3((unsigned)nb), dim3(SCAN_THREADS), 0,
                     stream, in, n, sums);
  hipLaunchKernelGGL((scan_sums_kernel<OutT>), dim3(1), dim3(SCAN_THREADS), 0, stream, sums, nb);
  hipLaunchKernelGGL((scan_apply_kernel<InT, OutT, INCLUSIVE>), dim3((unsigned)nb),
                     dim3(SCAN_THREADS), 0, stream, in, n, sums, out);
  TGS_RETURN_LAUNCH("scan");
}

extern "C" size_t tgs_scan_workspace_size(uint64_t n) {
  return (size_t)(scan_blocks(n) + 1) * sizeof(int64_t);
}

// out[i] = sum(in[0..i]) (int32 in, int64 out), as torch.cumsum does in
// isect_tiles.cu:165.
extern "C" int tgs_inclusive_scan_i32_i64(const int32_t* in, int64_t* out, uint64_t n,
                                          void* workspace, size_t workspace_bytes,
                                          hipStream_t stream) {
  if (n == 0) return TGS_OK;
  TGS_CHECK_ARG(in && out && workspace, "inclusive_scan: null pointer");
  if (workspace_bytes < tgs_scan_workspace_size(n)) {
    tgs_set_error("inclusive_scan: workspace %zu < %zu bytes", workspace_bytes,
                  tgs_scan_workspace_size(n));
    return TGS_ERR_WORKSPACE;
  }
  return launch_scan<int32_t, int64_t, true>(in, out, n, (int64_t*)workspace, stream);
}

// Exclusive scan of uint32 -> uint32 (radix histograms, compaction).
static int exclusive_scan_u32(const uint32_t* in, uint32_t* out, uint64_t n, void* ws,
                              hipStream_t stream) {
  return launch_scan<uint32_t, uint32_t, false>(in, out, n, (uint32_t*)ws, stream);
}

extern "C" int tgs_exclusive_scan_u32(const uint32_t* in, uint32_t* out, uint64_t n,
                                      void* workspace, size_t workspace_bytes,
                                      hipStream_t stream) {
  if (n == 0) return TGS_OK;
  TGS_CHECK_ARG(in && out && workspace, "exclusive_scan_u32: null pointer");
  if (workspace_bytes < tgs_scan_workspace_size(n)) {
    tgs_set_error("exclusive_scan_u32: workspace too small");
    return TGS_ERR_WORKSPACE;
  }
  return exclusive_scan_u32(in, out, n, workspace, stream);
}

// ---------------------------------------------------------------------------
// Radix sort
//
// Segmented LSD passes: the key range [0, n) is split into segments (one for
// a plain sort; one per camera for the fused step, where entries and
// intersections are already grouped by camera) and tiles never straddle a
// segment, so one pass sorts every segment independently.
//
// A pass needs, per (tile, digit), the output slot of the digit's first key:
// the segment's start, plus the segment's keys of smaller digits, plus the
// keys of this digit in the segment's earlier tiles.
//   Large sorts: the histogram is laid out [segment][digit][tile of segment]
//   and its exclusive scan (three more launches) is that slot.
//   Small sorts (LOCAL, at most RADIX_LOCAL_KEYS keys): the histogram is laid
//   out [tile][digit] and the scatter adds its tile's column up by itself,
//   from one row per RADIX_GROUP earlier tiles (summed by the histogram
//   kernel's atomics) and the rows since.  A pass is two launches, not five:
//   the scan's three kernels take 11-16 us of a pass whose histogram and
//   scatter take 15 us at 10k keys and 25 us at 2.7M.  Above the line the
//   scatters' row sums cost more than the scan: with 64-bit keys as soon as the
//   768 workgroups that the chip holds at once (3 per CU by their LDS) do not
//   take every tile, with 32-bit ones later.  Whole sorts, with the scan and
//   without, in us:
//     46 bits of 64-bit keys, 4-byte values  10k 134 -> 58, 300k 169 -> 115,
//                                            2.7M 235 -> 221, 3.14M 242 -> 228,
//                                            3.3M 279 -> 305, 4.1M 303 -> 343
//     25 bits of 32-bit keys, 8-byte values  10k 87 -> 34, 300k 112 -> 56,
//                                            2.7M 148 -> 115, 4.1M 177 -> 164
// ---------------------------------------------------------------------------
#define RADIX_GROUP 32
#define RADIX_LOCAL_KEYS(key_bytes) ((key_bytes) == 8 ? 3u << 20 : 1u << 22)

struct RadixSegs {
  uint32_t n;                             // number of segments (>= 1)
  uint32_t key_off[RADIX_MAX_SEGS + 1];   // key_off[0] = 0, key_off[n] = n_keys
  uint32_t tile_base[RADIX_MAX_SEGS + 1]; // first tile of each segment
  // first group of RADIX_GROUP tiles of each segment (LOCAL passes)
  uint32_t group_base[RADIX_MAX_SEGS + 1];
  // 32-bit keys are ranked as min(key - key_base, key_cap) (keys below the
  // base as 0): an order-preserving map of a key range onto its low bits, with
  // every key past the range tied at key_cap.  (0, ~0) ranks the keys as they are.
  uint32_t key_base = 0, key_cap = 0xffffffffu;
  // 64-bit keys are ranked as (high word << low_bits) | (low word - key_base): low
  // words known to lie in [key_base, key_base + 2^low_bits) take no more bits
  // than their range.  (0, 32) ranks the keys as they are.
  uint32_t low_bits = 32;
};

struct TileRange {
  uint32_t start, count;  // keys [start, start + count)
  uint32_t seg, t, nts;   // segment, tile within it, tiles of it
};

template <uint32_t TILE>
__device__ __forceinline__ TileRange radix_tile(const RadixSegs& sg, uint32_t b) {
  uint32_t lo = 0, hi = sg.n;  // largest s with tile_base[s] <= b
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (sg.tile_base[mid] <= b) lo = mid;
    else hi = mid;
  }
  TileRange r;
  r.seg = lo;
  r.t = b - sg.tile_base[lo];
  r.nts = sg.tile_base[lo + 1] - sg.tile_base[lo];
  r.start = sg.key_off[lo] + r.t * TILE;
  const uint32_t end = sg.key_off[lo + 1];
  r.count = end > r.start ? min(TILE, end - r.start) : 0u;
  return r;
}

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K key, const RadixSegs& sg, int shift,
                                            uint32_t mask) {
  if constexpr (sizeof(K) == 4) {
    // max-then-subtract is a clamped (saturating) subtract; the same select
    // written as (k < base ? 0 : min(k - base, cap)) compiles for gfx950 to an
    // unclamped subtract, so keys below the base would wrap
    const uint32_t r = min(max((uint32_t)key, sg.key_base) - sg.key_base, sg.key_cap);
    return (r >> shift) & mask;
  } else {
    const uint64_t r = ((uint64_t)key >> 32 << sg.low_bits) | ((uint32_t)key - sg.key_base);
    return (uint32_t)(r >> shift) & mask;
  }
}

// nbins: the pass's digit count (1 << bits); the histogram holds nbins counts
// per tile.  LOCAL: hist[tile][digit], and each count is added to its group's
// row of group_hist [group][digit] (zeroed by the caller; null where no segment
// has more than one group).
template <typename K, int ITEMS, bool LOCAL>
__global__ void __launch_bounds__(SORT_THREADS) radix_hist_kernel(const K* __restrict__ keys,
                                                                  RadixSegs sg, int shift,
                                                                  uint32_t mask, uint32_t nbins,
                                                                  uint32_t* __restrict__ hist,
                                                                  uint32_t* __restrict__ group_hist) {
  __shared__ uint32_t s_h[SORT_THREADS / 64][SORT_BINS];
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int w = 0; w < SORT_THREADS / 64; ++w) s_h[w][threadIdx.x] = 0;
  __syncthreads();
  const TileRange tr = radix_tile<SORT_THREADS * ITEMS>(sg, blockIdx.x);
  // A wavefront whose keys share one digit (common for the high digits of
  // sorted-ish keys) adds its count once instead of 64 conflicting atomics.
  // all of the thread's keys are loaded before any is counted, so the tile's
  // loads are in flight together
  K kr[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t i = (uint32_t)r * SORT_THREADS + threadIdx.x;
    kr[r] = i < tr.count ? keys[tr.start + i] : (K)0;
  }
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t i = (uint32_t)r * SORT_THREADS + threadIdx.x;
    const bool valid = i < tr.count;
    const uint32_t d = valid ? digit_of(kr[r], sg, shift, mask) : 0u;
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
    const uint64_t vm = tgs_ballot(valid);
    const uint64_t same = tgs_ballot(valid && d == d0);
    if (same == vm) {
      if ((threadIdx.x & 63) == 0 && vm) atomicAdd(&s_h[wave][d0], (uint32_t)__popcll(vm));
    } else if (valid) {
      atomicAdd(&s_h[wave][d], 1u);
    }
  }
  __syncthreads();
  uint32_t c = 0;
#pragma unroll
  for (int w = 0; w < SORT_THREADS / 64; ++w) c += s_h[w][threadIdx.x];
  // only the pass's digits: a narrower pass stores (and scans) fewer counts,
  // each a line of its own in the [digit][tile] layout
  if (threadIdx.x < nbins) {
    if (LOCAL) {
      hist[blockIdx.x * nbins + threadIdx.x] = c;
      if (group_hist && c)
        atomicAdd(&group_hist[(sg.group_base[tr.seg] + tr.t / RADIX_GROUP) * nbins + threadIdx.x],
                  c);
    } else {
      hist[sg.tile_base[tr.seg] * nbins + tr.t + threadIdx.x * tr.nts] = c;
    }
  }
}

// One tile of 256 x ITEMS keys per block.  Wave w owns 64 x ITEMS consecutive
// keys of the tile in rounds of 64; for each round 8 ballots give a lane the lanes of
// its wave with the same digit, and a per-wave digit counter in LDS carries
// the count of earlier rounds.  The tile is then scattered into LDS in
// (digit, position) order and written out by consecutive threads, so each
// digit's run of the tile is one contiguous store.
template <typename K, typename V, int ITEMS, bool LOCAL>
__global__ void __launch_bounds__(SORT_THREADS) __attribute__((amdgpu_waves_per_eu(4))) radix_scatter_kernel(
    const K* __restrict__ keys_in, const V* __restrict__ vals_in, RadixSegs sg, int shift,
    uint32_t mask, uint32_t nbins, const uint32_t* __restrict__ hist,
    const uint32_t* __restrict__ group_hist, K* __restrict__ keys_out, V* __restrict__ vals_out) {
  constexpr int WAVES = SORT_THREADS / 64;
  constexpr uint32_t TILE = SORT_THREADS * ITEMS;
  __shared__ K s_k[TILE];
  __shared__ V s_v[TILE];
  // per-wave digit counters, then each (wave, digit)'s first position in the
  // tile (counts and positions stay below the tile size: 16 bits, so the 8-byte
  // value form's LDS lets 3 workgroups share a CU)
  __shared__ uint16_t s_wh[WAVES][SORT_BINS];
  __shared__ uint32_t s_gofs[SORT_BINS];
  __shared__ uint64_t s_scan[WAVES];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const uint64_t lt_mask = (1ull << lane) - 1ull;
  const TileRange tr = radix_tile<TILE>(sg, blockIdx.x);
#pragma unroll
  for (int w = 0; w < WAVES; ++w) s_wh[w][threadIdx.x] = 0;

  K k[ITEMS];
  V v[ITEMS];
  uint32_t rk[ITEMS];
  const uint32_t wbase = (uint32_t)wave * 64u * ITEMS;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t li = wbase + (uint32_t)r * 64u + lane;
    if (li < tr.count) {
      k[r] = keys_in[tr.start + li];
      v[r] = vals_in[tr.start + li];
    } else {
      k[r] = 0;
      v[r] = 0;
    }
  }
  // LOCAL: this thread's share of digit (thread mod nbins)'s column: the
  // segment's keys of the digit, and those in the tiles before this one
  uint32_t seg_total = 0, before_tile = 0;
  if (LOCAL) {
    const uint32_t d = threadIdx.x & mask, parts = SORT_THREADS / nbins;
    const uint32_t p = threadIdx.x / nbins;
    const uint32_t* rows = hist + (uint64_t)sg.tile_base[tr.seg] * nbins + d;
    uint32_t r0 = 0;
    if (group_hist) {
      const uint32_t* groups = group_hist + (uint64_t)sg.group_base[tr.seg] * nbins + d;
      const uint32_t ng = sg.group_base[tr.seg + 1] - sg.group_base[tr.seg];
      const uint32_t tg = tr.t / RADIX_GROUP;
#pragma unroll 8
      for (uint32_t g = p; g < ng; g += parts) {
        const uint32_t c = groups[g * nbins];
        seg_total += c;
        before_tile += g < tg ? c : 0u;
      }
      r0 = tg * RADIX_GROUP;
    }
    const uint32_t r1 = group_hist ? tr.t : tr.nts;
#pragma unroll 8
    for (uint32_t r = r0 + p; r < r1; r += parts) {
      const uint32_t c = rows[r * nbins];
      seg_total += group_hist ? 0u : c;
      before_tile += r < tr.t ? c : 0u;
    }
    uint32_t* s_part = reinterpret_cast<uint32_t*>(s_k);  // 2 x 256 words, before the reorder
    static_assert(sizeof(s_k) >= 2 * SORT_THREADS * 4, "the tile holds the partial sums");
    s_part[threadIdx.x] = seg_total;
    s_part[SORT_THREADS + threadIdx.x] = before_tile;
    __syncthreads();
    seg_total = before_tile = 0;
    if (threadIdx.x < nbins) {
      for (uint32_t q = threadIdx.x; q < SORT_THREADS; q += nbins) {
        seg_total += s_part[q];
        before_tile += s_part[SORT_THREADS + q];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t li = wbase + (uint32_t)r * 64u + lane;
    const bool valid = li < tr.count;
    const uint32_t d = digit_of(k[r], sg, shift, mask);
    uint64_t peers = tgs_ballot(valid);
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
    if (tgs_ballot(valid && d == d0) != peers) {  // else every valid lane shares d0
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t m = tgs_ballot(bit);
        peers &= bit ? m : ~m;
      }
    }
    const uint32_t before = s_wh[wave][d];
    __builtin_amdgcn_wave_barrier();
    // the highest lane of each digit group advances the wave's counter
    if (valid && (peers >> lane) == 1ull) s_wh[wave][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
    __builtin_amdgcn_wave_barrier();
    rk[r] = before + (uint32_t)__popcll(peers & lt_mask);
  }
  __syncthreads();
  // thread t owns digit t: per-wave counts, tile total, tile start, then each
  // wave's first position of the digit in the tile
  uint32_t cw[WAVES];
  uint32_t tot = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    cw[w] = s_wh[w][threadIdx.x];
    tot += cw[w];
  }
  uint32_t st, first;  // digit's first position in the tile; its first output slot
  if (LOCAL) {
    // one scan for both: the tile's counts in the low word (their sum stays
    // below the tile size), the segment's in the high word
    uint64_t all;
    const uint64_t ex =
        block_exclusive_scan<uint64_t>(((uint64_t)seg_total << 32) | tot, s_scan, all);
    st = (uint32_t)ex;
    first = sg.key_off[tr.seg] + (uint32_t)(ex >> 32) + before_tile;
  } else {
    uint32_t all;
    st = block_exclusive_scan<uint32_t>(tot, reinterpret_cast<uint32_t*>(s_scan), all);
    first = threadIdx.x < nbins
                ? hist[sg.tile_base[tr.seg] * nbins + tr.t + threadIdx.x * tr.nts] : st;
  }
  uint32_t run = st;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    s_wh[w][threadIdx.x] = (uint16_t)run;
    run += cw[w];
  }
  // digits past nbins never occur in this pass
  s_gofs[threadIdx.x] = first - st;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const uint32_t li = wbase + (uint32_t)r * 64u + lane;
    if (li < tr.count) {
      const uint32_t d = digit_of(k[r], sg, shift, mask);
      const uint32_t pos = (uint32_t)s_wh[wave][d] + rk[r];
      s_k[pos] = k[r];
      s_v[pos] = v[r];
    }
  }
  __syncthreads();
  for (uint32_t j = threadIdx.x; j < tr.count; j += SORT_THREADS) {
    const K kk = s_k[j];
    const uint32_t o = s_gofs[digit_of(kk, sg, shift, mask)] + j;
    keys_out[o] = kk;
    vals_out[o] = s_v[j];
  }
}

// Keys per thread: a small sort takes quarter tiles (1024 keys), so that it
// spreads over four times the CUs and each workgroup's chain of ranking rounds
// is a quarter as long (300k keys: 129 -> 108 us with 64-bit keys, 74 -> 56
// with 32-bit ones).  From a workgroup per CU and more on, the longer digit runs
// of whole tiles win: with 64-bit keys at 1.2M (172 against 164 us), with
// 32-bit ones later (1.2M 82 against 97, 2.7M 157 against 113).
#define SORT_ITEMS_SMALL 4
static uint64_t sort_small_line(uint32_t key_bytes) { return key_bytes == 8 ? 1u << 20 : 3u << 19; }
static uint32_t sort_items(uint64_t n, uint32_t key_bytes) {
  return n < sort_small_line(key_bytes) ? SORT_ITEMS_SMALL : SORT_ITEMS;
}

// Most tiles a sort of n keys in n_segments segments can have (a caller's
// precounted first pass takes SORT_TILE tiles: no more than these).
static uint64_t sort_tiles_max(uint64_t n, uint32_t key_bytes, uint64_t n_segments) {
  const uint64_t tile = (uint64_t)SORT_THREADS * sort_items(n, key_bytes);
  return (n + tile - 1) / tile + n_segments;
}

static size_t radix_workspace(uint64_t tiles) {
  const uint64_t hist = tiles * SORT_BINS;
  // hist + scanned hist + scan block sums, each 256-byte aligned.
  auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
  return (size_t)(al(hist * 4) * 2 + al(tgs_scan_workspace_size(hist)));
}

// What a sort of n keys takes, and what it and every sort of fewer keys (in no more
// segments) takes: a workspace sized once for the largest sort serves them all.  The
// sorts below the line take quarter tiles, so the largest of them counts too (2 MB
// of histograms with 64-bit keys, 3 MB with 32-bit ones).
static size_t sort_workspace(uint64_t n, uint32_t key_bytes, uint64_t n_segments) {
  return radix_workspace(sort_tiles_max(n, key_bytes, n_segments));
}
static size_t sort_workspace_up_to(uint64_t n, uint32_t key_bytes, uint64_t n_segments) {
  const uint64_t line = sort_small_line(key_bytes);
  const size_t own = sort_workspace(n, key_bytes, n_segments);
  const size_t small = n < line ? 0 : sort_workspace(line - 1, key_bytes, n_segments);
  return own > small ? own : small;
}

extern "C" size_t tgs_radix_sort_workspace_size(uint64_t n) { return sort_workspace_up_to(n, 8, 0); }

extern "C" size_t tgs_segmented_sort_workspace_size(uint64_t n, uint32_t n_segments) {
  return sort_workspace_up_to(n, 4, n_segments);
}

// Tile and group bases of the segments (key_off set) for tiles of `items` keys
// per thread.
static void radix_bases(RadixSegs& sg, uint32_t items) {
  const uint32_t tile = SORT_THREADS * items;
  uint32_t tiles = 0, groups = 0;
  for (uint32_t s = 0; s < sg.n; ++s) {
    const uint32_t nt = (uint32_t)(((uint64_t)sg.key_off[s + 1] - sg.key_off[s] + tile - 1) / tile);
    sg.tile_base[s] = tiles;
    sg.group_base[s] = groups;
    tiles += nt;
    groups += (nt + RADIX_GROUP - 1) / RADIX_GROUP;
  }
  sg.tile_base[sg.n] = tiles;
  sg.group_base[sg.n] = groups;
}

template <typename K, typename V, int ITEMS, bool LOCAL>
static int radix_pass(const K* kin, const V* vin, K* kout, V* vout, const RadixSegs& sg, int shift,
                      int bits, uint32_t* hist, uint32_t* scan_or_groups, void* scan_ws,
                      bool hist_ready, hipStream_t stream) {
  const uint32_t tiles = sg.tile_base[sg.n];
  const uint32_t mask = (1u << bits) - 1u;
  // a histogram the caller counted keeps the 256-digit layout
  const uint32_t nbins = hist_ready ? (uint32_t)SORT_BINS : mask + 1u;
  if (!hist_ready) {
    hipLaunchKernelGGL((radix_hist_kernel<K, ITEMS, LOCAL>), dim3(tiles), dim3(SORT_THREADS), 0,
                       stream, kin, sg, shift, mask, nbins, hist, LOCAL ? scan_or_groups : nullptr);
    TGS_LAUNCH_CHECK("radix_hist");
  }
  const uint32_t* counts = hist;
  if (!LOCAL) {
    const int rc = exclusive_scan_u32(hist, scan_or_groups, (uint64_t)tiles * nbins, scan_ws, stream);
    if (rc) return rc;
    counts = scan_or_groups;
  }
  hipLaunchKernelGGL((radix_scatter_kernel<K, V, ITEMS, LOCAL>), dim3(tiles), dim3(SORT_THREADS), 0,
                     stream, kin, vin, sg, shift, mask, nbins, counts,
                     LOCAL ? scan_or_groups : nullptr, kout, vout);
  TGS_LAUNCH_CHECK("radix_scatter");
  return TGS_OK;
}

// Runs the passes over key bits [begin_bit, end_bit), splitting the range
// into the fewest passes of at most 8 bits with widths as even as possible.
// sg holds the segments' key offsets; first_hist_ready: the first pass's
// histogram (SORT_TILE tiles, 256 digits) is already in the workspace.
template <typename K, typename V>
static int radix_passes(K* keys, V* vals, K* keys_alt, V* vals_alt, RadixSegs& sg,
                        int begin_bit, int end_bit, void* workspace, int* selector,
                        hipStream_t stream, bool first_hist_ready = false) {
  const uint32_t items = first_hist_ready ? SORT_ITEMS : sort_items(sg.key_off[sg.n], sizeof(K));
  radix_bases(sg, items);
  const uint64_t tiles = sg.tile_base[sg.n];
  if (tiles == 0) return TGS_OK;
  const uint64_t hist_max = tiles * SORT_BINS;  // the workspace's layout
  auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
  uint8_t* ws = (uint8_t*)workspace;
  uint32_t* hist = (uint32_t*)ws;
  uint32_t* hist_scan = (uint32_t*)(ws + al(hist_max * 4));
  void* scan_ws = ws + 2 * al(hist_max * 4);
  int passes = (end_bit - begin_bit + 7) / 8;
  // per-pass group rows of a LOCAL sort, in the space of the scanned histogram
  // (64 short segments can need more rows than that holds: then the scan runs)
  const uint64_t group_words = (uint64_t)sg.group_base[sg.n] * SORT_BINS;
  uint32_t most = 0;
  for (uint32_t s = 0; s < sg.n; ++s) {
    const uint32_t nt = sg.tile_base[s + 1] - sg.tile_base[s];
    most = nt > most ? nt : most;
  }
  const bool grouped = most > RADIX_GROUP;
  const bool local = !first_hist_ready && sg.key_off[sg.n] <= RADIX_LOCAL_KEYS(sizeof(K)) &&
                     (!grouped || group_words * passes <= hist_max);
  if (local && grouped) {
    const int rc = tgs_fill_u32(hist_scan, group_words * passes, 0u, stream);
    if (rc) return rc;
  }
  K* kin = keys;
  V* vin = vals;
  K* kout = keys_alt;
  V* vout = vals_alt;
  int sel = 0;
  int shift = begin_bit;
  uint32_t* groups = local && grouped ? hist_scan : nullptr;
  while (shift < end_bit) {
    const int bits = (end_bit - shift + passes - 1) / passes;
    int rc;
    if (local && items == SORT_ITEMS_SMALL)
      rc = radix_pass<K, V, SORT_ITEMS_SMALL, true>(kin, vin, kout, vout, sg, shift, bits, hist,
                                                    groups, scan_ws, false, stream);
    else if (local)
      rc = radix_pass<K, V, SORT_ITEMS, true>(kin, vin, kout, vout, sg, shift, bits, hist, groups,
                                              scan_ws, false, stream);
    else if (items == SORT_ITEMS_SMALL)
      rc = radix_pass<K, V, SORT_ITEMS_SMALL, false>(kin, vin, kout, vout, sg, shift, bits, hist,
                                                     hist_scan, scan_ws, false, stream);
    else
      rc = radix_pass<K, V, SORT_ITEMS, false>(kin, vin, kout, vout, sg, shift, bits, hist,
                                               hist_scan, scan_ws,
                                               first_hist_ready && shift == begin_bit, stream);
    if (rc) return rc;
    if (groups) groups += group_words;
    K* tk = kin;
    kin = kout;
    kout = tk;
    V* tv = vin;
    vin = vout;
    vout = tv;
    sel ^= 1;
    shift += bits;
    --passes;
  }
  *selector = sel;
  return TGS_OK;
}

// Stable ascending sort of (keys, vals) on key bits [begin_bit, end_bit).
// Data ping-pongs between (keys, vals) and (keys_alt, vals_alt); *selector is
// set to 0 if the result is in keys/vals and 1 if in keys_alt/vals_alt
// (the cub::DoubleBuffer convention used at isect_tiles.cu:196-217).
static int radix_sort_u64(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt, uint32_t* vals_alt,
                          uint64_t n, uint32_t key_base, uint32_t low_bits, int begin_bit,
                          int end_bit, void* workspace, size_t workspace_bytes, int* selector,
                          hipStream_t stream) {
  TGS_CHECK_ARG(selector != nullptr, "radix_sort: null selector");
  *selector = 0;
  if (n <= 1 || end_bit <= begin_bit) return TGS_OK;
  TGS_CHECK_ARG(keys && vals && keys_alt && vals_alt && workspace, "radix_sort: null pointer");
  TGS_CHECK_ARG(begin_bit >= 0 && end_bit <= 64, "radix_sort: bit range out of [0,64]");
  TGS_CHECK_ARG(n < (1ull << 32) - SORT_TILE, "radix_sort: n too large");
  if (workspace_bytes < sort_workspace(n, 8, 0)) {
    tgs_set_error("radix_sort: workspace %zu < %zu", workspace_bytes,
                  sort_workspace(n, 8, 0));
    return TGS_ERR_WORKSPACE;
  }
  RadixSegs sg{};
  sg.n = 1;
  sg.key_base = key_base;
  sg.low_bits = low_bits;
  sg.key_off[0] = 0;
  sg.key_off[1] = (uint32_t)n;
  return radix_passes<uint64_t, uint32_t>(keys, vals, keys_alt, vals_alt, sg, begin_bit, end_bit,
                                          workspace, selector, stream);
}

extern "C" int tgs_radix_sort_pairs(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                                    uint32_t* vals_alt, uint64_t n, int begin_bit, int end_bit,
                                    void* workspace, size_t workspace_bytes, int* selector,
                                    hipStream_t stream) {
  return radix_sort_u64(keys, vals, keys_alt, vals_alt, n, 0u, 32u, begin_bit, end_bit, workspace,
                        workspace_bytes, selector, stream);
}

// The same sort on the keys' order when every low word is known to lie in
// [low_base, low_base + 2^low_bits) and every high word below 2^high_bits: low_bits
// + high_bits bits instead of 32 + high_bits (the tile intersections' depth bits:
// 25 to 27 of 32 for depths within a factor of 4 to 30, so five passes, not six).
extern "C" int tgs_radix_sort_pairs_range(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                                          uint32_t* vals_alt, uint64_t n, uint32_t low_base,
                                          int low_bits, int high_bits, void* workspace,
                                          size_t workspace_bytes, int* selector,
                                          hipStream_t stream) {
  TGS_CHECK_ARG(low_bits >= 0 && low_bits <= 32 && high_bits >= 0 && high_bits <= 32,
                "radix_sort_range: low_bits and high_bits in [0, 32]");
  return radix_sort_u64(keys, vals, keys_alt, vals_alt, n, low_base, (uint32_t)low_bits, 0,
                        low_bits + high_bits, workspace, workspace_bytes, selector, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free variant of tgs_radix_sort_pairs for callers that cannot
// allocate device memory (code under HIP graph capture, serving loops that
// forbid hipMalloc).  Its histograms, their scan and the scan's block sums
// live in a file-scope device array sized for TGS_NOALLOC_SORT_MAX_KEYS keys
// (16.0 MiB held by every GPU the library runs on until the process ends).
// Every pass writes each histogram entry before any is read, so the array
// needs no clearing between calls; calls that overlap on one GPU share it and
// race.  Host code reaches the array only through the address that
// hipGetSymbolAddress returns per device (the symbol's name is a host-side
// stand-in, not a device address).
// ---------------------------------------------------------------------------
#define TGS_NOALLOC_SORT_MAX_KEYS (1ull << 25)
#define TGS_NOALLOC_SORT_TILES ((TGS_NOALLOC_SORT_MAX_KEYS + SORT_TILE - 1) / SORT_TILE)
#define TGS_ALIGN256(b) ((((uint64_t)(b)) + 255ull) & ~255ull)
#define TGS_NOALLOC_SORT_HIST (TGS_NOALLOC_SORT_TILES * SORT_BINS)
#define TGS_NOALLOC_SORT_BYTES                          \
  (TGS_ALIGN256(TGS_NOALLOC_SORT_HIST * 4ull) * 2ull + \
   TGS_ALIGN256((TGS_NOALLOC_SORT_HIST + SCAN_CHUNK - 1) / SCAN_CHUNK * 8ull + 8ull))
#define TGS_MAX_DEVICES 64

static __device__ __align__(256) uint8_t scratch[TGS_NOALLOC_SORT_BYTES];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[TGS_MAX_DEVICES] = {};

// Device address of `scratch` on the current device, looked up once per device.
static int noalloc_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    tgs_set_error("radix_sort_noalloc: hipGetDevice failed: %s", hipGetErrorString(e));
    return (int)e;
  }
  if (dev < 0 || dev >= TGS_MAX_DEVICES) {
    tgs_set_error("radix_sort_noalloc: device %d out of range", dev);
    return TGS_ERR_ARG;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      tgs_set_error("radix_sort_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
      return e != hipSuccess ? (int)e : TGS_ERR_ARG;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return TGS_OK;
}

extern "C" int tgs_radix_sort_pairs_noalloc(uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                                            uint32_t* vals_alt, uint64_t n, int begin_bit,
                                            int end_bit, int* selector, hipStream_t stream) {
  TGS_CHECK_ARG(selector != nullptr, "radix_sort_noalloc: null selector");
  *selector = 0;
  if (n > TGS_NOALLOC_SORT_MAX_KEYS) {
    tgs_set_error("radix_sort_noalloc: %llu keys exceed the allocation-free maximum of %llu; "
                  "use tgs_radix_sort_pairs with a workspace",
                  (unsigned long long)n, (unsigned long long)TGS_NOALLOC_SORT_MAX_KEYS);
    return TGS_ERR_ARG;
  }
  if (n <= 1 || end_bit <= begin_bit) return TGS_OK;
  TGS_CHECK_ARG(keys && vals && keys_alt && vals_alt, "radix_sort_noalloc: null pointer");
  TGS_CHECK_ARG(begin_bit >= 0 && end_bit <= 64, "radix_sort_noalloc: bit range out of [0,64]");
  static_assert(TGS_NOALLOC_SORT_BYTES >=
                    TGS_ALIGN256(TGS_NOALLOC_SORT_HIST * 4ull) * 2ull +
                        TGS_ALIGN256((TGS_NOALLOC_SORT_HIST + SCAN_CHUNK - 1) / SCAN_CHUNK * 8ull +
                                     8ull),
                "scratch smaller than the sort workspace");
  if (sort_workspace(n, 8, 0) > TGS_NOALLOC_SORT_BYTES) {
    tgs_set_error("radix_sort_noalloc: workspace %zu exceeds the scratch array",
                  sort_workspace(n, 8, 0));
    return TGS_ERR_WORKSPACE;
  }
  void* ws = nullptr;
  const int rc = noalloc_scratch(&ws);
  if (rc) return rc;
  RadixSegs sg{};
  sg.n = 1;
  sg.key_off[0] = 0;
  sg.key_off[1] = (uint32_t)n;
  return radix_passes<uint64_t, uint32_t>(keys, vals, keys_alt, vals_alt, sg, begin_bit, end_bit,
                                          ws, selector, stream);
}

// Segmented stable sort of uint32 keys with 4- or 8-byte values: each segment
// [seg_offsets[s], seg_offsets[s+1]) is sorted on its own.  seg_offsets is a
// HOST array of n_segments+1 non-decreasing offsets from 0 to n.
static int segmented_sort_u32(uint32_t* keys, void* vals, uint32_t* keys_alt, void* vals_alt,
                              uint32_t value_bytes, uint64_t n, uint32_t n_segments,
                              const uint32_t* seg_offsets, uint32_t key_base, uint32_t key_cap,
                              int begin_bit, int end_bit, void* workspace, size_t workspace_bytes,
                              int* selector, hipStream_t stream, bool first_hist_ready);

extern "C" int tgs_segmented_sort_pairs_u32(uint32_t* keys, void* vals, uint32_t* keys_alt,
                                            void* vals_alt, uint32_t value_bytes, uint64_t n,
                                            uint32_t n_segments, const uint32_t* seg_offsets,
                                            int begin_bit, int end_bit, void* workspace,
                                            size_t workspace_bytes, int* selector,
                                            hipStream_t stream) {
  return segmented_sort_u32(keys, vals, keys_alt, vals_alt, value_bytes, n, n_segments,
                            seg_offsets, 0u, 0xffffffffu, begin_bit, end_bit, workspace,
                            workspace_bytes, selector, stream, false);
}

// The same sort (4-byte values) with the first pass's per-tile digit counts
// already in the workspace, counted by the producer of the keys: uint32 word
// tile_base[s] * 256 + d * (tile_base[s + 1] - tile_base[s]) + t holds the
// count of digit d ((key >> begin_bit) & (2^w - 1), w the first pass's width:
// the key bits split into ceil(bits / 8) passes of ceil(bits / passes) bits)
// among keys [t * 4096, t * 4096 + 4096) of segment s, where tile_base[s] sums
// ceil(segment size / 4096) over the segments before s.
extern "C" int tgs_segmented_sort_pairs_u32_hist0(uint32_t* keys, uint32_t* vals,
                                                  uint32_t* keys_alt, uint32_t* vals_alt,
                                                  uint64_t n, uint32_t n_segments,
                                                  const uint32_t* seg_offsets, int begin_bit,
                                                  int end_bit, void* workspace,
                                                  size_t workspace_bytes, int* selector,
                                                  hipStream_t stream) {
  TGS_CHECK_ARG(begin_bit == 0, "segmented_sort_hist0: the precounted first pass starts at bit 0");
  return segmented_sort_u32(keys, vals, keys_alt, vals_alt, 4, n, n_segments, seg_offsets, 0u,
                            0xffffffffu, begin_bit, end_bit, workspace, workspace_bytes, selector,
                            stream, true);
}

// The same sort on key_bits bits of min(key - key_base, 2^key_bits - 1) (keys
// below key_base as 0): a key range known to lie in [key_base, key_base +
// 2^key_bits - 1) is sorted in fewer or narrower passes, and keys past it
// (a sentinel such as 0xffffffff) tie at the top, in their input order.
extern "C" int tgs_segmented_sort_pairs_u32_range(uint32_t* keys, void* vals, uint32_t* keys_alt,
                                                  void* vals_alt, uint32_t value_bytes, uint64_t n,
                                                  uint32_t n_segments,
                                                  const uint32_t* seg_offsets, uint32_t key_base,
                                                  int key_bits, void* workspace,
                                                  size_t workspace_bytes, int* selector,
                                                  hipStream_t stream) {
  TGS_CHECK_ARG(key_bits >= 1 && key_bits <= 32, "segmented_sort_range: key_bits in [1, 32]");
  const uint32_t cap = key_bits == 32 ? 0xffffffffu : (1u << key_bits) - 1u;
  return segmented_sort_u32(keys, vals, keys_alt, vals_alt, value_bytes, n, n_segments,
                            seg_offsets, key_base, cap, 0, key_bits, workspace, workspace_bytes,
                            selector, stream, false);
}

static int segmented_sort_u32(uint32_t* keys, void* vals, uint32_t* keys_alt, void* vals_alt,
                              uint32_t value_bytes, uint64_t n, uint32_t n_segments,
                              const uint32_t* seg_offsets, uint32_t key_base, uint32_t key_cap,
                              int begin_bit, int end_bit, void* workspace, size_t workspace_bytes,
                              int* selector, hipStream_t stream, bool first_hist_ready) {
  TGS_CHECK_ARG(selector != nullptr, "segmented_sort: null selector");
  *selector = 0;
  if (n <= 1 || end_bit <= begin_bit) return TGS_OK;
  TGS_CHECK_ARG(keys && vals && keys_alt && vals_alt && workspace && seg_offsets,
                "segmented_sort: null pointer");
  TGS_CHECK_ARG(value_bytes == 4 || value_bytes == 8, "segmented_sort: value_bytes must be 4 or 8");
  TGS_CHECK_ARG(begin_bit >= 0 && end_bit <= 32, "segmented_sort: bit range out of [0,32]");
  TGS_CHECK_ARG(n < (1ull << 32) - (uint64_t)SORT_TILE * (RADIX_MAX_SEGS + 1),
                "segmented_sort: n too large");
  TGS_CHECK_ARG(n_segments >= 1 && n_segments <= RADIX_MAX_SEGS,
                "segmented_sort: n_segments must be in [1, 64]");
  TGS_CHECK_ARG(seg_offsets[0] == 0 && seg_offsets[n_segments] == n,
                "segmented_sort: segments must cover [0, n)");
  RadixSegs sg{};
  sg.n = n_segments;
  sg.key_base = key_base;
  sg.key_cap = key_cap;
  for (uint32_t s = 0; s < n_segments; ++s) {
    TGS_CHECK_ARG(seg_offsets[s + 1] >= seg_offsets[s], "segmented_sort: offsets decrease");
    sg.key_off[s] = seg_offsets[s];
  }
  sg.key_off[n_segments] = (uint32_t)n;
  if (workspace_bytes < sort_workspace(n, 4, n_segments)) {
    tgs_set_error("segmented_sort: workspace %zu < %zu", workspace_bytes,
                  sort_workspace(n, 4, n_segments));
    return TGS_ERR_WORKSPACE;
  }
  if (value_bytes == 4)
    return radix_passes<uint32_t, uint32_t>(keys, (uint32_t*)vals, keys_alt, (uint32_t*)vals_alt,
                                            sg, begin_bit, end_bit, workspace, selector, stream,
                                            first_hist_ready);
  TGS_CHECK_ARG(!first_hist_ready, "segmented_sort: a precounted first pass needs 4-byte values");
  return radix_passes<uint32_t, uint64_t>(keys, (uint64_t*)vals, keys_alt, (uint64_t*)vals_alt, sg,
                                          begin_bit, end_bit, workspace, selector, stream);
}
