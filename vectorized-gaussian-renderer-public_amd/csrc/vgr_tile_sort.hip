// Depth order inside every tile: the second half of the global ordering.
//
// The radix passes (vgr_sort.hip) partition the intersections by tile and by the
// leading depth bits that fit the same passes; here each tile's list is sorted by
// (depth bits, record), which together is the order of the full key.  A list is
// read and written about once (24 bytes per intersection), where three more 9-bit
// radix passes over the depth bits move 72 and pay a look-back chain each.
//
//   tile_sort_kernel  : one workgroup per tile sorts lists of up to 2048 entries
//                       in LDS.  A longer list is cut where the leading depth bits
//                       change into parts that fit: they are sorted one after the
//                       other, or queued when there are many or one does not fit;
//   small_tile_sort_kernel : the same for tiles of up to 4x4 pixels, of which a
//                       workgroup takes four: a list of up to 512 entries is one
//                       wave's, the rest the workgroup's;
//   spread_long_kernel: parts that do not fit the LDS of run_sort_kernel either are
//                       spread over up to 4096 depth bins in global memory and queued as
//                       runs of whole bins that do; a bin that does not fit is spread
//                       again over its own range (over the tie order when all its
//                       depths are equal), or sorted in place when its tie words are
//                       equal too (a scene whose Gaussian IDs repeat);
//   run_sort_kernel   : a persistent grid over the queue (runs of up to 8192 entries).
// The split follows the LDS: 2048 entries leave six workgroups on a CU to hide
// each other's barriers, and two of 8192 entries fit.  Bound by those barriers and
// the LDS round trips between them.  Measured on 64 cameras of 640x480 over 1M
// Gaussians (127M intersections, lists of 1651 on average): the whole ordering
// 5.27 -> 3.62 ms, of it 1.72 for the two partition passes, 0.30 for their histogram,
// 0.29 for the ranges, 0.49 for the lists of up to 2048 entries (82M entries, 4.4 ps
// each at 24 bytes in and out) and 0.79 for the longer ones; 1 camera of 640x480 over
// 100k: 118 -> 70 us.
#include "vgr_tile_sort_device.h"

namespace vgr {
namespace {

using namespace dev;

// Consecutive entries of one tile to sort in LDS: `count` entries from `begin` of
// buffer pair `pair` (0: the partitioned input, 1: the result's own buffers).
struct alignas(16) Run {
  uint32_t begin, count, tile, pair;
};

constexpr int kTileThreads = 256;
constexpr int kTileCapacity = 2048;  // 24 KB of LDS: six workgroups per CU
constexpr int kWaveCapacity = 512;   // of a wave that sorts a list alone
constexpr int kRunThreads = 512;
constexpr int kRunCapacity = 8192;
constexpr int kRunBins = 3072;  // 78 KB of LDS with the entries: two workgroups per CU

struct TileSortArgs {
  const uint64_t* keys_in;   // partitioned by tile
  const int32_t* values_in;
  uint64_t* keys_out;
  int32_t* values_out;
  const int32_t* tile_starts;
  int32_t* tile_ends;
  int64_t tiles;
  PartitionKey partition;
  int64_t* failures;          // look-back waits the partition gave up: its order is wrong
  const vgr_record* records;  // spatially ordered scenes: ties by the record's Gaussian ID; else null
  int64_t visible_capacity;
  Run* runs;                  // queue of the parts for run_sort_kernel
  uint32_t run_capacity;
  Run* long_runs;             // queue of the parts for spread_long_kernel
  uint32_t long_capacity;
  uint32_t* state;            // [0] queued runs, [1] taken runs, [2] queued long parts, [3] taken ones
};

// Order of entries of equal depth: the Gaussian ID, which is the order of the
// values themselves (records of a camera, and slots of a training forward, are
// written in Gaussian order) unless the scene is stored in a spatial order.
struct TieOrder {
  const vgr_record* records;
  int64_t visible_capacity;
  __device__ __forceinline__ uint32_t word(int32_t value) const {
    if (records == nullptr) return static_cast<uint32_t>(value);
    return value >= 0 && value < visible_capacity ? static_cast<uint32_t>(records[value].gaussian_id) : 0u;
  }
  // The value itself only tells apart records that a corrupted list repeats.
  __device__ __forceinline__ uint64_t operator()(int32_t value) const {
    return (static_cast<uint64_t>(word(value)) << 32) | static_cast<uint32_t>(value);
  }
};

__device__ __forceinline__ uint32_t depth_word(const uint64_t* keys, int64_t i) {
  return reinterpret_cast<const uint32_t*>(keys)[2 * i];  // low half: depth bits
}

// Queues a part; false if the queue is full.  Called by one thread.
__device__ __forceinline__ bool push_run(const TileSortArgs& args, const Run& run) {
  const bool fits = run.count <= static_cast<uint32_t>(kRunCapacity);
  const uint32_t slot = atomicAdd(&args.state[fits ? 0 : 2], 1u);
  if (slot >= (fits ? args.run_capacity : args.long_capacity)) return false;
  (fits ? args.runs : args.long_runs)[slot] = run;
  return true;
}

// Sorts entries [at, at + length) of a buffer pair into the result's buffers with a
// bitonic network in global memory, by the whole workgroup: for parts that the queue
// has no room for, crowded bins beyond kSpreadStack in one list, and entries that
// nothing but the value itself tells apart.  Barriers inside and at the end.
template <int kThreads>
__device__ __forceinline__ void sort_in_place(const TileSortArgs& args, int64_t at, uint32_t length,
                                              const uint64_t* source_keys, const int32_t* source_values) {
  const TieOrder tie{args.records, args.visible_capacity};
  if (source_keys != args.keys_out) {
    for (uint32_t i = threadIdx.x; i < length; i += kThreads) {
      args.keys_out[at + i] = source_keys[at + i];
      args.values_out[at + i] = source_values[at + i];
    }
  }
  uint32_t padded = 2u;
  while (padded < length) padded <<= 1;
  for (uint32_t size = 2u; size != 0u && size <= padded; size <<= 1) {
    for (uint32_t stride = size >> 1; stride > 0u; stride >>= 1) {
      __threadfence_block();
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < padded / 2u; i += kThreads) {
        const uint32_t low_bits = i & (stride - 1u);
        const uint32_t a = ((i - low_bits) << 1) + low_bits;
        const uint32_t b = stride == (size >> 1) ? ((i - low_bits) << 1) + size - 1u - low_bits : a + stride;
        if (b >= length) continue;
        const uint64_t ka = args.keys_out[at + a], kb = args.keys_out[at + b];
        const int32_t va = args.values_out[at + a], vb = args.values_out[at + b];
        if (kb < ka || (kb == ka && tie(vb) < tie(va))) {
          args.keys_out[at + a] = kb;
          args.keys_out[at + b] = ka;
          args.values_out[at + a] = vb;
          args.values_out[at + b] = va;
        }
      }
    }
  }
  __threadfence_block();
  __syncthreads();
}

// Entries of the sorted-by-lead list [begin, count) that are counted by `below`, which
// holds for a prefix of them: the length of that prefix, found by the workgroup with
// kThreads probes at a time.  Every thread gets the result; barriers inside.
template <int kThreads, typename S, typename Below>
__device__ __forceinline__ uint32_t prefix_length(S& s, uint32_t begin, uint32_t count, Below&& below) {
  uint32_t low = begin, high = count;  // the prefix ends in [low, high]
  while (low < high) {                 // uniform
    const uint32_t step = (high - low + kThreads - 1) / kThreads;
    const uint32_t probe = low + threadIdx.x * step;
    const bool inside = probe < high && below(probe);
    const uint32_t votes = static_cast<uint32_t>(__popcll(__ballot(inside)));
    if ((threadIdx.x & (kWave - 1)) == 0) s.wave_a[threadIdx.x / kWave] = votes;
    __syncthreads();
    uint32_t hits = 0u;
#pragma unroll
    for (int w = 0; w < S::kWaves; ++w) hits += s.wave_a[w];
    __syncthreads();
    // Probes 0 .. hits - 1 are inside, probe `hits` (if any) is not.
    const uint32_t first_out = low + hits * step;
    high = first_out < high ? first_out : high;
    low = hits == 0u ? low : low + (hits - 1u) * step + 1u;
    if (hits == 0u) high = low;
  }
  return low - begin;
}

// Sorts the list [start, start + count) of a tile, or queues it or parts of it, with the
// workgroup.  Without kSplit crowded parts are queued; kMayRefuse where the queue may have
// no place for them (launch_tile_sort).  Ends behind a barrier.
template <bool kSplit, bool kMayRefuse, int kThreads, int kCapacity, int kBins>
__device__ __forceinline__ void sort_list(const TileSortArgs& args, TileSort<kThreads, kCapacity, kBins>& s,
                                          bool& s_queued, int64_t tile, int64_t start, uint32_t count) {
  // Uniform bases and 32-bit offsets: the addresses stay out of the vector registers.
  const uint32_t* const all_depths = reinterpret_cast<const uint32_t*>(args.keys_in + start);
  const auto lead = [&](uint32_t i) {
    return (all_depths[2u * static_cast<uint64_t>(i)] - args.partition.depth_base) >> args.partition.lead_shift;
  };
  const uint64_t tile_bits = static_cast<uint64_t>(tile) << 32;
  // Lists of a few parts are sorted here; more parts share the work with run_sort_kernel.
  const bool here = count <= 4u * kCapacity;
  for (uint32_t begin = 0u; begin < count;) {  // uniform
    uint32_t n = count - begin;
    if (n > static_cast<uint32_t>(kCapacity)) {
      // Whole leading-bit groups that fit, or the one group that does not.
      const uint32_t next = lead(begin + kCapacity);
      n = prefix_length<kThreads>(s, begin, begin + kCapacity, [&](uint32_t i) { return lead(i) < next; });
      if (n == 0u) {
        n = kCapacity + prefix_length<kThreads>(s, begin + kCapacity, count,
                                                [&](uint32_t i) { return lead(i) <= next; });
      }
    }
    bool sorted = false;
    if (n <= static_cast<uint32_t>(kCapacity) && here) {
      const uint32_t* const depths = all_depths + 2u * static_cast<uint64_t>(begin);
      const int32_t* const list = args.values_in + start + begin;
      uint64_t* const keys_out = args.keys_out + start + begin;
      int32_t* const values_out = args.values_out + start + begin;
      sorted = tile_sort<kSplit>(
          s, n, [&](uint32_t i) { return depths[2u * i]; }, [&](uint32_t i) { return list[i]; },
          TieOrder{args.records, args.visible_capacity}, [&](uint32_t rank, uint32_t key, int32_t value) {
            keys_out[rank] = tile_bits | key;
            values_out[rank] = value;
          });
    }
    if (!sorted) {  // uniform
      if (threadIdx.x == 0) {
        const bool queued =
            push_run(args, Run{static_cast<uint32_t>(start) + begin, n, static_cast<uint32_t>(tile), 0u});
        if constexpr (kMayRefuse) {
          s_queued = queued;
        } else if (!queued) {
          atomicAdd(reinterpret_cast<unsigned long long*>(args.failures), 1ull);  // never, by the bound
        }
      }
      if constexpr (kMayRefuse) {
        __syncthreads();
        if (!s_queued) sort_in_place<kThreads>(args, start + begin, n, args.keys_in, args.values_in);
      }
    }
    begin += n;
    __syncthreads();  // LDS free for the next part
  }
}

// A failed partition leaves lists that overlap and slots nobody wrote: the render is
// invalid and reported as such, and its lists are emptied rather than sorted.

// 8x8 and 16x16 tiles: a workgroup per tile.
template <bool kMayRefuse>
__global__ __launch_bounds__(kTileThreads, 6) void tile_sort_kernel(TileSortArgs args) {
  __shared__ TileSort<kTileThreads, kTileCapacity, kTileCapacity> s;
  __shared__ bool s_queued;
  const bool failed = *args.failures != 0;
  for (int64_t tile = blockIdx.x; tile < args.tiles; tile += gridDim.x) {
    const int64_t start = args.tile_starts[tile];
    const int64_t count = static_cast<int64_t>(args.tile_ends[tile]) - start;
    if (count <= 0) continue;
    if (failed) {
      if (threadIdx.x == 0) args.tile_ends[tile] = static_cast<int32_t>(start);
      continue;
    }
    sort_list<false, kMayRefuse>(args, s, s_queued, tile, start, static_cast<uint32_t>(count));
  }
}

// Tiles of up to 4x4 pixels: a workgroup takes four, each wave the list of one if it
// fits the wave's share of the LDS, then the whole workgroup those that are longer or
// crowded, which it splits itself: the lists of pixels that look at a wall are.  Their
// lengths are known on the device only and run from 68 entries on average (128x128
// views of a 5M-Gaussian room at tile size 1, with the depth cutoff) to 660 (without)
// and thousands (4x4 tiles).  Lists sorted by one wave each, with longer and crowded
// ones queued for run_sort_kernel, against this: depth order of that room with the
// cutoff 120 -> 114 us and without 2,208 -> 1,413, of a room of 1M Gaussians at tile
// size 1 532 -> 394 and at 2x2 402 -> 290.
constexpr int kSmallTiles = kTileThreads / kWave;

union SmallTiles {
  TileSort<kWave, kWaveCapacity, kWaveCapacity> of_wave[kSmallTiles];
  TileSort<kTileThreads, kTileCapacity, kTileCapacity> of_group;
};

// Not a loop over groups of tiles: hoisted out of one, the addresses of both forms spill.
__global__ __launch_bounds__(kTileThreads, 6) void small_tile_sort_kernel(TileSortArgs args, int64_t first_tile) {
  __shared__ SmallTiles s;
  __shared__ bool s_queued;
  __shared__ uint32_t s_left[kSmallTiles];  // entries of the lists that the waves leave to the workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t first = first_tile + static_cast<int64_t>(blockIdx.x) * kSmallTiles;
  const int64_t own = first + wave;
  const int32_t start = __builtin_amdgcn_readfirstlane(own < args.tiles ? args.tile_starts[own] : 0);
  const int32_t count = __builtin_amdgcn_readfirstlane(own < args.tiles ? args.tile_ends[own] : 0) - start;
  if (*args.failures != 0) {
    if (count > 0 && (threadIdx.x & (kWave - 1)) == 0) args.tile_ends[own] = start;
    return;
  }
  bool sorted = count <= 0;
  if (count > 0 && count <= kWaveCapacity) {
    const uint32_t* const depths = reinterpret_cast<const uint32_t*>(args.keys_in + start);
    const int32_t* const list = args.values_in + start;
    uint64_t* const keys_out = args.keys_out + start;
    int32_t* const values_out = args.values_out + start;
    const uint64_t tile_bits = static_cast<uint64_t>(own) << 32;
    sorted = tile_sort<false>(
        s.of_wave[wave], static_cast<uint32_t>(count), [&](uint32_t i) { return depths[2u * i]; },
        [&](uint32_t i) { return list[i]; }, TieOrder{args.records, args.visible_capacity},
        [&](uint32_t rank, uint32_t key, int32_t value) {
          keys_out[rank] = tile_bits | key;
          values_out[rank] = value;
        });
  }
  if ((threadIdx.x & (kWave - 1)) == 0) s_left[wave] = sorted ? 0u : static_cast<uint32_t>(count);
  if (!__syncthreads_or(sorted ? 0 : 1)) return;
  for (int q = 0; q < kSmallTiles; ++q) {
    const uint32_t left = __builtin_amdgcn_readfirstlane(s_left[q]);
    if (left == 0u) continue;  // uniform
    const int64_t list_start = __builtin_amdgcn_readfirstlane(args.tile_starts[first + q]);
    sort_list<true, true>(args, s.of_group, s_queued, first + q, list_start, left);
  }
}

__global__ __launch_bounds__(kRunThreads, 4) void run_sort_kernel(TileSortArgs args) {
  __shared__ TileSort<kRunThreads, kRunCapacity, kRunBins> s;
  __shared__ uint32_t s_item;
  const uint32_t queued = args.state[0] < args.run_capacity ? args.state[0] : args.run_capacity;
  if (queued == 0u) return;
  for (;;) {
    if (threadIdx.x == 0) s_item = atomicAdd(&args.state[1], 1u);
    __syncthreads();
    if (s_item >= queued) return;
    const Run run = args.runs[s_item];
    const uint32_t n = run.count;
    const uint32_t* const depths =
        reinterpret_cast<const uint32_t*>((run.pair != 0u ? args.keys_out : args.keys_in) + run.begin);
    const int32_t* const list = (run.pair != 0u ? args.values_out : args.values_in) + run.begin;
    uint64_t* const keys_out = args.keys_out + run.begin;
    int32_t* const values_out = args.values_out + run.begin;
    const uint64_t tile_bits = static_cast<uint64_t>(run.tile) << 32;
    // A run already in the result's buffers is read whole before any of it is written.
    tile_sort<true>(
        s, n, [&](uint32_t i) { return depths[2u * i]; }, [&](uint32_t i) { return list[i]; },
        TieOrder{args.records, args.visible_capacity}, [&](uint32_t rank, uint32_t key, int32_t value) {
          keys_out[rank] = tile_bits | key;
          values_out[rank] = value;
        });
    __syncthreads();  // LDS free for the next run
  }
}

constexpr int kSpreadThreads = 1024;
// Depth bins of a spread: one per 1024 entries.  Every bin in use keeps a cache line of
// keys and one of values open for writing, so more of them cost: 256 cameras of four
// resolutions (the spread of 446M intersections' long lists) 3.9 ms with 4096 bins
// always, 2.2 with a bin per 256 or 1024 entries, 2.4 per 2048; 16 views of 128x128 over
// 2M Gaussians (lists of 45,000) 672, 414, 322 and 313 us.
constexpr int kSpreadBins = 4096;
constexpr uint32_t kSpreadBinEntries = 1024;
constexpr uint32_t kSpreadLeastBins = 32;
constexpr int kSpreadStack = 256;
constexpr int kSpreadLoads = 4;  // entries in flight per thread
constexpr uint32_t kSpreadSample = 4096;

struct SpreadShared {
  static constexpr int kWaves = kSpreadThreads / kWave;
  uint32_t cursor[kSpreadBins];
  uint32_t first[kSpreadBins + 1];  // first entry of every bin of the segment being spread
  uint32_t wave_a[kWaves];
  uint32_t wave_b[kWaves];
  // Segments still to spread: offset and length in the part, and the pair that holds them.
  uint32_t stack_begin[kSpreadStack];
  uint32_t stack_count[kSpreadStack];
  uint32_t stack_pair[kSpreadStack];
  uint32_t depth;
  uint32_t item;
  bool queued;
};

template <bool kMayRefuse>
__global__ __launch_bounds__(kSpreadThreads, 8) void spread_long_kernel(TileSortArgs args) {
  __shared__ SpreadShared s;
  const int t = threadIdx.x;
  const TieOrder tie{args.records, args.visible_capacity};
  // The spread ping-pongs between the two buffer pairs.
  uint64_t* const keys_of[2] = {const_cast<uint64_t*>(args.keys_in), args.keys_out};
  int32_t* const values_of[2] = {const_cast<int32_t*>(args.values_in), args.values_out};
  const uint32_t queued = args.state[2] < args.long_capacity ? args.state[2] : args.long_capacity;
  if (queued == 0u) return;
  for (;;) {
    __syncthreads();
    if (t == 0) s.item = atomicAdd(&args.state[3], 1u);
    __syncthreads();
    if (s.item >= queued) return;
    const Run part = args.long_runs[s.item];
    const int64_t list = part.begin;
    const uint32_t tile = part.tile;
    if (t == 0) {
      s.stack_begin[0] = 0u;
      s.stack_count[0] = part.count;
      s.stack_pair[0] = 0u;
      s.depth = 1u;
    }
    __syncthreads();
    bool whole_list = true;
    while (s.depth != 0u) {  // uniform: changed between barriers only
      const uint32_t top = s.depth - 1u;
      const uint32_t begin = s.stack_begin[top];
      const uint32_t count = s.stack_count[top];
      const int from = static_cast<int>(s.stack_pair[top]);
      const int to = 1 - from;
      const int64_t base = list + begin;
      const uint64_t* const source_keys = keys_of[from];
      const int32_t* const source_values = values_of[from];
      __syncthreads();
      if (t == 0) s.depth = top;

      // Range of the depths: from a sample of a whole list (its outliers share the end
      // bins), exact for a crowded bin, whose entries are spread by their tie order when
      // they all have the same depth.
      const uint32_t step = whole_list ? count / kSpreadSample : 1u;  // count > kRunCapacity
      whole_list = false;
      uint32_t lo = 0xffffffffu, hi = 0u;
      for (uint32_t i = t * step; i < count; i += kSpreadThreads * step) {
        const uint32_t key = depth_word(source_keys, base + i);
        lo = key < lo ? key : lo;
        hi = key > hi ? key : hi;
      }
      block_min_max(s, lo, hi);
      const bool by_tie = step == 1u && lo == hi;
      if (by_tie) {
        __syncthreads();
        lo = 0xffffffffu;
        hi = 0u;
        for (uint32_t i = t; i < count; i += kSpreadThreads) {
          const uint32_t word = tie.word(source_values[base + i]);
          lo = word < lo ? word : lo;
          hi = word > hi ? word : hi;
        }
        block_min_max(s, lo, hi);
        if (lo == hi) {  // uniform
          // No bin splits entries of one depth and one tie word.  Every other segment comes
          // out smaller: over an exact range, lo and hi fall into different bins.
          sort_in_place<kSpreadThreads>(args, base, count, source_keys, source_values);
          continue;
        }
      }
      uint32_t bins = count / kSpreadBinEntries;
      bins = bins < kSpreadLeastBins ? kSpreadLeastBins : (bins < kSpreadBins ? bins : kSpreadBins);
      const BinMap bin_of(lo, hi, bins);
      for (int b = t; b < kSpreadBins; b += kSpreadThreads) s.cursor[b] = 0u;
      __syncthreads();
      for (uint32_t i0 = 0u; i0 < count; i0 += kSpreadThreads * kSpreadLoads) {
        uint32_t word[kSpreadLoads];
#pragma unroll
        for (int r = 0; r < kSpreadLoads; ++r) {
          const uint32_t i = i0 + r * kSpreadThreads + t;
          word[r] = i < count ? (by_tie ? tie.word(source_values[base + i]) : depth_word(source_keys, base + i)) : 0u;
        }
#pragma unroll
        for (int r = 0; r < kSpreadLoads; ++r) {
          if (i0 + r * kSpreadThreads + t < count) atomicAdd(&s.cursor[bin_of(word[r])], 1u);
        }
      }
      __syncthreads();
      constexpr int kPer = kSpreadBins / kSpreadThreads;
      uint32_t counts[kPer], own = 0u;
#pragma unroll
      for (int b = 0; b < kPer; ++b) {
        counts[b] = s.cursor[t * kPer + b];
        own += counts[b];
      }
      const uint32_t inclusive = wave_inclusive_sum_u32(own);
      if ((t & (kWave - 1)) == kWave - 1) s.wave_a[t / kWave] = inclusive;
      __syncthreads();
      uint32_t running = inclusive - own;
      for (int w = 0; w < t / kWave; ++w) running += s.wave_a[w];
#pragma unroll
      for (int b = 0; b < kPer; ++b) {
        s.cursor[t * kPer + b] = running;
        s.first[t * kPer + b] = running;
        running += counts[b];
      }
      if (t == 0) s.first[kSpreadBins] = count;
      __syncthreads();
      for (uint32_t i0 = 0u; i0 < count; i0 += kSpreadThreads * kSpreadLoads) {
        uint64_t key[kSpreadLoads];
        int32_t value[kSpreadLoads];
#pragma unroll
        for (int r = 0; r < kSpreadLoads; ++r) {
          const uint32_t i = i0 + r * kSpreadThreads + t;
          key[r] = i < count ? source_keys[base + i] : 0ull;
          value[r] = i < count ? source_values[base + i] : 0;
        }
#pragma unroll
        for (int r = 0; r < kSpreadLoads; ++r) {
          if (i0 + r * kSpreadThreads + t < count) {
            const uint32_t word = by_tie ? tie.word(value[r]) : static_cast<uint32_t>(key[r]);
            const uint32_t position = atomicAdd(&s.cursor[bin_of(word)], 1u);
            keys_of[to][base + position] = key[r];
            values_of[to][base + position] = value[r];
          }
        }
      }
      __threadfence_block();
      __syncthreads();
      // Runs of whole bins that fit run_sort_kernel are queued; a bin that does not is pushed.
      uint32_t bin = 0u;
      while (bin < static_cast<uint32_t>(kSpreadBins)) {  // uniform
        const uint32_t run_begin = s.first[bin];
        uint32_t low = bin, high = kSpreadBins;  // largest end with first[end] - run_begin <= capacity
        while (low < high) {
          const uint32_t middle = (low + high + 1u) >> 1;
          if (s.first[middle] - run_begin <= static_cast<uint32_t>(kRunCapacity)) {
            low = middle;
          } else {
            high = middle - 1u;
          }
        }
        if (low > bin) {
          const uint32_t length = s.first[low] - run_begin;
          bin = low;
          if (length == 0u) continue;  // uniform
          if (t == 0) {
            const bool queued = push_run(args, Run{static_cast<uint32_t>(base) + run_begin, length, tile,
                                                   static_cast<uint32_t>(to)});
            if constexpr (kMayRefuse) {
              s.queued = queued;
            } else if (!queued) {
              atomicAdd(reinterpret_cast<unsigned long long*>(args.failures), 1ull);  // never, by the bound
            }
          }
          if constexpr (kMayRefuse) {
            __syncthreads();
            if (!s.queued) sort_in_place<kSpreadThreads>(args, base + run_begin, length, keys_of[to], values_of[to]);
            __syncthreads();  // s.queued read before the next run
          }
          continue;
        }
        const uint32_t length = s.first[bin + 1] - run_begin;
        const uint32_t depth = s.depth;
        __syncthreads();
        if (depth < static_cast<uint32_t>(kSpreadStack)) {
          if (t == 0) {
            s.stack_begin[depth] = begin + run_begin;
            s.stack_count[depth] = length;
            s.stack_pair[depth] = static_cast<uint32_t>(to);
            s.depth = depth + 1u;
          }
          __syncthreads();
        } else {
          sort_in_place<kSpreadThreads>(args, base + run_begin, length, keys_of[to], values_of[to]);
        }
        ++bin;
      }
      __syncthreads();  // bins read before the next segment reuses them
    }
  }
}

}  // namespace

int launch_tile_sort(const vgr_scene& scene, const vgr_cameras& cameras, const vgr_workspace& ws,
                     const ScratchLayout& layout, char* scratch, int64_t global_tiles, int tile_size,
                     bool partitioned_in_out, hipStream_t stream) {
  if (global_tiles <= 0) return 0;
  TileSortArgs args;
  args.keys_in = partitioned_in_out ? ws.keys_out : ws.keys_in;
  args.values_in = partitioned_in_out ? ws.values_out : ws.values_in;
  args.keys_out = partitioned_in_out ? ws.keys_in : ws.keys_out;
  args.values_out = partitioned_in_out ? ws.values_in : ws.values_out;
  args.tile_starts = ws.tile_starts;
  args.tile_ends = ws.tile_ends;
  args.tiles = global_tiles;
  args.failures = ws.counters + VGR_COUNTER_SORT_FAILURES;
  args.records = scene.gaussian_ids != nullptr ? ws.records : nullptr;
  args.visible_capacity = ws.visible_capacity;
  args.partition = layout.partition;
  // The look-back flags are read no more: their scratch holds the queues, with a place
  // per sort tile (at most 8192 entries) for a part of over 8192 entries, so those always
  // fit.  The other parts number at most 101 per 8192 entries: 32 crowded ones of over
  // kSplitLeast, nine of longer lists (two neighbours hold over 2048 entries) and four
  // runs per spread of the part or bin that holds them, of which there is one over a
  // sampled range and, at kSpreadLeastBins or more a time, seven over a 32-bit depth and
  // seven over a 32-bit tie word.  The default digits leave at least 127 places;
  // explicit digits of four or five bits may leave fewer, and parts beyond them are
  // sorted where they are found, by the workgroup that found them.  tile_sort_kernel and
  // spread_long_kernel have a form of their own for that: in the usual ones the code costs
  // scalar registers and 9 % (127M entries 497 -> 542 us), or two barriers a run (7 %);
  // under small tiles it costs nothing.
  static_assert(sizeof(Run) == 16 && kSortThreads * kDefaultSortItems <= kRunCapacity,
                "a part that is spread takes more entries than a sort tile");
  args.long_runs = reinterpret_cast<Run*>(scratch + layout.sort_flags);
  args.long_capacity = static_cast<uint32_t>(layout.sort_tiles);
  args.runs = args.long_runs + args.long_capacity;
  args.run_capacity = static_cast<uint32_t>(layout.sort_flag_words / 4 - layout.sort_tiles);
  args.state = reinterpret_cast<uint32_t*>(scratch + layout.work_counter) + 4;
  constexpr int kSpreads = 1 + 2 * 7;
  static_assert(kSpreadLeastBins == 32, "five bits a spread");
  constexpr int64_t kPartsPerSortTile =
      kRunCapacity / kSplitLeast + 2 * kRunCapacity / kTileCapacity + 1 + 4 * kSpreads;
  static_assert(kPartsPerSortTile == 101, "the bound above");
  const bool may_refuse = args.run_capacity < kPartsPerSortTile * layout.sort_tiles;
  const int64_t capacity = ws.intersection_capacity;
  constexpr int64_t kMaxGrid = 1 << 22;
  if (tile_size <= 4) {
    constexpr int64_t kMost = kMaxGrid * kSmallTiles;  // tiles of a grid
    for (int64_t first = 0; first < global_tiles; first += kMost) {
      const int64_t rest = global_tiles - first < kMost ? global_tiles - first : kMost;
      hipLaunchKernelGGL(small_tile_sort_kernel, dim3(static_cast<unsigned>((rest + kSmallTiles - 1) / kSmallTiles)),
                         dim3(kTileThreads), 0, stream, args, first);
    }
  } else {
    hipLaunchKernelGGL(may_refuse ? tile_sort_kernel<true> : tile_sort_kernel<false>,
                       dim3(static_cast<unsigned>(global_tiles < kMaxGrid ? global_tiles : kMaxGrid)),
                       dim3(kTileThreads), 0, stream, args);
  }
  // A list holds a Gaussian once for every time its camera is active (active_ids may
  // repeat a camera), so a small scene has no long ones (nor crowded ones up to
  // kSplitLeast).
  const int64_t longest = scene.gaussian_count * (cameras.active_ids != nullptr ? cameras.active_count : 1);
  // Persistent grids of two workgroups per CU; an empty queue ends every one at once.
  constexpr int64_t kPersistent = 512;
  if (longest > kRunCapacity) {
    const int64_t most = capacity / kRunCapacity + 1;
    hipLaunchKernelGGL(may_refuse ? spread_long_kernel<true> : spread_long_kernel<false>,
                       dim3(static_cast<unsigned>(most < kPersistent ? most : kPersistent)), dim3(kSpreadThreads), 0,
                       stream, args);
  }
  if (longest > kSplitLeast) {
    const int64_t most = capacity / kSplitLeast + 1;
    hipLaunchKernelGGL(run_sort_kernel, dim3(static_cast<unsigned>(most < kPersistent ? most : kPersistent)),
                       dim3(kRunThreads), 0, stream, args);
  }
  const hipError_t error = hipGetLastError();
  if (error != hipSuccess) {
    set_error("tile sort launch failed: %s", hipGetErrorString(error));
    return VGR_E_LAUNCH;
  }
  return 0;
}

}  // namespace vgr
