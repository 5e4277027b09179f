// Sort of one tile's intersections in LDS, by a workgroup or by a wave: the depth
// order inside a tile of the global ordering.
//
// The entries are spread over as many bins as there are entries (up to kBins),
// evenly over the range of their keys, by LDS counters; each entry then counts
// the smaller entries of its own bin.  With one or two entries per bin this
// costs one returning LDS atomic, one scatter and a few LDS reads per entry,
// where a stable LSD radix sort pays nine ballots per entry and 9-bit digit.
// Where depths crowd (a wall seen through empty space), every bin is split once
// more into as many parts as it holds entries; a part that stays crowded (equal
// depths) sends the list to a bitonic network, O(n log^2 n) whatever the keys.
// The result is the order of (key, tie), a total order, so it does not depend
// on the order the entries arrive in or the atomics are served in.
#ifndef VGR_TILE_SORT_DEVICE_H
#define VGR_TILE_SORT_DEVICE_H

#include "vgr_internal.h"

namespace vgr {
namespace dev {

constexpr uint32_t kSplitLeast = 256;  // shorter lists count through crowded bins

template <int kThreads, int kCapacity, int kBins>
struct TileSort {
  static_assert(kCapacity % kThreads == 0 && kBins % kThreads == 0 && (kCapacity & (kCapacity - 1)) == 0,
                "whole items and bins per thread; the bitonic network needs a power of two");
  static constexpr int kItems = kCapacity / kThreads;
  static constexpr int kWaves = kThreads / kWave;
  static constexpr uint32_t kCrowd = 32;      // entries of a bin worth splitting further
  static constexpr uint32_t kPartCrowd = 32;  // entries of a part that a network sorts faster
  uint32_t keys[kCapacity];
  int32_t values[kCapacity];
  uint32_t start[kBins + 1];
  uint32_t wave_a[kWaves];
  uint32_t wave_b[kWaves];
};

// Order-preserving map of [low, low + range] onto [0, bins); keys outside go to
// the end bins.
struct BinMap {
  uint32_t low, range, bins, multiplier;
  __device__ __forceinline__ BinMap(uint32_t lo, uint32_t hi, uint32_t count) : low(lo), range(hi - lo), bins(count) {
    // floor(bins * 2^32 / (range + 1)) up to float rounding; any multiplier is monotone.
    multiplier = range >= bins ? static_cast<uint32_t>(static_cast<float>(bins) * 4294967040.0f /
                                                       (static_cast<float>(range) + 1.0f))
                               : 0u;
  }
  __device__ __forceinline__ uint32_t operator()(uint32_t key) const {
    const uint32_t offset = key > low ? key - low : 0u;
    const uint32_t bin = range >= bins ? __umulhi(offset, multiplier) : offset;
    return bin < bins ? bin : bins - 1u;
  }
  // Place of the key within its bin, in 2^-32 of the bin's width.
  __device__ __forceinline__ uint32_t fraction(uint32_t key) const {
    const uint32_t offset = key > low ? key - low : 0u;
    if (range < bins) return 0u;  // one key per bin
    return __umulhi(offset, multiplier) < bins ? offset * multiplier : 0xffffffffu;
  }
};

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
  for (int offset = kWave / 2; offset > 0; offset >>= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), offset, kWave));
    v = o < v ? o : v;
  }
  return v;
}

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
  for (int offset = kWave / 2; offset > 0; offset >>= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), offset, kWave));
    v = o > v ? o : v;
  }
  return v;
}

__device__ __forceinline__ uint32_t wave_inclusive_sum_u32(uint32_t v) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int offset = 1; offset < kWave; offset <<= 1) {
    const uint32_t t = static_cast<uint32_t>(__shfl_up(static_cast<int>(v), offset, kWave));
    if (lane >= offset) v += t;
  }
  return v;
}

// Barrier of kThreads threads that sort a list together: a wave, which runs its LDS and
// memory instructions in order and waits only for the compiler, or the whole workgroup.
template <int kThreads>
__device__ __forceinline__ void team_sync() {
  if constexpr (kThreads == kWave) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// The calling thread's number among the kThreads that sort a list together.
template <int kThreads>
__device__ __forceinline__ uint32_t team_thread() {
  return kThreads == kWave ? threadIdx.x & (kWave - 1) : threadIdx.x;
}

// Smallest and largest of the team's (lo, hi); ends behind a barrier that also orders
// LDS writes made before the call.
template <typename S>
__device__ __forceinline__ void block_min_max(S& s, uint32_t& lo, uint32_t& hi) {
  const uint32_t t = team_thread<S::kWaves * kWave>();
  lo = wave_min_u32(lo);
  hi = wave_max_u32(hi);
  if ((t & (kWave - 1)) == 0) {
    s.wave_a[t / kWave] = lo;
    s.wave_b[t / kWave] = hi;
  }
  team_sync<S::kWaves * kWave>();
#pragma unroll
  for (int w = 0; w < S::kWaves; ++w) {
    lo = s.wave_a[w] < lo ? s.wave_a[w] : lo;
    hi = s.wave_b[w] > hi ? s.wave_b[w] : hi;
  }
}

// Sorts n <= kCapacity entries by (key, tie(value)) and hands every entry with
// its rank to emit(rank, key, value).  key_of(i) and value_of(i) load entry i;
// every load is done before the first emit.  `tie` is consulted only between
// equal keys and must tell all values apart.  Without kSplit a crowded list of
// more than kSplitLeast entries is refused: false is returned and nothing
// emitted.  The caller synchronizes before the call if other threads may still
// read `s`, and before it writes to `s` again.  Nobody else writes the entries
// during the call: the split loads them again and relies on finding the same.
template <bool kSplit, int kThreads, int kCapacity, int kBins, typename Key, typename Value, typename Tie,
          typename Emit>
__device__ __forceinline__ bool tile_sort(TileSort<kThreads, kCapacity, kBins>& s, uint32_t n, Key&& key_of,
                                          Value&& value_of, Tie&& tie, Emit&& emit) {
  using S = TileSort<kThreads, kCapacity, kBins>;
  constexpr int kItems = S::kItems;
  const uint32_t t = team_thread<kThreads>();
  const int lane = t & (kWave - 1);
  const int wave = t / kWave;
  uint32_t keys[kItems];
  int32_t values[kItems];
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    const uint32_t i = r * kThreads + t;
    keys[r] = i < n ? key_of(i) : 0u;
    values[r] = i < n ? value_of(i) : 0;
  }
  const auto less = [&](uint32_t ka, int32_t va, uint32_t kb, int32_t vb) {
    return ka < kb || (ka == kb && tie(va) < tie(vb));
  };
  // About one bin per entry; every thread scans the same number of bins.
  uint32_t per = (n + kThreads - 1) / kThreads;
  per = per < kBins / kThreads ? per : kBins / kThreads;
  const uint32_t bins = per * kThreads;
  for (uint32_t i = t; i < bins; i += kThreads) s.start[i] = 0u;
  uint32_t lo = 0xffffffffu, hi = 0u;
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    if (r * kThreads + t < n) {
      lo = keys[r] < lo ? keys[r] : lo;
      hi = keys[r] > hi ? keys[r] : hi;
    }
  }
  block_min_max(s, lo, hi);
  const BinMap bin_of(lo, hi, bins);
  uint32_t ranks[kItems];
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    ranks[r] = 0u;
    if (r * kThreads + t < n) ranks[r] = atomicAdd(&s.start[bin_of(keys[r])], 1u);
  }
  team_sync<kThreads>();
  // Exclusive scan of the counters (per consecutive bins per thread) and the fullest bin.
  uint32_t own = 0u, fullest = 0u;
  for (uint32_t b = 0; b < per; ++b) {
    const uint32_t c = s.start[t * per + b];
    own += c;
    fullest = c > fullest ? c : fullest;
  }
  const uint32_t inclusive = wave_inclusive_sum_u32(own);
  fullest = wave_max_u32(fullest);
  if (lane == kWave - 1) {
    s.wave_a[wave] = inclusive;
    s.wave_b[wave] = fullest;
  }
  team_sync<kThreads>();
  uint32_t running = inclusive - own;
#pragma unroll
  for (int w = 0; w < S::kWaves; ++w) {
    if (w < wave) running += s.wave_a[w];
    fullest = s.wave_b[w] > fullest ? s.wave_b[w] : fullest;
  }
  const bool crowded = fullest > S::kCrowd;  // uniform over the workgroup
  if (!kSplit && crowded && n > kSplitLeast) return false;
  for (uint32_t b = 0; b < per; ++b) {
    const uint32_t c = s.start[t * per + b];
    s.start[t * per + b] = running;
    running += c;
  }
  if (t == 0) s.start[bins] = n;
  // Part of a crowded list's entry: bin b's entries share the numbers [start(b), start(b + 1)).
  const auto part_of = [&](uint32_t key) {
    const uint32_t bin = bin_of(key);
    const uint32_t first = s.start[bin];
    return first + __umulhi(bin_of.fraction(key), s.start[bin + 1] - first);
  };
  team_sync<kThreads>();
  if (kSplit && crowded) {
    // The entries are loaded again rather than kept: registers that only this path
    // uses would cost every list some of its waves.
    uint32_t* const parts = reinterpret_cast<uint32_t*>(s.values);
    for (uint32_t i = t; i < n; i += kThreads) parts[i] = 0u;
    team_sync<kThreads>();
#pragma unroll 1
    for (uint32_t i = t; i < n; i += kThreads) atomicAdd(&parts[part_of(key_of(i))], 1u);
    team_sync<kThreads>();
    const uint32_t share = (n + kThreads - 1) / kThreads;
    const uint32_t share_begin = t * share, share_end = share_begin + share < n ? share_begin + share : n;
    own = 0u;
    fullest = 0u;
#pragma unroll 1
    for (uint32_t i = share_begin; i < share_end; ++i) {
      const uint32_t c = parts[i];
      own += c;
      fullest = c > fullest ? c : fullest;
    }
    const uint32_t up_to = wave_inclusive_sum_u32(own);
    fullest = wave_max_u32(fullest);
    if (lane == kWave - 1) {
      s.wave_a[wave] = up_to;
      s.wave_b[wave] = fullest;
    }
    team_sync<kThreads>();
    running = up_to - own;
    for (int w = 0; w < S::kWaves; ++w) {
      if (w < wave) running += s.wave_a[w];
      fullest = s.wave_b[w] > fullest ? s.wave_b[w] : fullest;
    }
#pragma unroll 1
    for (uint32_t i = share_begin; i < share_end; ++i) {
      const uint32_t c = parts[i];
      parts[i] = running;
      running += c;
    }
    team_sync<kThreads>();
#pragma unroll 1
    for (uint32_t i = t; i < n; i += kThreads) s.keys[atomicAdd(&parts[part_of(key_of(i))], 1u)] = i;
    team_sync<kThreads>();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const uint32_t i = r * kThreads + t;
      const uint32_t entry = i < n ? s.keys[i] : 0u;
      keys[r] = key_of(entry);
      values[r] = value_of(entry);
    }
    team_sync<kThreads>();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
      const uint32_t i = r * kThreads + t;
      if (i < n) {
        s.keys[i] = keys[r];
        s.values[i] = values[r];
      }
    }
    team_sync<kThreads>();
    if (fullest <= S::kPartCrowd) {  // uniform over the workgroup
#pragma unroll 1
      for (uint32_t i = t; i < n; i += kThreads) {
        // The neighbours in the same part, which lies around the entry.
        const uint32_t key = s.keys[i];
        const int32_t value = s.values[i];
        const uint32_t part = part_of(key);
        uint32_t rank = i;
        for (uint32_t j = i; j-- > 0u && part_of(s.keys[j]) == part;) {
          if (less(key, value, s.keys[j], s.values[j])) --rank;
        }
        for (uint32_t j = i + 1u; j < n && part_of(s.keys[j]) == part; ++j) {
          if (less(s.keys[j], s.values[j], key, value)) ++rank;
        }
        emit(rank, key, value);
      }
      return true;
    }
    uint32_t padded = 2u;
    while (padded < n) padded <<= 1;
    for (uint32_t size = 2u; size <= padded; size <<= 1) {
      for (uint32_t stride = size >> 1; stride > 0u; stride >>= 1) {
#pragma unroll 1
        for (uint32_t i = t; i < padded / 2u; i += kThreads) {
          // The first step of a merge pairs mirrored entries, so every block ascends
          // and the padding behind entry n would never move: its pairs are skipped.
          const uint32_t low_bits = i & (stride - 1u);
          const uint32_t a = ((i - low_bits) << 1) + low_bits;
          const uint32_t b = stride == (size >> 1) ? ((i - low_bits) << 1) + size - 1u - low_bits : a + stride;
          if (b < n) {
            const uint32_t ka = s.keys[a], kb = s.keys[b];
            const int32_t va = s.values[a], vb = s.values[b];
            if (less(kb, vb, ka, va)) {
              s.keys[a] = kb;
              s.values[a] = vb;
              s.keys[b] = ka;
              s.values[b] = va;
            }
          }
        }
        team_sync<kThreads>();
      }
    }
    for (uint32_t i = t; i < n; i += kThreads) emit(i, s.keys[i], s.values[i]);
    return true;
  }
#pragma unroll
  for (int r = 0; r < kItems; ++r) {
    if (r * kThreads + t < n) {
      const uint32_t position = s.start[bin_of(keys[r])] + ranks[r];
      s.keys[position] = keys[r];
      s.values[position] = values[r];
    }
  }
  team_sync<kThreads>();
  // Not unrolled: the workgroups sharing the CU hide the reads, and the registers
  // that eight bins at a time would take cost some of them.
#pragma unroll 1
  for (uint32_t i = t; i < n; i += kThreads) {
    const uint32_t key = s.keys[i];
    const int32_t value = s.values[i];
    const uint32_t bin = bin_of(key);
    const uint32_t first = s.start[bin], last = s.start[bin + 1];
    uint32_t rank = first;
    for (uint32_t j = first; j < last; ++j) {
      if (j != i && less(s.keys[j], s.values[j], key, value)) ++rank;
    }
    emit(rank, key, value);
  }
  return true;
}

}  // namespace dev
}  // namespace vgr

#endif  // VGR_TILE_SORT_DEVICE_H
