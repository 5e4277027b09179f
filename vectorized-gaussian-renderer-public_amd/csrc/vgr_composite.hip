// Fused RGB / expected-depth / alpha / semantic compositing for gfx950.
//
// Reference behaviour: composite_tiles_kernel<false,false,FULL>
// (renderer_cuda.cu:1973-2305).  One workgroup renders one (active camera,
// tile): tile_size^2 lanes, one pixel each (16x16 = four wave64s).  The
// depth-sorted intersection list of the tile is consumed in batches: every
// lane gathers whole 48-byte records (three 16-byte loads) for the next batch
// into registers while the current batch is composited out of LDS, so the
// gather latency overlaps the blend loop.  Inside the loop every lane reads
// the same LDS address, which the LDS serves as a broadcast.
//
// The per-pixel arithmetic is the reference's, term by term, with vgr_expf in
// place of __expf.  The semantic winner is tracked as a Gaussian index and the
// int64 semantic label is gathered once per pixel at the end.
#include <type_traits>

#include "vgr_composite_device.h"
#include "vgr_project_device.h"

namespace vgr {
namespace {

using namespace dev;

// ---- tile launch order -------------------------------------------------------
// Blocks sorted by descending list length (counting sort, 32 buckets an octave): the
// longest tiles start first and the short ones fill in behind them, instead of
// a long tile starting late and running alone at the end of the grid.  One
// workgroup; the order inside a length bucket is unspecified (it changes only the
// schedule: every tile's outputs are its own).  On 16 cameras of 512x512 (lists
// of ~950 entries on average, up to 5k) the forward goes 2.85 -> 2.24 ms and
// forward+backward 9.6 -> 8.0 ms.
constexpr int kOrderBuckets = 1024;
constexpr int kOrderThreads = 1024;
// A tile is long when it takes more than about half of the list entries that a CU gets on
// average: a wave that walks it alone would still run when the other CUs are done (alone
// on its SIMD a wave takes some 390 cycles an entry, a full CU 180).  What a tile takes is
// its reach where that is known (tile_reach_kernel), else the length of its list, of
// which up to 4,096 entries count towards the average, since a tile with more is mostly
// opaque before its end.  By length, 0.45 and 0.5: a VGA view of 1M Gaussians 195 and 175
// us, of 300k 102 and 108, four 320x240 views in a room of 500k 163 and 189; by reach,
// which overestimates the sum more than the longest, 0.40 and 0.43: 16 views of 128x128
// over 300k 586 and 490, 48 room cameras of 160x120 1,203 and 1,278.
constexpr int32_t kLongCap = 4096;
constexpr float kLongReachShare = 0.43f / 256.0f;
constexpr float kLongShare = 0.5f / 256.0f;
// Where whole and long tiles compete for the CUs (three workgroups and more a CU) and the
// lists are long (5,000 entries on average, known on the device only), the reach decides
// instead of the length, for 11 to 16 us.  No tile long / by length / by reach, with
// those: 16 views of 128x128 over an open 1M 583 / 774 / 537 us and 300k 508 / 560 / 500,
// 13 of 700k 600 / 595 / 526, ten 160x120 views of 1M 461 / 548 / 461, 16 room cameras of
// 128x128 over 5M 517 / 345 / 318; but twelve of 160x120 over 3M 289 / 280 / 340.  With
// shorter lists it gains little and may lose: two 480x320 views of 1M (lists of 2,781)
// 222 / 254 / 225, four 320x240 views of 500k 307 / 311 / 304, 48 room cameras of 160x120
// in three submissions 1,906 / 1,182 / 1,304.  A capacity that was fixed beforehand does
// not hint at long lists, and finding none on the device costs such a submission 10 us, 1
// % of those room cameras' 2.9 ms: there the length decides.
constexpr int64_t kReachTiles = 768;
constexpr int64_t kReachLists = 5000;

__device__ __forceinline__ int32_t list_length(const CameraParams* __restrict__ table,
                                               const int32_t* __restrict__ tile_starts,
                                               const int32_t* __restrict__ tile_ends, int active_count,
                                               int uniform_tiles, const int32_t* __restrict__ reach, int64_t block) {
  if (reach != nullptr) return reach[block];
  int active;
  int64_t image_tile;
  if (uniform_tiles > 0) {
    active = static_cast<int>(block / uniform_tiles);
    if (active >= active_count) return 0;
    image_tile = block - static_cast<int64_t>(active) * uniform_tiles;
  } else {
    active = find_active_camera(table, active_count, block);
    image_tile = block - table[active].active_tile_begin;
    if (image_tile >= static_cast<int64_t>(table[active].tiles_x) * table[active].tiles_y) return 0;
  }
  if (table[active].camera < 0) return 0;
  const uint32_t global_tile = table[active].tile_base + static_cast<uint32_t>(image_tile);
  const int64_t start = tile_starts[global_tile];
  const int64_t end = tile_ends[global_tile];
  return static_cast<int32_t>(start >= 0 && end > start ? end - start : 0);
}

// Empty lists, then 32 buckets an octave (at most 31 octaves).
__device__ __forceinline__ int order_bucket(int32_t length) {
  return length <= 0 ? 0 : static_cast<int>(__float_as_uint(static_cast<float>(length)) >> 18) - (127 << 5) + 1;
}

__global__ __launch_bounds__(kOrderThreads) void tile_order_kernel(const CameraParams* __restrict__ table,
                                                                   const int32_t* __restrict__ tile_starts,
                                                                   const int32_t* __restrict__ tile_ends,
                                                                   int active_count, int uniform_tiles, int64_t blocks,
                                                                   const int32_t* __restrict__ reach,
                                                                   const int64_t* __restrict__ intersections,
                                                                   int32_t* __restrict__ order,
                                                                   uint32_t* __restrict__ long_tiles) {
  if (reach != nullptr && *intersections < blocks * kReachLists) reach = nullptr;  // uniform: not written either
  __shared__ uint32_t s_next[kOrderBuckets];
  __shared__ uint32_t s_wave_totals[kOrderThreads / kWave];
  __shared__ float s_wave_entries[kOrderThreads / kWave];
  for (int i = threadIdx.x; i < kOrderBuckets; i += kOrderThreads) s_next[i] = 0;
  __syncthreads();
  float entries = 0.0f;
  for (int64_t b = threadIdx.x; b < blocks; b += kOrderThreads) {
    const int32_t length = list_length(table, tile_starts, tile_ends, active_count, uniform_tiles, reach, b);
    atomicAdd(&s_next[order_bucket(length)], 1u);
    entries += static_cast<float>(reach != nullptr || length < kLongCap ? length : kLongCap);
  }
  if (long_tiles != nullptr) {  // uniform
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) entries += __shfl_xor(entries, offset, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) s_wave_entries[threadIdx.x / kWave] = entries;
  }
  __syncthreads();
  // Exclusive scan in descending bucket order: thread t owns bucket kOrderBuckets-1-t.
  static_assert(kOrderBuckets == kOrderThreads, "one bucket per thread");
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int bucket = kOrderBuckets - 1 - static_cast<int>(threadIdx.x);
  const uint32_t count = s_next[bucket];
  uint32_t inclusive = count;
#pragma unroll
  for (int offset = 1; offset < kWave; offset <<= 1) {
    const uint32_t t = __shfl_up(inclusive, offset, kWave);
    if (lane >= offset) inclusive += t;
  }
  if (lane == kWave - 1) s_wave_totals[wave] = inclusive;
  __syncthreads();
  uint32_t prefix = 0;
  for (int w = 0; w < wave; ++w) prefix += s_wave_totals[w];
  s_next[bucket] = prefix + inclusive - count;
  if (long_tiles != nullptr) {
    float total = 0.0f;
    for (int w = 0; w < kOrderThreads / kWave; ++w) total += s_wave_entries[w];
    const int limit = order_bucket(static_cast<int32_t>(total * (reach != nullptr ? kLongReachShare : kLongShare)));
    if (bucket == limit) *long_tiles = prefix + inclusive - count;  // the tiles of the buckets above
  }
  __syncthreads();
  for (int64_t b = threadIdx.x; b < blocks; b += kOrderThreads) {
    const int k = order_bucket(list_length(table, tile_starts, tile_ends, active_count, uniform_tiles, reach, b));
    order[atomicAdd(&s_next[k], 1u)] = static_cast<int32_t>(b);
  }
}

struct CompositeArgs {
  const CameraParams* table;
  const int32_t* tile_starts;
  const int32_t* tile_ends;
  const int32_t* sorted_values;
  const vgr_record* records;
  const int64_t* semantic_ids;
  float* rgb;
  float* depth;
  float* alpha;
  int64_t* semantic;
  int64_t* statistics;   // optional: [0] += evaluated (pixel, Gaussian) pairs
  int64_t visible_capacity;
  int64_t gaussian_count;
  uint32_t* work_counter;  // queue of the tiles left open (zeroed before the launch)
  const int32_t* tile_order;  // launch order of the (camera, tile) items
  const uint32_t* long_tiles;  // how many of the first in that order are long
  int64_t total_items;     // (camera, tile) items in the launch
  int64_t first_item;      // of this launch: a grid holds less than 2^32 threads
  int active_count;
  int uniform_tiles;     // tiles per camera when every camera has the same resolution, else 0
  int output_srgb;
  float semantic_min_alpha;
  float* final_transmittance;  // optional per-pixel checkpoint (training forward)
  int32_t* last_blended;       // optional: tile-list position one past the last blended splat
  const int32_t* slot_records;  // training forward: the sorted values are slots, mapped to records here
};

// Tile-front ordering: the lists hold packed Gaussian indices (the records are
// recomputed from the scene), a list may be a truncated front of the tile's
// bucket (front_lengths = full bucket sizes), and a tile with a pixel still
// open at the end of a truncated list is appended to open_tiles.
struct FrontCompositeArgs : CompositeArgs {
  ProjectionArgs projection;
  const int32_t* front_lengths;  // null: no open-tile detection (the recomposite pass)
  int32_t* open_tiles;
  uint32_t* open_count;
  const uint32_t* item_count;  // the pass over the tiles left open: their count, on the device
};

template <int kDegree>
using CompositeArgsFor = typename std::conditional<(kDegree < 0), CompositeArgs, FrontCompositeArgs>::type;

// Writes a finished pixel (renderer_cuda.cu:2264-2304).
template <bool kFull>
__device__ __forceinline__ void store_pixel(const CompositeArgs& args, int64_t pixel, float transmittance, float red,
                                            float green, float blue, float depth_sum, float best_weight,
                                            int best_gaussian) {
  const float accumulated_alpha = 1.0f - transmittance;
  if (args.output_srgb) {
    red = vgr_linear_to_srgb(red);
    green = vgr_linear_to_srgb(green);
    blue = vgr_linear_to_srgb(blue);
  }
  args.rgb[pixel * 3 + 0] = red;
  args.rgb[pixel * 3 + 1] = green;
  args.rgb[pixel * 3 + 2] = blue;
  if (kFull) {
    args.alpha[pixel] = accumulated_alpha;
    args.depth[pixel] = accumulated_alpha > 1.0e-8f ? depth_sum / accumulated_alpha : __int_as_float(0x7f800000);
    const bool labelled = best_weight >= 0.0f && accumulated_alpha >= args.semantic_min_alpha &&
                          best_gaussian >= 0 && best_gaussian < args.gaussian_count;
    args.semantic[pixel] = labelled ? args.semantic_ids[best_gaussian] : -1;
  }
}

// Gathers one batch: stored records (kDegree < 0) or records recomputed from
// the listed Gaussians (kDegree = SH degree, tile-front lists).
template <int kThreads, int kBatch, int kPerThread, int kDegree, bool kSlots = false>
__device__ __forceinline__ void gather_any(const CompositeArgsFor<kDegree>& args, const CameraParams& cam,
                                           int64_t batch_start,
                                           int64_t range_end, int lane, f32x4 (&a)[kPerThread],
                                           f32x4 (&b)[kPerThread], f32x4 (&c)[kPerThread]) {
  if constexpr (kDegree < 0) {
    gather_batch<kThreads, kBatch, kPerThread, kSlots>(args.sorted_values, args.records, args.visible_capacity,
                                                       batch_start, range_end, lane, a, b, c, args.slot_records);
  } else {
#pragma unroll
    for (int k = 0; k < kPerThread; ++k) {
      const int64_t index = batch_start + k * kThreads + lane;
      if (k * kThreads + lane < kBatch && index < range_end) {
        const int32_t g = args.sorted_values[index];
        if (g >= 0 && g < args.projection.gaussian_count) {
          record_from_gaussian<kDegree>(args.projection, cam, g, a[k], b[k], c[k]);
        } else {
          a[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          b[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          c[k] = f32x4{0.0f, 0.0f, __int_as_float(-1), 0.0f};
        }
      }
    }
  }
}

// Renders one (active camera, tile) work item with the whole workgroup.  With
// kCheckpoint the final transmittance and the list position one past the last
// blended splat are stored per pixel for the backward pass.
template <int kTileSize, int kBatch, bool kFull, bool kCount, bool kCheckpoint, int kDegree = -1>
__device__ __forceinline__ void composite_tile(const CompositeArgsFor<kDegree>& args, int64_t block,
                                               WaveLists<kTileSize, kBatch>& s) {
  using Lists = WaveLists<kTileSize, kBatch>;
  constexpr int kThreads = Lists::kThreads;
  constexpr int kPerThread = Lists::kPerThread;
  static_assert(kThreads % kWave == 0, "tile must be a whole number of waves");

  int active;
  int64_t image_tile;
  if (args.uniform_tiles > 0) {
    active = static_cast<int>(block / args.uniform_tiles);
    if (active >= args.active_count) return;
    image_tile = block - static_cast<int64_t>(active) * args.uniform_tiles;
  } else {
    active = find_active_camera(args.table, args.active_count, block);
    image_tile = block - args.table[active].active_tile_begin;
    if (image_tile >= static_cast<int64_t>(args.table[active].tiles_x) * args.table[active].tiles_y) return;
  }
  const CameraParams& cam = args.table[active];
  if (cam.camera < 0) return;
  const int tile_x = static_cast<int>(image_tile % cam.tiles_x);
  const int tile_y = static_cast<int>(image_tile / cam.tiles_x);
  const uint32_t global_tile = cam.tile_base + static_cast<uint32_t>(image_tile);
  const int lane = threadIdx.x;
  const int wave = lane / kWave;
  const int pixel_x = tile_x * kTileSize + Lists::pixel_dx(lane);
  const int pixel_y = tile_y * kTileSize + Lists::pixel_dy(lane);
  const bool valid_pixel = pixel_x < cam.width && pixel_y < cam.height;
  const float px = static_cast<float>(pixel_x) + 0.5f;
  const float py = static_cast<float>(pixel_y) + 0.5f;
  // Pixel-centre rectangle of tile column span and of each wave's rows.
  const float rect_x0 = static_cast<float>(tile_x * kTileSize) + 0.5f;
  const float rect_y_base = static_cast<float>(tile_y * kTileSize) + 0.5f;

  float transmittance = 1.0f;
  float red = 0.0f, green = 0.0f, blue = 0.0f, depth_sum = 0.0f;
  float best_weight = -1.0f;
  int best_gaussian = -1;
  bool done = !valid_pixel;
  int evaluations = 0;
  int last_blended = 0;

  const int64_t range_start = args.tile_starts[global_tile];
  const int64_t range_end = args.tile_ends[global_tile];
  if (range_start >= 0 && range_end > range_start) {
    f32x4 next_a[kPerThread] = {}, next_b[kPerThread] = {}, next_c[kPerThread] = {};
    gather_any<kThreads, kBatch, kPerThread, kDegree, kCheckpoint>(args, cam, range_start, range_end, lane, next_a,
                                                                   next_b, next_c);
    for (int64_t batch_start = range_start; batch_start < range_end; batch_start += kBatch) {
      const int count = static_cast<int>(range_end - batch_start < kBatch ? range_end - batch_start : kBatch);
      __syncthreads();  // previous batch fully consumed
      build_wave_lists<kTileSize, kBatch>(s, next_a, next_b, next_c, count, lane, rect_x0, rect_y_base);
      if (batch_start + kBatch < range_end) {
        gather_any<kThreads, kBatch, kPerThread, kDegree, kCheckpoint>(args, cam, batch_start + kBatch, range_end,
                                                                       lane, next_a, next_b, next_c);
      }
      if (!done) {
        const uint32_t list_count = s.count(wave);
        const int position_base = static_cast<int>(batch_start - range_start);
        // Blends one evaluated splat; returns true when the pixel terminates.
        auto blend = [&](int item, const f32x4& sh, float splat_alpha) -> bool {
          if (splat_alpha < VGR_ALPHA_THRESHOLD) return false;
          const float next_transmittance = transmittance * (1.0f - splat_alpha);
          if (next_transmittance <= VGR_TRANSMITTANCE_THRESHOLD) return true;
          const f32x4 col = s.colour[item];
          const float weight = transmittance * splat_alpha;
          red = fmaf(weight, col.x, red);
          green = fmaf(weight, col.y, green);
          blue = fmaf(weight, col.z, blue);
          if (kFull) {
            depth_sum = fmaf(weight, sh.w, depth_sum);
            if (weight > best_weight) {
              best_weight = weight;
              best_gaussian = __float_as_int(col.w);
            }
          }
          if (kCheckpoint) last_blended = position_base + item + 1;
          transmittance = next_transmittance;
          return false;
        };
        uint32_t i = 0;
        // kUnroll list entries per iteration: their powers and exponentials are
        // independent and overlap (the loop is latency-bound); blending stays in
        // list order, so the per-pixel result is unchanged.
        constexpr int kUnroll = 4;
        for (; i + kUnroll <= list_count; i += kUnroll) {
          int items[kUnroll];
          f32x4 shading[kUnroll];
          float alphas[kUnroll];
          bool passes[kUnroll];
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) items[u] = s.list[wave][i + u];
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) {
            const f32x4 g = s.geometry[items[u]];
            shading[u] = s.shading[items[u]];
            const float dx = px - g.x, dy = py - g.y;
            const float power = g.z * dx * dx + g.w * dx * dy + shading[u].x * dy * dy;
            passes[u] = !(power > 0.0f || power < shading[u].z);
            alphas[u] = passes[u] ? fminf(VGR_MAX_ALPHA, shading[u].y * vgr_expf_bounded(power)) : 0.0f;
          }
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) {
            if (done) break;
            if (kCount) ++evaluations;
            if (passes[u] && blend(items[u], shading[u], alphas[u])) done = true;
          }
          if (done) break;
        }
        while (!done && i < list_count) {
          const int item = s.list[wave][i++];
          if (kCount) ++evaluations;
          const f32x4 g = s.geometry[item];
          const f32x4 sh = s.shading[item];
          const float delta_x = px - g.x;
          const float delta_y = py - g.y;
          const float power = g.z * delta_x * delta_x + g.w * delta_x * delta_y + sh.x * delta_y * delta_y;
          if (!(power > 0.0f || power < sh.z)) {
            if (blend(item, sh, fminf(VGR_MAX_ALPHA, sh.y * vgr_expf_bounded(power)))) done = true;
          }
        }
      }
      if (!__syncthreads_or(done ? 0 : 1)) break;
    }
  }
  if constexpr (kDegree >= 0) {
    if (args.front_lengths != nullptr) {
      // Truncated list with a pixel still open: the rest of the bucket matters;
      // the tile is sorted in full and composited again.
      const int64_t full = args.front_lengths[global_tile];
      const bool truncated = (range_start >= 0 && range_end > range_start ? range_end - range_start : 0) < full;
      if (truncated && __syncthreads_or(done ? 0 : 1) && threadIdx.x == 0) {
        args.open_tiles[atomicAdd(args.open_count, 1u)] = static_cast<int32_t>(global_tile);
      }
    }
  }

  if (kCount) {
    int64_t total = evaluations;
    for (int offset = 32; offset > 0; offset >>= 1) total += __shfl_xor(total, offset, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0 && total != 0) {
      atomicAdd(reinterpret_cast<unsigned long long*>(args.statistics), static_cast<unsigned long long>(total));
    }
  }
  if (!valid_pixel) return;
  const int64_t pixel = cam.pixel_offset + static_cast<int64_t>(pixel_y) * cam.width + pixel_x;
  store_pixel<kFull>(args, pixel, transmittance, red, green, blue, depth_sum, best_weight, best_gaussian);
  if (kCheckpoint) {
    args.final_transmittance[pixel] = transmittance;
    args.last_blended[pixel] = last_blended;
  }
}

// ---- how far tiles are composited --------------------------------------------------
//
// A tile's work is the part of its list up to where its last pixel turns opaque, which
// the length of the list says little about: tiles of a room that look out of it are
// read to the end, while 128x128 views of an open million are opaque after 5,000 entries
// of lists of up to 107,000.  A workgroup per tile samples the front of the list and adds up,
// at 8x8 points of the tile, the optical thickness that every sample spreads there (its
// integral over the plane, as a Gaussian widened so that small splats count for their
// neighbourhood); the point that takes longest to pass the depth at which pixels end
// sets the tile's.  Only the schedule depends on it.  A model of it with the crossing
// sample instead of the interpolated part, against the entries that are read, on four
// workloads of 1,024 and 1,280 tiles: the sum over the tiles is 1.06 to 1.39 of it, 99 %
// of the tiles of each at 0.92 of theirs or more.  Fewer points miss tiles that are open
// in one corner, which then end the grid alone.
constexpr int kReachLeast = 512;         // shorter lists are taken as they are
constexpr int kReachSpan = 8192;         // entries that the samples are spread over
constexpr int kReachWaves = 4;           // of a tile
constexpr int kReachParts = 4;           // of a wave's samples, whose sums are kept
constexpr int kReachSamples = 8;         // of a part
constexpr float kReachDepth = 1.25f * 9.21f;  // of a transmittance of 1e-4, with an allowance
constexpr float kReachWiden = 8.0f;      // variance added to a splat's
// A sample stands for up to 64 entries; where one near splat does so, it does not make
// the tile opaque alone.
constexpr float kReachSampleDepth = 2.0f;

template <bool kSlots>
__global__ __launch_bounds__(kReachWaves* kWave) void tile_reach_kernel(CompositeArgs args,
                                                                        const int64_t* __restrict__ intersections,
                                                                        int32_t* __restrict__ reach) {
  if (*intersections < static_cast<int64_t>(gridDim.x) * kReachLists) return;
  constexpr int kOwn = kReachParts * kReachSamples;  // samples of a wave
  constexpr int kCount = kReachWaves * kOwn;
  __shared__ f32x4 s_form[kCount];      // mean, xx and xy coefficients of the exponent
  __shared__ float2 s_peak[kCount];      // yy coefficient, thickness at the mean
  __shared__ float s_sums[kReachWaves * kReachParts][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t block = blockIdx.x;
  const int32_t length = list_length(args.table, args.tile_starts, args.tile_ends, args.active_count,
                                     args.uniform_tiles, nullptr, block);
  if (length <= kReachLeast) {
    if (threadIdx.x == 0) reach[block] = length;
    return;
  }
  const int active = args.uniform_tiles > 0 ? static_cast<int>(block / args.uniform_tiles)
                                            : find_active_camera(args.table, args.active_count, block);
  const CameraParams& cam = args.table[active];
  const int image_tile = static_cast<int>(block - (args.uniform_tiles > 0
                                                       ? static_cast<int64_t>(active) * args.uniform_tiles
                                                       : cam.active_tile_begin));
  const int x = image_tile % cam.tiles_x * 16 + (lane & 7) * 2, y = image_tile / cam.tiles_x * 16 + (lane >> 3) * 2;
  const int32_t span = length < kReachSpan ? length : kReachSpan;
  const float weight = static_cast<float>(span) / kCount;  // entries a sample stands for
  if (lane < kOwn) {
    const int i = wave * kOwn + lane;
    // The middle entry of those it stands for: the first of a list are the largest.
    int32_t record = args.sorted_values[args.tile_starts[cam.tile_base + static_cast<uint32_t>(image_tile)] +
                                        static_cast<int64_t>(2 * i + 1) * span / (2 * kCount)];
    if (kSlots) record = record >= 0 ? args.slot_records[record] : -1;
    f32x4 a = {}, b = {};
    if (record >= 0 && record < args.visible_capacity) {  // else a corrupted list
      const f32x4* src = reinterpret_cast<const f32x4*>(args.records + record);
      a = src[0];  // mean_x, mean_y, conic_0, conic_1
      b = src[1];  // conic_2, opacity, depth, red
    }
    const float inverse = __builtin_amdgcn_rcpf(fmaxf(a.z * b.x - a.w * a.w, 1.0e-12f));
    const float xx = b.x * inverse + kReachWiden, yy = a.z * inverse + kReachWiden, xy = -a.w * inverse;
    const float wide = __builtin_amdgcn_rcpf(xx * yy - xy * xy);
    const float scale = -0.7213475f * wide;  // -1/2 log2(e)
    s_form[i] = f32x4{a.x, a.y, scale * yy, -2.0f * scale * xy};
    // The integral of -ln(1 - alpha) over the plane is 2 pi / sqrt(det) times the
    // dilogarithm of the opacity, here its first terms.
    const float o = b.y;
    s_peak[i] = float2{scale * xx, weight * o * (1.0f + o * (0.25f + o * (0.1111f + o * 0.0625f))) *
                                      __builtin_amdgcn_sqrtf(inverse * wide)};
  }
  __syncthreads();
  const float px = static_cast<float>(x + 1), py = static_cast<float>(y + 1);
#pragma unroll
  for (int part = 0; part < kReachParts; ++part) {
    float thickness = 0.0f;
#pragma unroll
    for (int k = 0; k < kReachSamples; ++k) {
      const int i = (wave * kReachParts + part) * kReachSamples + k;
      const f32x4 form = s_form[i];
      const float2 peak = s_peak[i];
      const float dx = px - form.x, dy = py - form.y;
      const float power = dx * (form.z * dx + form.w * dy) + peak.x * dy * dy;
      thickness += fminf(kReachSampleDepth, peak.y * __builtin_amdgcn_exp2f(power));
    }
    s_sums[wave * kReachParts + part][lane] = thickness;
  }
  __syncthreads();
  if (wave != 0) return;
  // Parts up to the one in which the point's depth is passed, and the share of that one.
  float total = 0.0f, parts = 0.0f;
#pragma unroll
  for (int p = 0; p < kReachWaves * kReachParts; ++p) {
    const float own = s_sums[p][lane];
    parts += fminf(1.0f, fmaxf(0.0f, kReachDepth - total) / fmaxf(own, 1.0e-6f));
    total += own;
  }
  constexpr float kAll = kReachWaves * kReachParts;
  float entries = weight * kReachSamples * (total < kReachDepth ? kAll * kReachDepth / fmaxf(total, 1.0e-6f) : parts);
  if (x >= cam.width || y >= cam.height) entries = 0.0f;  // no pixel to finish
#pragma unroll
  for (int offset = 1; offset < kWave; offset <<= 1) entries = fmaxf(entries, __shfl_xor(entries, offset, kWave));
  if (lane == 0) reach[block] = entries < static_cast<float>(length) ? static_cast<int32_t>(entries) : length;
}

// ---- few long lists: a workgroup per 8x8 block ---------------------------------------
//
// Where a handful of tiles outlast the rest of the grid (a small image; tiles that
// look out of a closed scene and never saturate), the time is what one wave takes for
// its block's list: some 45 vector instructions an entry, four cycles each.  Only a
// third of them, the blend, has to follow the order of the list.  Here a workgroup
// renders one 8x8 block: one wave blends while three evaluate the alphas of the
// entries ahead into LDS, on the other SIMDs of the CU, and all four stage the list,
// keeping the entries whose ellipse reaches the block.  The alphas, their tests and the
// blends are those of composite_tile, in the same order.  On a full grid it costs 1.4
// to 1.7 times the time of composite_tile (every block stages the whole list, the
// alphas pass through LDS), so only long tiles take it: a 128x96 view of 20k Gaussians
// composites in 74 us instead of 126, one 320x240 view of 100k in 79 instead of 131,
// 48 room cameras of 160x120 in 1,186 instead of 1,829.
constexpr int kBlockBatch = 256;                      // list entries staged at a time, one per thread
constexpr int kBlockShare = 8;                        // entries of a step per evaluating wave
constexpr int kBlockStep = 3 * kBlockShare;
constexpr int kBlockRows = 16 * kBlockStep;           // kept entries: staged while a whole batch fits

struct BlockShared {
  f32x4 geometry[kBlockRows];
  f32x4 shading[kBlockRows];
  f32x4 colour[kBlockRows];
  int32_t position[kBlockRows];                       // list position
  float alpha[2][kBlockStep][kWave];                  // one step is blended while the next is evaluated
  uint32_t live[2][3];                                // its entries with an alpha at some pixel
  uint32_t totals[2][4];
  uint32_t open;                                      // a pixel goes on
};

template <int kTileSize, bool kFull, bool kCheckpoint, int kDegree>
__device__ __forceinline__ void composite_block(const CompositeArgsFor<kDegree>& args, int64_t block, int quadrant,
                                                BlockShared& s) {
  constexpr int kBlocksX = kTileSize / 8;
  int active;
  int64_t image_tile;
  if (args.uniform_tiles > 0) {
    active = static_cast<int>(block / args.uniform_tiles);
    if (active >= args.active_count) return;
    image_tile = block - static_cast<int64_t>(active) * args.uniform_tiles;
  } else {
    active = find_active_camera(args.table, args.active_count, block);
    image_tile = block - args.table[active].active_tile_begin;
    if (image_tile >= static_cast<int64_t>(args.table[active].tiles_x) * args.table[active].tiles_y) return;
  }
  const CameraParams& cam = args.table[active];
  if (cam.camera < 0) return;
  const uint32_t global_tile = cam.tile_base + static_cast<uint32_t>(image_tile);
  const int block_x = static_cast<int>(image_tile % cam.tiles_x) * kTileSize + (quadrant % kBlocksX) * 8;
  const int block_y = static_cast<int>(image_tile / cam.tiles_x) * kTileSize + (quadrant / kBlocksX) * 8;
  if (block_x >= cam.width || block_y >= cam.height) return;
  const int thread = threadIdx.x;
  const int lane = thread & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(thread / kWave);  // 0 blends, 1 to 3 evaluate
  const int pixel_x = block_x + (lane & 7), pixel_y = block_y + (lane >> 3);
  const bool valid_pixel = pixel_x < cam.width && pixel_y < cam.height;
  const float px = static_cast<float>(pixel_x) + 0.5f, py = static_cast<float>(pixel_y) + 0.5f;
  const float x0 = static_cast<float>(block_x) + 0.5f, y0 = static_cast<float>(block_y) + 0.5f;
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));

  float transmittance = 1.0f;
  float red = 0.0f, green = 0.0f, blue = 0.0f, depth_sum = 0.0f;
  float best_weight = -1.0f;
  int best_gaussian = -1;
  int last_blended = 0;
  bool done = !valid_pixel;

  const int64_t range_start = args.tile_starts[global_tile];
  const int64_t range_end = args.tile_ends[global_tile];
  if (range_start >= 0 && range_end > range_start) {
    // Blends the step evaluated into alpha buffer `buffer`, entries [first, first + kBlockStep).
    const auto blend_step = [&](int buffer, int first) {
      uint32_t live = s.live[buffer][0] | (s.live[buffer][1] << kBlockShare) | (s.live[buffer][2] << (2 * kBlockShare));
      live = __builtin_amdgcn_readfirstlane(live);
      constexpr int kGroup = 4;  // entries whose LDS reads are issued together
#pragma unroll
      for (int u0 = 0; u0 < kBlockStep; u0 += kGroup) {
        if (((live >> u0) & ((1u << kGroup) - 1u)) == 0u) continue;  // uniform
        float alphas[kGroup], depths[kGroup];
        f32x4 colours[kGroup];
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
          alphas[u] = s.alpha[buffer][u0 + u][lane];
          colours[u] = s.colour[first + u0 + u];
          depths[u] = kFull ? s.shading[first + u0 + u].w : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
          if (alphas[u] > 0.0f && !done) {
            const float next = transmittance * (1.0f - alphas[u]);
            if (next <= VGR_TRANSMITTANCE_THRESHOLD) {
              done = true;
            } else {
              const float weight = transmittance * alphas[u];
              red = fmaf(weight, colours[u].x, red);
              green = fmaf(weight, colours[u].y, green);
              blue = fmaf(weight, colours[u].z, blue);
              if (kFull) {
                depth_sum = fmaf(weight, depths[u], depth_sum);
                if (weight > best_weight) {
                  best_weight = weight;
                  best_gaussian = __float_as_int(colours[u].w);
                }
              }
              if (kCheckpoint) last_blended = s.position[first + u0 + u] + 1;
              transmittance = next;
            }
          }
        }
      }
    };
    // This wave's share of the step: alphas of entries that pass, else 0.
    const auto evaluate_step = [&](int buffer, int first, int kept) {
      const int share = (wave - 1) * kBlockShare;
      uint32_t live = 0u;
#pragma unroll
      for (int u = 0; u < kBlockShare; ++u) {
        const int row = first + share + u;
        if (row < kept) {  // uniform
          const f32x4 g = s.geometry[row];
          const f32x4 sh = s.shading[row];
          const float dx = px - g.x, dy = py - g.y;
          const float power = g.z * dx * dx + g.w * dx * dy + sh.x * dy * dy;
          const float alpha = fminf(VGR_MAX_ALPHA, sh.y * vgr_expf_bounded(power));
          const bool passes = !(power > 0.0f || power < sh.z) && alpha >= VGR_ALPHA_THRESHOLD;
          s.alpha[buffer][share + u][lane] = passes ? alpha : 0.0f;
          if (__ballot(passes) != 0ull) live |= 1u << u;
        } else {
          s.alpha[buffer][share + u][lane] = 0.0f;
        }
      }
      if (lane == 0) s.live[buffer][wave - 1] = live;
    };

    f32x4 next_a[1] = {}, next_b[1] = {}, next_c[1] = {};
    gather_any<kBlockBatch, kBlockBatch, 1, kDegree, kCheckpoint>(args, cam, range_start, range_end, thread, next_a,
                                                                 next_b, next_c);
    int64_t batch_start = range_start;
    int parity = 0;
    while (batch_start < range_end) {  // uniform
      // Stage batches while another one fits the rows whole.
      int kept = 0;
      while (batch_start < range_end && kept <= kBlockRows - kBlockBatch) {
        const bool listed = batch_start + thread < range_end;
        StagedSplat staged;
        bool keep = false;
        if (listed) {
          staged = stage_record(next_a[0], next_b[0], next_c[0]);
          const SplatReach reach(next_a[0], next_b[0], staged.shading.z);
          keep = reach.hits(x0, y0, 7.0f, 7.0f);
        }
        const uint64_t vote = __ballot(keep);
        if (lane == 0) s.totals[parity][wave] = static_cast<uint32_t>(__popcll(vote));
        __syncthreads();
        int row = kept + static_cast<int>(__popcll(vote & below));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int total = static_cast<int>(s.totals[parity][q]);
          if (q < wave) row += total;
          kept += total;
        }
        parity ^= 1;  // the next batch's totals do not meet late readers of these
        if (keep) {
          s.geometry[row] = staged.geometry;
          s.shading[row] = staged.shading;
          s.colour[row] = staged.colour;
          s.position[row] = static_cast<int32_t>(batch_start - range_start) + thread;
        }
        batch_start += kBlockBatch;
        if (batch_start < range_end) {
          gather_any<kBlockBatch, kBlockBatch, 1, kDegree, kCheckpoint>(args, cam, batch_start, range_end, thread,
                                                                       next_a, next_b, next_c);
        }
      }
      __syncthreads();
      // Steps: wave 0 blends one behind the evaluating waves.
      int buffer = 0;
      for (int first = 0; first < kept + kBlockStep; first += kBlockStep, buffer ^= 1) {
        if (wave == 0) {
          if (first > 0) blend_step(buffer ^ 1, first - kBlockStep);
        } else if (first < kept) {
          evaluate_step(buffer, first, kept);
        }
        __syncthreads();
      }
      if (wave == 0) {
        const uint64_t going = __ballot(!done);
        if (lane == 0) s.open = going != 0ull ? 1u : 0u;
      }
      __syncthreads();
      if (s.open == 0u) break;  // uniform
    }
  }
  if (wave != 0 || !valid_pixel) return;
  const int64_t pixel = cam.pixel_offset + static_cast<int64_t>(pixel_y) * cam.width + pixel_x;
  store_pixel<kFull>(args, pixel, transmittance, red, green, blue, depth_sum, best_weight, best_gaussian);
  if (kCheckpoint) {
    args.final_transmittance[pixel] = transmittance;
    args.last_blended[pixel] = last_blended;
  }
}

template <int kTileSize, bool kFull, bool kCheckpoint>
__global__ __launch_bounds__(kBlockBatch) void composite_block_kernel(CompositeArgs args) {
  __shared__ BlockShared s;
  constexpr int kBlocks = kTileSize * kTileSize / 64;
  composite_block<kTileSize, kFull, kCheckpoint, -1>(args, args.tile_order[blockIdx.x / kBlocks],
                                                     static_cast<int>(blockIdx.x % kBlocks), s);
}

// Over a queue of tiles whose length is known on the device only.
template <int kTileSize, bool kFull, bool kCheckpoint, int kDegree>
__global__ __launch_bounds__(kBlockBatch) void composite_block_persistent_kernel(CompositeArgsFor<kDegree> args) {
  constexpr int kBlocks = kTileSize * kTileSize / 64;
  __shared__ BlockShared s;
  __shared__ int64_t s_item;
  const int64_t total = static_cast<int64_t>(*args.item_count) * kBlocks;
  for (;;) {
    if (threadIdx.x == 0) s_item = static_cast<int64_t>(atomicAdd(args.work_counter, 1u));
    __syncthreads();
    const int64_t item = s_item;
    __syncthreads();
    if (item >= total) break;
    composite_block<kTileSize, kFull, kCheckpoint, kDegree>(
        args, args.tile_order[item / kBlocks], static_cast<int>(item % kBlocks), s);
    __syncthreads();
  }
}

// ---- small tiles (1x1, 2x2, 4x4): one thread per pixel ---------------------------
//
// The tile lists are short and private to a few pixels, so there is nothing to
// stage in LDS: each thread walks its tile's list with direct record loads (the
// threads of one tile read the same records, which the caches share).  The
// per-pixel equation is the tiled compositor's: the same alpha test, blend,
// stop rule, depth normalisation and semantic pick (renderer_cuda.cu:2076-2304).
template <bool kFull, bool kCount>
__global__ __launch_bounds__(256) void composite_pixels_kernel(CompositeArgs args, int tile_size,
                                                               int64_t thread_count) {
  const int64_t index = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (index >= thread_count) return;
  const int tile_pixels = tile_size * tile_size;
  const int64_t block = index / tile_pixels;
  const int local = static_cast<int>(index - block * tile_pixels);
  int active;
  int64_t image_tile;
  if (args.uniform_tiles > 0) {
    active = static_cast<int>(block / args.uniform_tiles);
    if (active >= args.active_count) return;
    image_tile = block - static_cast<int64_t>(active) * args.uniform_tiles;
  } else {
    active = find_active_camera(args.table, args.active_count, block);
    image_tile = block - args.table[active].active_tile_begin;
    if (image_tile >= static_cast<int64_t>(args.table[active].tiles_x) * args.table[active].tiles_y) return;
  }
  const CameraParams& cam = args.table[active];
  if (cam.camera < 0) return;
  const int tile_x = static_cast<int>(image_tile % cam.tiles_x);
  const int tile_y = static_cast<int>(image_tile / cam.tiles_x);
  const int pixel_x = tile_x * tile_size + local % tile_size;
  const int pixel_y = tile_y * tile_size + local / tile_size;
  if (pixel_x >= cam.width || pixel_y >= cam.height) return;
  const uint32_t global_tile = cam.tile_base + static_cast<uint32_t>(image_tile);
  const float px = static_cast<float>(pixel_x) + 0.5f;
  const float py = static_cast<float>(pixel_y) + 0.5f;

  float transmittance = 1.0f;
  float red = 0.0f, green = 0.0f, blue = 0.0f, depth_sum = 0.0f;
  float best_weight = -1.0f;
  int best_gaussian = -1;
  int64_t evaluations = 0;
  const int64_t range_start = args.tile_starts[global_tile];
  const int64_t range_end = args.tile_ends[global_tile];
  for (int64_t i = range_start < 0 ? range_end : range_start; i < range_end; ++i) {
    const int32_t record = args.sorted_values[i];
    if (record < 0 || record >= args.visible_capacity) continue;  // only with a corrupted list
    const f32x4* src = reinterpret_cast<const f32x4*>(args.records + record);
    const f32x4 a = src[0];  // mean_x, mean_y, conic_0, conic_1
    const f32x4 b = src[1];  // conic_2, opacity, depth, red
    if (kCount) ++evaluations;
    const float dx = px - a.x;
    const float dy = py - a.y;
    const float power = -0.5f * (a.z * dx * dx + 2.0f * a.w * dx * dy + b.x * dy * dy);
    if (power > 0.0f || power < -20.0f) continue;
    const float alpha = fminf(VGR_MAX_ALPHA, b.y * vgr_expf_bounded(power));
    if (alpha < VGR_ALPHA_THRESHOLD) continue;
    const float next_transmittance = transmittance * (1.0f - alpha);
    if (next_transmittance <= VGR_TRANSMITTANCE_THRESHOLD) break;
    const f32x4 c = src[2];  // green, blue, gaussian id bits, camera bits
    const float weight = transmittance * alpha;
    red = fmaf(weight, b.w, red);
    green = fmaf(weight, c.x, green);
    blue = fmaf(weight, c.y, blue);
    if (kFull) {
      depth_sum = fmaf(weight, b.z, depth_sum);
      if (weight > best_weight) {
        best_weight = weight;
        best_gaussian = __float_as_int(c.z);
      }
    }
    transmittance = next_transmittance;
  }
  if (kCount) {
    int64_t total = evaluations;
    for (int offset = 32; offset > 0; offset >>= 1) total += __shfl_xor(total, offset, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0 && total != 0) {
      atomicAdd(reinterpret_cast<unsigned long long*>(args.statistics), static_cast<unsigned long long>(total));
    }
  }
  const int64_t pixel = cam.pixel_offset + static_cast<int64_t>(pixel_y) * cam.width + pixel_x;
  store_pixel<kFull>(args, pixel, transmittance, red, green, blue, depth_sum, best_weight, best_gaussian);
}

// ---- exact-ray compositing ---------------------------------------------------------
//
// One workgroup per kRaster x kRaster raster tile, reading the sorted list of the
// bin that holds it (32x32 bins under 16x16 raster tiles; bins equal raster tiles
// at 8x8).  A batch of list entries is staged in LDS (record and precision rows,
// coalesced), then every thread evaluates its pixel's ray against the batch in
// list order (renderer_cuda.cu:2176-2262): alpha is opacity x exp(-m^2/2) for the
// ray's closest approach m (0 beyond the support, capped at 1), each entry with
// alpha > 0 is blended, and the pixel stops after the entry that takes its
// transmittance to 1e-4.
//
// Bound by vector instructions on large grids and by the latency of the gathers on
// small ones.  The closest approach is first tested without its division (ray_misses),
// four entries at a time; the division, the exponential and the blend follow where a
// ray of the wave may pass within the support.  The next batch is loaded while this
// one is composited, and the raster tiles of a bin, which stage the same list, run on
// one XCD.  One VGA view of 300k Gaussians 292 -> 232 us, six 333x251 views of 200k
// 620 -> 536, four 320x240 views of 200k with 8x8 tiles 366 -> 329; 16 VGA views of 1M
// stay at 4.18 ms (86M staged entries, most of those kept hit some ray of their wave).
struct RayApproach {
  float along, cross2;  // the squared approach is mPm - cross2 / along
};

// a = (P00, 2 P01, 2 P02, P11), b = (2 P12, P22, Pm0, Pm1), c = (Pm2, mPm, opacity, depth).
__device__ __forceinline__ RayApproach ray_approach(float ray_x, float ray_y, const f32x4& a, const f32x4& b,
                                                    const f32x4& c) {
  RayApproach r;
  r.along = a.x * ray_x * ray_x + a.y * ray_x * ray_y + a.z * ray_x + a.w * ray_y * ray_y + b.x * ray_y + b.y;
  const float cross = ray_x * b.z + ray_y * b.w + c.x;
  r.cross2 = cross * cross;
  return r;
}

// The ray's alpha is 0: it runs away from the splat, or its approach is beyond the
// support by more than the rounding of the exact test in ray_alpha (mPm lowered by
// 2^-20 of itself, against 2^-24 for each of the four roundings; the constant covers
// products in the denormal range).  `limit` is the squared support raised by 2^-20.
__device__ __forceinline__ bool ray_misses(const RayApproach& r, float mpm, float limit) {
  const float beyond = fmaf(mpm, 1.0f - 0x1p-20f, -limit);
  return !(r.along > 0.0f) || r.cross2 < fmaf(beyond, r.along, -1.0e-36f);
}

__device__ __forceinline__ float ray_alpha(const RayApproach& r, float mpm, float opacity, float support_sigma) {
  const float distance2 = fmaxf(0.0f, mpm - r.cross2 / r.along);
  if (distance2 > support_sigma * support_sigma) return 0.0f;
  return fminf(1.0f, opacity * vgr_expf_nonpositive(-0.5f * distance2));
}

constexpr int kXcds = 8;
constexpr int kXcdBins = 4;  // 1, 4 and 16 measure the same within 2 %

template <int kRaster, bool kFull>
__global__ __launch_bounds__(kRaster* kRaster, kRaster == 16 ? 4 : 1) void composite_ray_kernel(CompositeArgs args,
                                                                         const float* __restrict__ ray_records,
                                                                         float support_sigma, int bins, int bin_size) {
  constexpr int kThreads = kRaster * kRaster;
  __shared__ f32x4 s_a[kThreads];
  __shared__ f32x4 s_b[kThreads];
  __shared__ f32x4 s_c[kThreads];
  __shared__ f32x4 s_colour[kThreads];  // red, green, blue, gaussian id bits
  // Each wave owns an 8x8 pixel block (16x16 raster tiles: four quadrants) and
  // walks the batch entries whose cull box reaches it, compacted in list order;
  // with 8x8 raster tiles the bin is the tile, whose box every entry reaches.
  constexpr int kWaves = kThreads / kWave;
  constexpr bool kCull = kWaves > 1;
  constexpr int kBlocksX = kRaster / 8;
  __shared__ uint16_t s_list[kWaves][kThreads];
  __shared__ uint32_t s_totals[kWaves][kWaves];  // [source wave][list]
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  const int wave_lane = static_cast<int>(threadIdx.x) & (kWave - 1);
  const int block_x0 = (wave % kBlocksX) * 8, block_y0 = (wave / kBlocksX) * 8;
  // Workgroups go round robin over the XCDs: those of one XCD (blockIdx.x mod kXcds)
  // take kXcdBins neighbouring bins at a time, the raster tiles of a bin in turn.
  const int split = bin_size / kRaster;
  const int64_t turn = (args.first_item + blockIdx.x) / kXcds;
  const int64_t bin_turn = turn / (split * split);
  const int part = static_cast<int>(turn - bin_turn * (split * split));
  const int64_t bin = (bin_turn / kXcdBins * kXcds + blockIdx.x % kXcds) * kXcdBins + bin_turn % kXcdBins;
  const int active = static_cast<int>(bin / bins);
  if (active >= args.active_count) return;
  const CameraParams& cam = args.table[active];
  if (cam.camera < 0) return;
  const int camera_bin = static_cast<int>(bin - static_cast<int64_t>(active) * bins);
  const int bin_x = camera_bin % cam.tiles_x, bin_y = camera_bin / cam.tiles_x;
  const int tile_x = bin_x * split + part % split;
  const int tile_y = bin_y * split + part / split;
  if (tile_x * kRaster >= cam.width || tile_y * kRaster >= cam.height) return;  // past a ragged edge
  const int pixel_x = tile_x * kRaster + block_x0 + (wave_lane & 7);
  const int pixel_y = tile_y * kRaster + block_y0 + (wave_lane >> 3);
  const bool valid_pixel = pixel_x < cam.width && pixel_y < cam.height;
  const uint32_t global_bin = cam.tile_base + static_cast<uint32_t>(bin_y * cam.tiles_x + bin_x);
  const float ray_x = ((static_cast<float>(pixel_x) + 0.5f) - cam.center_x) / cam.focal_x;
  const float ray_y = ((static_cast<float>(pixel_y) + 0.5f) - cam.center_y) / cam.focal_y;

  float transmittance = 1.0f;
  float red = 0.0f, green = 0.0f, blue = 0.0f, depth_sum = 0.0f;
  float best_weight = -1.0f;
  int best_gaussian = -1;
  bool done = !valid_pixel;
  const int64_t range_start = args.tile_starts[global_bin];
  const int64_t range_end = args.tile_ends[global_bin];
  const float support_limit = support_sigma * support_sigma * (1.0f + 0x1p-20f);
  if (range_start >= 0 && range_end > range_start) {
    f32x4 next_a, next_b, next_c, next_colour;
    float next_x = 0.0f, next_y = 0.0f, next_half_x = 0.0f, next_half_y = 0.0f;
    bool next_valid = false;
    const auto gather = [&](int64_t begin) {
      next_valid = false;
      if (begin + threadIdx.x >= range_end) return;
      const int32_t record = args.sorted_values[begin + threadIdx.x];
      if (record < 0 || record >= args.visible_capacity) return;  // a corrupted list: an entry that never blends
      next_valid = true;
      const f32x4* rec = reinterpret_cast<const f32x4*>(args.records + record);
      const f32x4* ray = reinterpret_cast<const f32x4*>(ray_records + static_cast<int64_t>(record) * 12);
      const f32x4 r0 = rec[0], r1 = rec[1], r2 = rec[2], q2 = ray[2];
      next_a = ray[0];
      next_b = ray[1];
      next_c = f32x4{q2.x, q2.y, r1.y, r1.z};
      next_colour = f32x4{r1.w, r2.x, r2.y, r2.z};
      next_x = r0.x;
      next_y = r0.y;
      next_half_x = q2.z;
      next_half_y = q2.w;
    };
    gather(range_start);
    for (int64_t batch_start = range_start; batch_start < range_end; batch_start += kThreads) {
      const int count = static_cast<int>(range_end - batch_start < kThreads ? range_end - batch_start : kThreads);
      __syncthreads();  // previous batch fully consumed
      uint32_t waves = 0u;
      if (static_cast<int>(threadIdx.x) < count) {
        if (next_valid) {
          s_a[threadIdx.x] = f32x4{next_a.x, 2.0f * next_a.y, 2.0f * next_a.z, next_a.w};
          s_b[threadIdx.x] = f32x4{2.0f * next_b.x, next_b.y, next_b.z, next_b.w};
          s_c[threadIdx.x] = next_c;
          s_colour[threadIdx.x] = next_colour;
          // Each wave's block of pixel centres against the entry's cull box (centre
          // next_x, next_y, half extents next_half_*): a wave outside it has alpha 0 at every
          // pixel, so the entry is left out of its list.
          waves = kCull ? 0u : 1u;
          if constexpr (kCull) {
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
              const float x0 = static_cast<float>(tile_x * kRaster + (w % kBlocksX) * 8) + 0.5f;
              const float y0 = static_cast<float>(tile_y * kRaster + (w / kBlocksX) * 8) + 0.5f;
              if (fabsf(next_x - fminf(fmaxf(next_x, x0), x0 + 7.0f)) <= next_half_x &&
                  fabsf(next_y - fminf(fmaxf(next_y, y0), y0 + 7.0f)) <= next_half_y) {
                waves |= 1u << w;
              }
            }
          }
        } else {
          s_a[threadIdx.x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          s_b[threadIdx.x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          s_c[threadIdx.x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          s_colour[threadIdx.x] = f32x4{0.0f, 0.0f, 0.0f, __int_as_float(-1)};
        }
      }
      // Per-wave lists in batch order: ballot prefix within the source wave, then
      // the totals of the source waves before it.
      int list_count = count;
      if constexpr (kCull) {
        const uint64_t below = wave_lane == 0 ? 0ull : (~0ull >> (kWave - wave_lane));
        uint32_t prefix[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const uint64_t vote = __ballot((waves >> w) & 1u);
          prefix[w] = static_cast<uint32_t>(__popcll(vote & below));
          if (wave_lane == 0) s_totals[wave][w] = static_cast<uint32_t>(__popcll(vote));
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          if ((waves >> w) & 1u) {
            uint32_t position = prefix[w];
            for (int q = 0; q < wave; ++q) position += s_totals[q][w];
            s_list[w][position] = static_cast<uint16_t>(threadIdx.x);
          }
        }
        list_count = 0;
#pragma unroll
        for (int q = 0; q < kWaves; ++q) list_count += static_cast<int>(s_totals[q][wave]);
      }
      if (batch_start + kThreads < range_end) gather(batch_start + kThreads);
      __syncthreads();
      if (!done) {
        constexpr int kUnroll = 4;
        for (int i = 0; !done && i < list_count; i += kUnroll) {
          int items[kUnroll];
          RayApproach approach[kUnroll];
          float mpm[kUnroll];
          bool hits[kUnroll];
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) {
            // Past the end the last entry again, left out below.
            const int at = i + u < list_count ? i + u : list_count - 1;
            items[u] = kCull ? static_cast<int>(s_list[wave][at]) : at;
          }
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) {
            const f32x4 c = s_c[items[u]];
            approach[u] = ray_approach(ray_x, ray_y, s_a[items[u]], s_b[items[u]], c);
            mpm[u] = c.y;
            hits[u] = i + u < list_count && !ray_misses(approach[u], c.y, support_limit);
          }
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) {
            if (!hits[u] || done) continue;
            const f32x4 c = s_c[items[u]];
            const float alpha = ray_alpha(approach[u], mpm[u], c.z, support_sigma);
            if (!(alpha > 0.0f)) continue;
            const float next_transmittance = transmittance * (1.0f - alpha);
            const f32x4 col = s_colour[items[u]];
            const float weight = transmittance * alpha;
            red = fmaf(weight, col.x, red);
            green = fmaf(weight, col.y, green);
            blue = fmaf(weight, col.z, blue);
            if (kFull) {
              depth_sum = fmaf(weight, c.w, depth_sum);
              if (weight > best_weight) {
                best_weight = weight;
                best_gaussian = __float_as_int(col.w);
              }
            }
            transmittance = next_transmittance;
            if (next_transmittance <= VGR_TRANSMITTANCE_THRESHOLD) done = true;
          }
        }
      }
      if (!__syncthreads_or(done ? 0 : 1)) break;
    }
  }
  if (!valid_pixel) return;
  const int64_t pixel = cam.pixel_offset + static_cast<int64_t>(pixel_y) * cam.width + pixel_x;
  store_pixel<kFull>(args, pixel, transmittance, red, green, blue, depth_sum, best_weight, best_gaussian);
}

// Launches items [0, blocks), one workgroup each, in grids of less than 2^32 threads,
// which is what a dispatch holds.  Slices are whole multiples of the XCD count.
template <int kThreads, typename Args, typename Launch>
void launch_slices(const Args& args, int64_t blocks, Launch&& launch) {
  constexpr int64_t kMost = ((1LL << 32) - 1) / kThreads / kXcds * kXcds;
  for (int64_t first = 0; first < blocks; first += kMost) {
    Args slice = args;
    slice.first_item = first;
    launch(slice, dim3(static_cast<unsigned>(blocks - first < kMost ? blocks - first : kMost)));
  }
}

template <int kRaster>
void launch_ray(const CompositeArgs& args, const vgr_options& options, const float* ray_records, int active_count,
                bool full, hipStream_t stream) {
  const int split = options.tile_size / kRaster;
  const int bins = args.uniform_tiles;
  constexpr int64_t kRound = kXcds * kXcdBins;
  const int64_t blocks = (static_cast<int64_t>(active_count) * bins + kRound - 1) / kRound * kRound * split * split;
  launch_slices<kRaster * kRaster>(args, blocks, [&](const CompositeArgs& slice, const dim3& grid) {
    const dim3 block(kRaster * kRaster);
    if (full) {
      hipLaunchKernelGGL((composite_ray_kernel<kRaster, true>), grid, block, 0, stream, slice, ray_records,
                         options.gaussian_support_sigma, bins, options.tile_size);
    } else {
      hipLaunchKernelGGL((composite_ray_kernel<kRaster, false>), grid, block, 0, stream, slice, ray_records,
                         options.gaussian_support_sigma, bins, options.tile_size);
    }
  });
}

// Minimum waves per SIMD for 16x16 tiles (launch-bounds occupancy target): eight
// means at most 64 VGPRs.  The blend loop is latency-bound, so waves in flight
// pay more than registers.  The evaluation-counting variant needs a few more
// registers and takes seven (no spills).
template <int kTileSize, int kBatch, bool kCount, int kDegree = -1>
constexpr int kCompositeWavesPerSimd =
    kTileSize != 16 ? 1
                    : (kDegree >= 2 ? 4  // recomputed records with SH2/3 coefficients in registers
                                    : (kDegree >= 0 ? 6
                                                    : (kBatch >= 512 ? 4 : (kCount ? 7 : 8))));

template <int kTileSize, int kBatch, bool kFull, bool kCount, bool kCheckpoint, int kDegree = -1>
__global__ __launch_bounds__(kTileSize* kTileSize, (kCompositeWavesPerSimd<kTileSize, kBatch, kCount, kDegree>)) void
composite_kernel(CompositeArgsFor<kDegree> args) {
  const int64_t block = args.tile_order != nullptr ? args.tile_order[blockIdx.x] : args.first_item + blockIdx.x;
  __shared__ WaveLists<kTileSize, kBatch> s;
  composite_tile<kTileSize, kBatch, kFull, kCount, kCheckpoint, kDegree>(args, block, s);
}

// The tiles left open, with evaluations counted: a fixed grid whose workgroups pull
// items from a device counter until the queue is empty; every workgroup exits once
// the counter passes the item count.
template <int kTileSize, int kBatch, bool kFull, bool kCount, bool kCheckpoint, int kDegree = -1>
__global__ __launch_bounds__(kTileSize* kTileSize, (kCompositeWavesPerSimd<kTileSize, kBatch, kCount, kDegree>)) void
composite_persistent_kernel(CompositeArgsFor<kDegree> args) {
  __shared__ WaveLists<kTileSize, kBatch> s;
  __shared__ int64_t s_item;
  const int64_t total = static_cast<int64_t>(*args.item_count);
  for (;;) {
    if (threadIdx.x == 0) s_item = static_cast<int64_t>(atomicAdd(args.work_counter, 1u));
    __syncthreads();
    const int64_t item = s_item;
    __syncthreads();
    if (item >= total) break;
    composite_tile<kTileSize, kBatch, kFull, kCount, kCheckpoint, kDegree>(
        args, args.tile_order[item], s);
  }
}

// The long tiles of a grid by block, the others whole.  The longest of both start
// first, four blocks and a whole tile in turn: with all blocks in front, the whole
// tiles just below the limit started late and ran on at the end (16 views of 128x128
// over 1M Gaussians: 933 us, in turn 763).
constexpr int kMixedWavesPerSimd = 5;  // what the LDS allows

template <int kBatch, bool kFull, bool kCheckpoint>
__global__ __launch_bounds__(kBlockBatch, kMixedWavesPerSimd) void composite_mixed_kernel(CompositeArgs args) {
  constexpr int kBlocks = 4;
  using Lists = WaveLists<16, kBatch>;
  __shared__ alignas(16) char lds[sizeof(Lists) > sizeof(BlockShared) ? sizeof(Lists) : sizeof(BlockShared)];
  const int64_t long_tiles = *args.long_tiles;
  const int64_t whole_tiles = args.total_items - long_tiles;
  const int64_t pairs = long_tiles < whole_tiles ? long_tiles : whole_tiles;
  const int64_t item = blockIdx.x;
  int64_t tile;
  int quadrant = -1;
  if (item < pairs * (kBlocks + 1)) {
    tile = item / (kBlocks + 1);
    quadrant = static_cast<int>(item % (kBlocks + 1));
    if (quadrant == kBlocks) {
      tile += long_tiles;
      quadrant = -1;
    }
  } else if (pairs < long_tiles) {
    const int64_t rest = item - pairs * (kBlocks + 1);
    tile = pairs + rest / kBlocks;
    quadrant = static_cast<int>(rest % kBlocks);
    if (tile >= long_tiles) return;
  } else {
    tile = item - long_tiles * (kBlocks - 1);
    if (tile >= args.total_items) return;
  }
  tile = args.tile_order[tile];
  if (quadrant >= 0) {
    composite_block<16, kFull, kCheckpoint, -1>(args, tile, quadrant, *reinterpret_cast<BlockShared*>(lds));
  } else {
    composite_tile<16, kBatch, kFull, false, kCheckpoint, -1>(args, tile, *reinterpret_cast<Lists*>(lds));
  }
}

// Grids up to this many tiles: at five workgroups a CU all of them are resident, so the
// lower occupancy of the mixed kernel (five waves a SIMD for eight) costs little.  1,200
// tiles: VGA views of 100k and 300k Gaussians 55 -> 42 and 143 -> 108 us.  At 2,400 and
// 3,600 tiles of open scenes the occupancy alone costs 36 and 41 %.
constexpr int64_t kMixedCompositeTiles = 1280;
// 8x8 tiles are a block each; up to this many all take the block kernel.  2,400 tiles
// 166 -> 81 us, 4,800 tiles 124 -> 128 (open scene) and 176 -> 115 (room); 14,400 tiles
// would go 182 -> 253.
constexpr int64_t kBlockCompositeTiles = 5120;

constexpr int kOpenWorkgroups = 256;  // of the pass over the tiles left open

template <int kTileSize, int kBatch, bool kFull, bool kCount, bool kCheckpoint = false, int kDegree = -1>
void launch_variant(const CompositeArgsFor<kDegree>& args, int64_t blocks, hipStream_t stream) {
  const dim3 block(kTileSize * kTileSize);
  constexpr int kBlocks = kTileSize * kTileSize / 64;
  if constexpr (kDegree >= 0) {
    // The tiles left open: few, with the longest lists, so always by block.  1024 room
    // cameras of 160x120 over 5M Gaussians (121 such tiles, lists up to 200k): 7.4 ->
    // 4.4 ms, 256 of 2M with checkpoints (385 tiles) 0.97 -> 0.79.
    if (args.item_count != nullptr) {
      if constexpr (kCount) {
        hipLaunchKernelGGL((composite_persistent_kernel<kTileSize, kBatch, kFull, kCount, kCheckpoint, kDegree>),
                           dim3(static_cast<unsigned>(blocks < kOpenWorkgroups ? blocks : kOpenWorkgroups)), block, 0,
                           stream, args);
      } else {
        hipLaunchKernelGGL((composite_block_persistent_kernel<kTileSize, kFull, kCheckpoint, kDegree>),
                           dim3(2 * kOpenWorkgroups), dim3(kBlockBatch), 0, stream, args);
      }
      return;
    }
  } else if constexpr (!kCount) {
    const dim3 grid(static_cast<unsigned>(blocks * kBlocks));
    if constexpr (kTileSize == 16) {
      if (blocks <= kMixedCompositeTiles) {
        hipLaunchKernelGGL((composite_mixed_kernel<kBatch, kFull, kCheckpoint>), grid, dim3(kBlockBatch), 0, stream,
                           args);
        return;
      }
    } else if (blocks <= kBlockCompositeTiles) {
      hipLaunchKernelGGL((composite_block_kernel<kTileSize, kFull, kCheckpoint>), grid, dim3(kBlockBatch), 0,
                         stream, args);
      return;
    }
  }
  // One workgroup a tile otherwise: the dispatcher hands tiles out in order as well as
  // a queue does, at eight waves a SIMD instead of six and without the queue's barriers
  // (256 cameras of four resolutions, 170k tiles: 21.1 -> 17.0 ms; tile-front lists of
  // 1024 room cameras 6.49 -> 5.87, of 256 with checkpoints 2.66 -> 2.39).
  launch_slices<kTileSize * kTileSize>(args, blocks, [&](const CompositeArgsFor<kDegree>& slice, const dim3& grid) {
    hipLaunchKernelGGL((composite_kernel<kTileSize, kBatch, kFull, kCount, kCheckpoint, kDegree>), grid, block, 0,
                       stream, slice);
  });
}

// Tile-front lists (16x16 tiles, 256-entry batches): records recomputed per SH degree.
template <int kDegree>
void launch_projected_degree(bool full, const FrontCompositeArgs& args, int64_t blocks, hipStream_t stream) {
  if (args.final_transmittance != nullptr) {
    // Checkpointed (pose-training) forward: final transmittance and last blended position.
    launch_variant<16, 256, true, false, true, kDegree>(args, blocks, stream);
  } else if (args.statistics != nullptr) {
    if (full) {
      launch_variant<16, 256, true, true, false, kDegree>(args, blocks, stream);
    } else {
      launch_variant<16, 256, false, true, false, kDegree>(args, blocks, stream);
    }
  } else if (full) {
    launch_variant<16, 256, true, false, false, kDegree>(args, blocks, stream);
  } else {
    launch_variant<16, 256, false, false, false, kDegree>(args, blocks, stream);
  }
}

void launch_projected(int degree, bool full, const FrontCompositeArgs& args, int64_t blocks, hipStream_t stream) {
  switch (degree) {
    case 1:
      launch_projected_degree<1>(full, args, blocks, stream);
      break;
    case 2:
      launch_projected_degree<2>(full, args, blocks, stream);
      break;
    case 3:
      launch_projected_degree<3>(full, args, blocks, stream);
      break;
    default:
      launch_projected_degree<0>(full, args, blocks, stream);
      break;
  }
}

template <int kTileSize, int kBatch>
void launch_full_or_rgb(bool full, const CompositeArgs& args, int64_t blocks, hipStream_t stream) {
  if (args.final_transmittance != nullptr) {
    launch_variant<kTileSize, kBatch, true, false, true>(args, blocks, stream);
  } else if (args.statistics != nullptr) {
    if (full) {
      launch_variant<kTileSize, kBatch, true, true>(args, blocks, stream);
    } else {
      launch_variant<kTileSize, kBatch, false, true>(args, blocks, stream);
    }
  } else if (full) {
    launch_variant<kTileSize, kBatch, true, false>(args, blocks, stream);
  } else {
    launch_variant<kTileSize, kBatch, false, false>(args, blocks, stream);
  }
}

template <int kTileSize>
void launch_batch(int batch, bool full, const CompositeArgs& args, int64_t blocks, hipStream_t stream) {
  switch (batch) {
    case 64:
      launch_full_or_rgb<kTileSize, 64>(full, args, blocks, stream);
      break;
    case 128:
      launch_full_or_rgb<kTileSize, 128>(full, args, blocks, stream);
      break;
    case 512:
      launch_full_or_rgb<kTileSize, 512>(full, args, blocks, stream);
      break;
    default:
      launch_full_or_rgb<kTileSize, 256>(full, args, blocks, stream);
      break;
  }
}

}  // namespace

int launch_tile_order(const CameraParams* table, const int32_t* tile_starts, const int32_t* tile_ends,
                      int active_count, int uniform_tiles, int64_t blocks, int32_t* order, hipStream_t stream,
                      uint32_t* long_tiles, const int32_t* reach, const int64_t* intersections) {
  if (blocks <= 0 || active_count <= 0) return 0;
  hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(kOrderThreads), 0, stream, table, tile_starts, tile_ends,
                     active_count, uniform_tiles, blocks, reach, intersections, order, long_tiles);
  const hipError_t error = hipGetLastError();
  if (error != hipSuccess) {
    set_error("tile order launch failed: %s", hipGetErrorString(error));
    return VGR_E_LAUNCH;
  }
  return 0;
}

int launch_composite(const vgr_scene& scene, const vgr_cameras& cameras, const vgr_outputs& outputs,
                     const vgr_options& options, const vgr_workspace& ws, const ScratchLayout& layout,
                     const char* scratch, bool sorted_in_out, hipStream_t stream) {
  if (cameras.active_count <= 0) return 0;
  CompositeArgs args;
  args.table = reinterpret_cast<const CameraParams*>(scratch + layout.camera_table);
  args.tile_starts = ws.tile_starts;
  args.tile_ends = ws.tile_ends;
  args.sorted_values = sorted_in_out ? ws.values_out : ws.values_in;
  args.records = ws.records;
  args.semantic_ids = scene.semantic_ids;
  args.rgb = outputs.rgb;
  args.depth = outputs.depth;
  args.alpha = outputs.alpha;
  args.semantic = outputs.semantic;
  args.statistics = options.statistics;
  args.visible_capacity = ws.visible_capacity;
  args.gaussian_count = scene.gaussian_count;
  args.active_count = cameras.active_count;
  args.output_srgb = options.output_srgb;
  args.semantic_min_alpha = options.semantic_min_alpha;
  args.final_transmittance = outputs.final_transmittance;
  args.last_blended = outputs.last_blended;
  args.slot_records = ws.slot_records;
  const bool front = options.ordering == VGR_ORDERING_TILE_FRONT;
  if (args.final_transmittance != nullptr && args.slot_records == nullptr && !front) {
    set_error("training forwards (transmittance checkpoints) need workspace.slot_records");
    return VGR_E_INVALID_ARGUMENT;
  }
  if (front && options.tile_size != 16) {
    set_error("tile-front ordering composites 16x16 tiles");
    return VGR_E_INVALID_ARGUMENT;
  }
  if (args.final_transmittance != nullptr &&
      (args.last_blended == nullptr || options.full_sensor_output == 0 || options.output_srgb != 0)) {
    set_error("transmittance checkpoints need last_blended, full sensor output and linear RGB");
    return VGR_E_INVALID_ARGUMENT;
  }
  int64_t blocks;
  if (cameras.widths == nullptr) {
    const int tiles_x = (options.width + options.tile_size - 1) / options.tile_size;
    const int tiles_y = (options.height + options.tile_size - 1) / options.tile_size;
    args.uniform_tiles = tiles_x * tiles_y;
    blocks = static_cast<int64_t>(cameras.active_count) * args.uniform_tiles;
  } else {
    args.uniform_tiles = 0;
    blocks = cameras.max_global_tiles;
  }
  if (blocks <= 0) return 0;
  if (blocks > 0x7fffffffLL) {
    set_error("composite grid of %lld tiles exceeds the launch limit", static_cast<long long>(blocks));
    return VGR_E_INVALID_ARGUMENT;
  }
  const bool full = options.full_sensor_output != 0;
  if (options.ray_evaluation != 0) {
    // options.tile_size is the bin size here (32 bins under 16x16 raster tiles).
    if (options.tile_size == 8) {
      launch_ray<8>(args, options, ws.ray_records, cameras.active_count, full, stream);
    } else {
      launch_ray<16>(args, options, ws.ray_records, cameras.active_count, full, stream);
    }
    const hipError_t error = hipGetLastError();
    if (error != hipSuccess) {
      set_error("composite launch failed: %s", hipGetErrorString(error));
      return VGR_E_LAUNCH;
    }
    return 0;
  }
  if (options.tile_size < 8) {
    const int64_t threads = blocks * options.tile_size * options.tile_size;
    const dim3 grid(static_cast<unsigned>((threads + 255) / 256)), block(256);
    const bool count = options.statistics != nullptr;
    if (full && count) {
      hipLaunchKernelGGL((composite_pixels_kernel<true, true>), grid, block, 0, stream, args, options.tile_size, threads);
    } else if (full) {
      hipLaunchKernelGGL((composite_pixels_kernel<true, false>), grid, block, 0, stream, args, options.tile_size,
                         threads);
    } else if (count) {
      hipLaunchKernelGGL((composite_pixels_kernel<false, true>), grid, block, 0, stream, args, options.tile_size,
                         threads);
    } else {
      hipLaunchKernelGGL((composite_pixels_kernel<false, false>), grid, block, 0, stream, args, options.tile_size,
                         threads);
    }
    const hipError_t error = hipGetLastError();
    if (error != hipSuccess) {
      set_error("composite launch failed: %s", hipGetErrorString(error));
      return VGR_E_LAUNCH;
    }
    return 0;
  }
  args.total_items = blocks;
  args.first_item = 0;
  args.work_counter = reinterpret_cast<uint32_t*>(const_cast<char*>(scratch) + layout.work_counter);
  // Longest tiles first pays when the grid is a few waves deep per SIMD; on deep
  // grids the tail is short already.
  args.tile_order = nullptr;
  if (blocks <= kOrderedCompositeBlocks) {
    int32_t* order = reinterpret_cast<int32_t*>(const_cast<char*>(scratch) + layout.tile_order);
    int32_t* reach = nullptr;
    if (!front && options.tile_size == 16 && options.statistics == nullptr && blocks > kReachTiles &&
        blocks <= kMixedCompositeTiles && options.fixed_capacity_sort == 0 &&
        ws.intersection_capacity >= blocks * kReachLists && layout.sort_flag_words >= blocks) {
      // The sort's flags are read no more.
      reach = reinterpret_cast<int32_t*>(const_cast<char*>(scratch) + layout.sort_flags);
      hipLaunchKernelGGL(args.final_transmittance != nullptr ? tile_reach_kernel<true> : tile_reach_kernel<false>,
                         dim3(static_cast<unsigned>(blocks)), dim3(kReachWaves * kWave), 0, stream, args,
                         ws.counters + VGR_COUNTER_INTERSECTIONS, reach);
    }
    const int order_status = launch_tile_order(args.table, args.tile_starts, args.tile_ends, args.active_count,
                                               args.uniform_tiles, blocks, order, stream, args.work_counter + 1,
                                               reach, ws.counters + VGR_COUNTER_INTERSECTIONS);
    if (order_status != 0) return order_status;
    args.tile_order = order;
    args.long_tiles = args.work_counter + 1;
  }
  if (front) {
    FrontCompositeArgs front_args;
    static_cast<CompositeArgs&>(front_args) = args;
    make_projection_args(scene, cameras, options, layout, scratch, front_args.projection);
    uint32_t* open_state = reinterpret_cast<uint32_t*>(const_cast<char*>(scratch) + layout.front_open_state);
    int32_t* open_tiles = reinterpret_cast<int32_t*>(const_cast<char*>(scratch) + layout.front_open_tiles);
    front_args.front_lengths = reinterpret_cast<const int32_t*>(scratch + layout.front_lengths);
    front_args.open_tiles = open_tiles;
    front_args.open_count = open_state + 0;
    front_args.item_count = nullptr;
    launch_fill_u32(open_state, 4, 0u, stream);
    launch_projected(scene.sh_degree, full, front_args, blocks, stream);
    // Tiles left open at the end of a truncated list: full sort, then composite
    // them again from their complete lists (fixed grids that exit at once when
    // no tile is open).
    const int status = launch_front_fallback_sort(scene, ws, layout, const_cast<char*>(scratch), kOpenWorkgroups,
                                                  stream);
    if (status != 0) return status;
    FrontCompositeArgs again = front_args;
    again.open_tiles = nullptr;
    again.front_lengths = nullptr;
    again.tile_order = open_tiles;
    again.item_count = open_state + 0;
    again.work_counter = open_state + 2;
    launch_projected(scene.sh_degree, full, again, blocks, stream);
    if (options.statistics != nullptr) launch_copy_u32_to_i64(open_state + 0, options.statistics + 3, stream);
  } else if (options.tile_size == 8) {
    launch_batch<8>(options.raster_batch, full, args, blocks, stream);
  } else {
    launch_batch<16>(options.raster_batch, full, args, blocks, stream);
  }
  const hipError_t error = hipGetLastError();
  if (error != hipSuccess) {
    set_error("composite launch failed: %s", hipGetErrorString(error));
    return VGR_E_LAUNCH;
  }
  return 0;
}

}  // namespace vgr
