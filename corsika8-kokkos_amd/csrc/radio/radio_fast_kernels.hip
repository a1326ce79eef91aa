// The fast CoREAS / ZHS projection: int64 window tiles of a group of observers in
// LDS, FP64 arithmetic of radio_pair_fast.hpp.
//
// A workgroup holds the tiles of `group` observers and takes each track of its
// chunk through all of them. What a track costs on its own (nine loads, the
// velocity, and per endpoint or midpoint two gathers from the propagation table,
// each lane from an L2 line of its own) is paid once per group: with one observer
// per workgroup the gathers alone are 4 L2 requests per track-antenna pair, and
// the kernel waits for them.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>

#include "radio_block.hpp"
#include "radio_device.hpp"
#include "radio_launch.hpp"
#include "radio_pair_fast.hpp"
#include "../runtime.hpp"

namespace c8mi::radio {
namespace {

// An observer through the scalar cache: its address is the same in every lane,
// and nothing writes observers while a projection runs.
using ObserverConst = __attribute__((address_space(4))) ObserverDev const;

template <class Observer>
__device__ __forceinline__ fast::View make_view(Observer const& d, std::uint32_t tile_begin, std::uint32_t tile_bins) {
  fast::View v;
  v.position = {d.position[0], d.position[1], d.position[2]};
  v.start = d.start_time;
  v.end = d.end_time;
  v.rate = d.sample_rate;
  v.grid = d.grid;
  v.two_pi_over_wavelength = d.two_pi_over_wavelength;
  std::uint64_t const bins = d.number_of_bins;
  std::uint64_t const end = static_cast<std::uint64_t>(tile_begin) + tile_bins;
  v.tile_begin = static_cast<double>(tile_begin);
  v.tile_end = static_cast<double>(static_cast<std::uint32_t>(bins < end ? bins : end));
  v.destination_height = d.destination_height;
  v.destination_index = d.destination_index;
  v.n_destination = d.n_destination;
  v.integrated_destination = d.integrated_destination;
  v.scale = d.fixed_scale;
  return v;
}

// Pairs of a wave whose CoREAS update takes the Cherenkov form. In air one pair
// in ten does (2^20 tracks x 160 antennas), so nearly every wave would run both
// forms; a wave lists them (LDS, entries of its own) and runs the second form on
// 64 of them at a time. (ZHS segments over more than two bins are too few for a
// list: loading their tracks again cost more than the branch.)
constexpr std::uint32_t kListEntries = 128;  // up to 63 left over + 64 new
constexpr std::uint32_t kForwardBit = 1u << 31;
constexpr std::uint32_t kMemberShift = 27;  // track in the chunk below, observer of the group above
static_assert(kMaxChunkTracks <= (std::uint64_t{1} << kMemberShift), "list entries hold a chunk's tracks");
static_assert(kMaxGroup <= 16, "list entries hold four bits of observer");
static_assert(kPairListBytesPerThread * 64 == kListEntries * sizeof(std::uint32_t), "LDS of the lists");
static_assert(kBudgetBytesPerObserver == kRanges * sizeof(Budget), "LDS of the budgets");

// Appends the lanes' entries where `listed`; true when a full wave of them is
// due (take_pair).
__device__ __forceinline__ bool list_pairs(std::uint32_t* entries, std::uint32_t& pending, bool listed,
                                           std::uint32_t entry) {
  unsigned long long const mask = __ballot(listed);
  if (mask == 0) return false;
  std::uint32_t const below = __builtin_amdgcn_mbcnt_hi(
      static_cast<std::uint32_t>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<std::uint32_t>(mask), 0u));
  if (listed) entries[pending + below] = entry;
  pending += static_cast<std::uint32_t>(__popcll(mask));
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wave's own entries, in order
  return pending >= 64;
}
__device__ __forceinline__ std::uint32_t take_pair(std::uint32_t const* entries, std::uint32_t& pending) {
  pending -= 64;
  std::uint32_t const entry = entries[pending + threadIdx.x % 64];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  return entry;
}

template <bool Coreas, bool Zhs, bool Homogeneous, int Block>
__device__ __forceinline__ void project_chunk(ProjectionLaunch const& L, ObserverDev const* coreas_observers,
                                              ObserverDev const* zhs_observers, std::uint32_t members,
                                              std::uint32_t tile_begin, std::uint64_t chunk_begin,
                                              std::uint64_t chunk_end, long long* tiles, bool count_valid,
                                              std::uint32_t* entries, std::uint32_t first, Budget* budgets,
                                              fast::Tally& tally) {
  PropagationDev const& prop = L.propagation;
  std::uint32_t const W = L.tile_bins;
  std::uint32_t const words = (Coreas ? 3 * W : 0) + (Zhs ? 3 * (W + 1) : 0);  // tile words of a member
  double const* const chunk = L.tracks + chunk_begin;
  std::uint32_t const count = static_cast<std::uint32_t>(chunk_end - chunk_begin);
  std::uint32_t pending = 0;  // this wave's listed pairs
  auto run_near = [&](std::uint32_t entry) {
    std::uint32_t const member = (entry & ~kForwardBit) >> kMemberShift;
    fast::Track t;
    (void)fast::load_track(chunk, L.stride, entry & ((1u << kMemberShift) - 1u), t);
    fast::coreas_near<Homogeneous>(t, prop, make_view(coreas_observers[member], tile_begin, W), tiles + member * words,
                                   W, {first + member, nullptr}, tally, (entry & kForwardBit) != 0);
  };
  for (std::uint32_t i = 0; i < count; i += Block) {
    fast::Track t;
    bool active = false;
    fast::Source start, end, middle;
    std::uint32_t start_kind, end_kind, middle_kind;
    double length2;
    active = i + threadIdx.x < count && fast::load_track(chunk + i, L.stride, threadIdx.x, t);
    if (active) {
      if constexpr (Coreas) {
        start = fast::make_source<Homogeneous>(prop, t.start, start_kind);
        end = fast::make_source<Homogeneous>(prop, t.end, end_kind);
      }
      if constexpr (Zhs) {
        middle = fast::make_source<Homogeneous>(prop, fast::midpoint(t), middle_kind);
        fast::V3 const d{t.end.x - t.start.x, t.end.y - t.start.y, t.end.z - t.start.z};
        length2 = fast::dot(d, d);
      }
      if (count_valid) ++tally.valid;
    }
    for (std::uint32_t k = 0; k < members; ++k) {
      long long* const tile = tiles + k * words;
      if constexpr (Zhs) {
        if (active) {
          fast::View const v = make_view(*(ObserverConst*)(zhs_observers + k), tile_begin, W);
          fast::zhs_update<Homogeneous>(t, middle, middle_kind, length2, prop, L.zhs_refinement, v,
                                        tile + (Coreas ? 3 * W : 0), W + 1, {first + k, budgets + k * kRanges}, tally, tile_begin == 0);
        }
      }
      if constexpr (Coreas) {
        bool near = false, forward = false;
        if (active) {
          fast::View const v = make_view(*(ObserverConst*)(coreas_observers + k), tile_begin, W);
          near = fast::coreas_far<Homogeneous>(t, start, start_kind, end, end_kind, prop, v, tile, W,
                                                {first + k, nullptr}, tally, forward);
        }
        std::uint32_t const entry =
            (i + threadIdx.x) | (k << kMemberShift) | (forward ? kForwardBit : 0u);
        if (list_pairs(entries, pending, near, entry)) run_near(take_pair(entries, pending));
      }
    }
  }
  if constexpr (Coreas) {
    if (threadIdx.x % 64 < pending) run_near(entries[threadIdx.x % 64]);
  }
}

// Four waves per SIMD (128 VGPRs); the 256-thread forms three (the pooled one's two
// tiles of an observer leave room for three workgroups a CU up to 1090 bins, and it
// holds the endpoints and the midpoint of a track: 168 VGPRs). Three such waves fill
// a SIMD's registers, so the front kernels on other streams wait: the benchmark's
// serving stream spends 1.1 s in scan and 0.53 s in scatter (0.37 and 0.34 beside
// a 128-register kernel) while it gained 1.2x as a whole.
template <bool Coreas, bool Zhs, bool Homogeneous, int Block>
__global__ void __launch_bounds__(Block, Block == 256 ? 3 : 4) radio_fast_kernel(ProjectionLaunch L) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ long long scan_scratch[Zhs ? Block / 64 : 1];
  __shared__ BlockTallies block;
  constexpr std::uint32_t kBudgets = Zhs ? most_observers(Block) * kRanges : 1;
  __shared__ Budget budgets[kBudgets];
  __shared__ std::uint32_t lists[Coreas ? Block / 64 : 1][Coreas ? kListEntries : 1];

  // the workgroup's chunk, observers [first, first + members) and window tile
  std::uint32_t first, members, within;
  std::uint64_t chunk_begin, chunk_end;
  CountersDev* counters = L.counters;
  bool count_valid;
  if (L.segments == nullptr) {
    std::uint32_t const groups = (L.observer_count + L.group - 1) / L.group;
    if (!decode_chunk(L, groups * L.bin_tiles, within, chunk_begin, chunk_end)) return;
    first = within / L.bin_tiles * L.group;
    members = L.observer_count - first < L.group ? L.observer_count - first : L.group;
    count_valid = L.count_valid && within == 0;
  } else {
    SegmentDev seg;
    std::uint64_t local;
    if (!decode_segment(L, seg, local)) return;
    std::uint32_t const observers = L.slot_observer_counts[seg.slot];
    std::uint32_t const per_chunk = (observers + L.group - 1) / L.group * L.bin_tiles;
    std::uint64_t const chunk = local / per_chunk;
    within = static_cast<std::uint32_t>(local % per_chunk);
    std::uint32_t const at = within / L.bin_tiles * L.group;
    members = observers - at < L.group ? observers - at : L.group;
    first = seg.slot * L.slot_observers + at;
    chunk_begin = seg.begin + chunk * L.chunk_size;
    chunk_end = chunk_begin + L.chunk_size < seg.end ? chunk_begin + L.chunk_size : seg.end;
    counters = L.counters + seg.slot;
    count_valid = L.count_valid && within == 0;
  }
  std::uint32_t const W = L.tile_bins;
  std::uint32_t const tile_begin = within % L.bin_tiles * W;  // below 2^31 bins (checked on the host)
  std::uint32_t const words = (Coreas ? 3 * W : 0) + (Zhs ? 3 * (W + 1) : 0);
  long long* const tiles = reinterpret_cast<long long*>(lds_raw);
  for (std::uint32_t i = threadIdx.x; i < members * words; i += Block) tiles[i] = 0;
  if (threadIdx.x < kBudgets) budgets[threadIdx.x] = 0.;
  clear_tallies(block);
  __syncthreads();

  ObserverDev const* const coreas_observers = L.coreas_observers + first;
  ObserverDev const* const zhs_observers = L.zhs_observers + first;
  std::uint32_t* const entries = lists[Coreas ? threadIdx.x / 64 : 0];
  fast::Tally tally;
  project_chunk<Coreas, Zhs, Homogeneous, Block>(L, coreas_observers, zhs_observers, members, tile_begin, chunk_begin,
                                                 chunk_end, tiles, count_valid, entries, first, budgets, tally);
  unsigned long long const counts[5] = {tally.coreas, tally.zhs, tally.subtracks + tally.single_subtracks, tally.valid,
                                        tally.overflow};
  add_tallies<Coreas, Zhs>(block, counts);
  __syncthreads();

  unsigned long long overflows = 0;
  for (std::uint32_t k = 0; k < members; ++k) {
    ObserverDev const& o = Coreas ? coreas_observers[k] : zhs_observers[k];
    std::uint64_t const nbins = o.number_of_bins;
    std::uint32_t const bins =
        tile_begin < nbins ? static_cast<std::uint32_t>(nbins - tile_begin < W ? nbins - tile_begin : W) : 0u;
    std::uint64_t const at = o.waveform_offset + tile_begin;
    long long* const coreas_tile = tiles + k * words;
    long long* const zhs_tile = coreas_tile + (Coreas ? 3 * W : 0);
    if constexpr (Zhs) {
      for (int c = 0; c < 3; ++c) block_inclusive_scan(zhs_tile + c * (W + 1), W, scan_scratch);
    }
    if constexpr (Coreas)
      overflows += flush_tile<true>(coreas_tile, W, bins, L.coreas_waves, L.coreas_total_bins, at);
    if constexpr (Zhs) overflows += flush_tile<true>(zhs_tile, W + 1, bins, L.zhs_waves, L.zhs_total_bins, at);
  }
  if (overflows) atomicAdd(&block.counts[4], overflows);
  __syncthreads();
  publish_tallies(block, counters);
}

template <bool Coreas, bool Zhs, bool Homogeneous, int Block>
void launch_typed(ProjectionLaunch const& launch, std::uint32_t grid, hipStream_t stream) {
  auto kernel = radio_fast_kernel<Coreas, Zhs, Homogeneous, Block>;
  static bool attribute_set = false;
  if (!attribute_set) {
    C8MI_HIP(hipFuncSetAttribute(reinterpret_cast<void const*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(fast_dynamic_lds_limit(Coreas, Zhs, Block))));
    attribute_set = true;
  }
  if (launch.group > most_observers(Block)) throw std::logic_error("radio: more observers than the workgroup takes");
  std::size_t const lds = launch.group * projection_lds_bytes(Coreas, Zhs, launch.tile_bins);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Block), lds, stream, launch);
  C8MI_HIP(hipGetLastError());
}

template <bool Coreas, bool Zhs, bool Homogeneous>
void launch_block(ProjectionLaunch const& launch, std::uint32_t block, std::uint32_t grid, hipStream_t stream) {
  switch (block) {
    case 256: launch_typed<Coreas, Zhs, Homogeneous, 256>(launch, grid, stream); break;
    case 512: launch_typed<Coreas, Zhs, Homogeneous, 512>(launch, grid, stream); break;
    case 1024: launch_typed<Coreas, Zhs, Homogeneous, 1024>(launch, grid, stream); break;
    default: throw std::invalid_argument("radio workgroup size must be 256, 512 or 1024");
  }
}

template <bool Coreas, bool Zhs>
void launch_medium(ProjectionLaunch const& launch, std::uint32_t block, std::uint32_t grid, hipStream_t stream) {
  if (launch.propagation.homogeneous_index > 0.) launch_block<Coreas, Zhs, true>(launch, block, grid, stream);
  else launch_block<Coreas, Zhs, false>(launch, block, grid, stream);
}

}  // namespace

void launch_fast(ProjectionLaunch const& launch, bool coreas, bool zhs, std::uint32_t block, std::uint32_t grid,
                 hipStream_t stream) {
  if (coreas && zhs) launch_medium<true, true>(launch, block, grid, stream);
  else if (coreas) launch_medium<true, false>(launch, block, grid, stream);
  else if (zhs) launch_medium<false, true>(launch, block, grid, stream);
}

}  // namespace c8mi::radio
