// Validation and device forms of radio configurations, shared by the radio
// accumulator and the per-slot radio of the EM pool.
#include "radio_setup.hpp"

#include "radio_launch.hpp"

#include <algorithm>
#include <cmath>
#include <limits>
#include <stdexcept>

namespace c8mi::radio {

// The observer checks of RadioAccumulator::validate: finite fields, positive
// rate, bins in [1, 2^31), positions inside the propagation table.
void validate_observers(c8mi_radio_observer const* observers, std::uint64_t count,
                        c8mi_radio_propagation const& p) {
  bool const homogeneous = p.homogeneous_refractive_index > 0.;
  if (count != 0 && observers == nullptr)
    throw std::invalid_argument("null radio observer list");
  for (std::uint64_t i = 0; i < count; ++i) {
    auto const& o = observers[i];
    if (!std::isfinite(o.start_time_s) || !std::isfinite(o.duration_s) ||
        !(o.duration_s >= 0.) || !std::isfinite(o.sample_rate_hz) ||
        !(o.sample_rate_hz > 0.) || o.number_of_bins == 0)
      throw std::invalid_argument("invalid radio observer");
    if (o.number_of_bins >= (std::uint64_t{1} << 31))
      throw std::length_error("radio observer with 2^31 or more bins");
    double const height = (o.position_m[2] - p.minimum_height_m) * p.inverse_step_per_m;
    if (!homogeneous && (!std::isfinite(height) || height < 0. ||
                         height + 0.5 >= static_cast<double>(p.table_size)))
      throw std::invalid_argument("radio observer outside propagation table");
    for (double coordinate : o.position_m)
      if (!std::isfinite(coordinate))
        throw std::invalid_argument("radio observer position is not finite");
  }
}

// RadioAccumulator::validate (corsika/detail/kokkos/radio/RadioAccumulator.inl:934-975).
void validate_radio_config(c8mi_radio_config const& config) {
  auto const& p = config.propagation;
  if (!config.coreas_enabled && !config.zhs_enabled)
    throw std::invalid_argument("enabled radio has no algorithm");
  if (!std::isfinite(config.fixed_point_field_limit_v_per_m) ||
      !(config.fixed_point_field_limit_v_per_m > 0.))
    throw std::invalid_argument("invalid radio fixed-point limit");
  if (config.zhs_subtrack_refinement < 1 || config.zhs_subtrack_refinement > 64)
    throw std::invalid_argument("ZHS subtrack refinement must be in [1,64]");
  if (!std::isfinite(p.homogeneous_refractive_index) || p.homogeneous_refractive_index < 0.)
    throw std::invalid_argument("invalid homogeneous radio refractive index");
  bool const homogeneous = p.homogeneous_refractive_index > 0.;
  if (!homogeneous &&
      (p.table_size < 11 || p.refractivity == nullptr || p.integrated_refractivity == nullptr ||
       !std::isfinite(p.minimum_height_m) || !std::isfinite(p.maximum_height_m) ||
       !(p.maximum_height_m > p.minimum_height_m) || !std::isfinite(p.step_m) ||
       !(p.step_m > 0.) || !std::isfinite(p.inverse_step_per_m) ||
       !(p.inverse_step_per_m > 0.)))
    throw std::invalid_argument("invalid flat-atmosphere radio snapshot");
  if (!homogeneous && p.table_size >= (std::uint64_t{1} << 32))
    throw std::length_error("radio propagation table above 2^32 entries");
  validate_observers(config.coreas_observers, config.coreas_enabled ? config.coreas_observer_count : 0, p);
  validate_observers(config.zhs_observers, config.zhs_enabled ? config.zhs_observer_count : 0, p);
}

// RadioAccumulator::makeObservers (RadioAccumulator.inl:591-617).
std::vector<ObserverDev> make_observers(c8mi_radio_observer const* input, std::uint64_t count,
                                        double limit, bool zhs_potential, c8mi_radio_propagation const& p,
                                        std::uint64_t& total_bins, std::uint64_t& max_bins) {
  std::vector<ObserverDev> result;
  result.reserve(count);
  total_bins = 0;
  max_bins = 0;
  for (std::uint64_t i = 0; i < count; ++i) {
    auto const& o = input[i];
    ObserverDev d{};
    for (int a = 0; a < 3; ++a) d.position[a] = o.position_m[a];
    d.start_time = o.start_time_s;
    d.duration = o.duration_s;
    d.sample_rate = o.sample_rate_hz;
    double const potential_factor = zhs_potential ? o.sample_rate_hz : 1.;
    d.fixed_scale = kHeadroom * potential_factor / limit;
    d.number_of_bins = o.number_of_bins;
    d.waveform_offset = total_bins;
    d.end_time = d.start_time + d.duration;
    d.grid = 1. / d.sample_rate;
    d.two_pi_over_wavelength = 2. * 3.141592653589793238462643383279502884 / (299792458. / d.sample_rate);
    d.n_destination = 1.;
    if (!(p.homogeneous_refractive_index > 0.)) {  // positions inside the table were checked
      d.destination_height = (d.position[2] - p.minimum_height_m) * p.inverse_step_per_m;
      auto const cell = static_cast<std::uint64_t>(d.destination_height + 0.5);
      d.destination_index = static_cast<double>(cell);
      d.n_destination = p.refractivity[cell] + 1.;
      d.integrated_destination = p.integrated_refractivity[cell];
    }
    if (o.number_of_bins > std::numeric_limits<std::uint64_t>::max() - total_bins)
      throw std::overflow_error("radio waveform bin overflow");
    total_bins += o.number_of_bins;
    max_bins = std::max<std::uint64_t>(max_bins, o.number_of_bins);
    result.push_back(d);
  }
  return result;
}

// observersCanShareTrackKinematics (RadioAccumulator.inl:619-632).
bool can_fuse(std::vector<ObserverDev> const& a, std::vector<ObserverDev> const& b) {
  if (a.size() != b.size() || a.empty()) return false;
  for (std::size_t i = 0; i < a.size(); ++i) {
    if (a[i].start_time != b[i].start_time || a[i].duration != b[i].duration ||
        a[i].sample_rate != b[i].sample_rate || a[i].number_of_bins != b[i].number_of_bins ||
        a[i].position[0] != b[i].position[0] || a[i].position[1] != b[i].position[1] ||
        a[i].position[2] != b[i].position[2])
      return false;
  }
  return true;
}


PropagationDev propagation_view(c8mi_radio_propagation const& p, double const* refractivity,
                                double const* integrated) {
  PropagationDev d{};
  d.homogeneous_index = p.homogeneous_refractive_index;
  d.minimum_height = p.minimum_height_m;
  d.maximum_height = p.maximum_height_m;
  d.step = p.step_m;
  d.inverse_step = p.inverse_step_per_m;
  d.slope_n_lower = p.slope_refractivity_lower;
  d.slope_i_lower = p.slope_integrated_refractivity_lower;
  d.slope_n_upper = p.slope_refractivity_upper;
  d.slope_i_upper = p.slope_integrated_refractivity_upper;
  d.refractivity = refractivity;
  d.integrated = integrated;
  d.table_size = p.homogeneous_refractive_index > 0. ? 0 : p.table_size;
  return d;
}

namespace {

// The launch shape of a fast projection: window tiles of an observer, observers
// of a workgroup (its tiles share the CU's LDS: one workgroup of 1024 threads, or
// two of 512 with one tile each) and track chunks (a multiple of eight: chunk c
// runs on XCD c % 8). A workgroup's time is its tracks times the cost of an
// update, plus clearing and flushing its tiles; the launch takes as many rounds
// as 256 CUs need for its workgroups, so a shape that just fills its rounds wins
// over one that leaves the last round empty.
//
// Costs, measured with 2^20 tracks on 160 antennas and 1024 and 2048 bins at 0.2
// ns: nanoseconds of a CU per track and observer with one observer a workgroup,
// and the share of it left with g (the track's loads, table gathers and velocity
// are paid once per workgroup). The estimate ordered the measured times of 26
// shapes of 40000 to 2^20 tracks, 40 to 160 antennas and 333 to 4096 bins except
// where two lay within 5%. The costs are those of air with whole ZHS tracks; in a
// constant index there are no gathers to share, and the parts of refined tracks share
// nothing. There the estimate's shapes were measured against one observer a workgroup
// (512 and 1024 threads) only: 24 launches of 1000 to 5e5 tracks on 7 to 160 antennas,
// 300 to 4096 bins, refinement 1 and 3, were 1.0 to 3.2 times faster, but for lists of
// 1000 tracks on 24 antennas, where ZHS takes 16 us instead of 14 (as in air).
constexpr double kCoreasNs = 5.0, kZhsNs = 2.75;
constexpr double kCoreasShare[kMaxGroup] = {1., .59, .51, .475, .46, .445, .435, .43};
constexpr double kZhsShare[kMaxGroup] = {1., .84, .755, .71, .685, .66, .65, .64};
constexpr double kRoundNs = 6000., kFlushNsPerBin = 4.;
constexpr std::uint64_t kCus = 256;
constexpr std::uint64_t kMaxRounds = 16;  // chunk counts tried: up to so many workgroups a CU

void shape_fast(ProjectionLaunch& L, bool zhs, std::uint64_t observers, std::uint64_t bins,
                std::uint64_t count) {
  bool const coreas = !zhs;
  auto const tile_bytes = [&](std::uint64_t tile) { return projection_lds_bytes(coreas, zhs, static_cast<std::uint32_t>(tile)); };
  constexpr std::size_t per_bin = 3;
  std::size_t const most_lds = fast_dynamic_lds_limit(coreas, zhs, 1024);
  std::uint64_t const capacity = (most_lds / sizeof(long long) - (zhs ? 3u : 0u)) / per_bin;
  std::uint64_t const preferred = default_tile_capacity(per_bin, zhs);
  std::uint64_t const last_tiles = (bins + preferred - 1) / preferred;
  // every tile of an observer computes the track's update again, so the fewest
  // that fit are tried too (windows of many tiles take the usual size)
  std::uint64_t const first_tiles = last_tiles <= 8 ? (bins + capacity - 1) / capacity : last_tiles;
  double best = std::numeric_limits<double>::infinity();
  for (std::uint64_t tiles = first_tiles; tiles <= last_tiles; ++tiles) {
    std::uint64_t const tile = (bins + tiles - 1) / tiles;
    std::uint64_t const used = (bins + tile - 1) / tile;  // tiles that hold bins
    for (std::uint32_t group = 1; group <= kMaxGroup && group <= observers; ++group) {
      if (group * tile_bytes(tile) > most_lds) break;
      std::uint64_t const per_chunk = (observers + group - 1) / group * used;
      double const update = zhs ? kZhsNs * kZhsShare[group - 1] : kCoreasNs * kCoreasShare[group - 1];
      double const round = kRoundNs + kFlushNsPerBin * static_cast<double>(group * tile);
      for (std::uint64_t chunks = kXcdCount;; chunks += kXcdCount) {
        std::uint64_t const chunk = (count + chunks - 1) / chunks;
        std::uint64_t const rounds = (per_chunk * chunks + kCus - 1) / kCus;
        if (chunk <= kMaxChunkTracks) {
          double const time = static_cast<double>(rounds) * (static_cast<double>(chunk * group) * update + round);
          if (time < best) {
            best = time;
            L.tile_bins = static_cast<std::uint32_t>(tile);
            L.bin_tiles = static_cast<std::uint32_t>(used);
            L.group = group;
            // two workgroups of one tile each share a CU; a large tile or a group takes it alone
            L.block_threads = group == 1 && 2 * (tile_bytes(tile) + fast_static_lds(coreas, zhs, 512)) <= kCuLdsBytes ? 512u : 1024u;
            L.chunk_size = chunk;
          }
        }
        if (chunk <= kMaxChunkTracks && (chunk <= 1024 || rounds >= kMaxRounds)) break;
      }
    }
  }
}

}  // namespace

LaunchTuning make_tuning(std::uint64_t chunk_tracks, std::uint32_t tile_bins, std::uint32_t target_workgroups,
                         std::uint32_t block_threads) {
  if (block_threads != 0 && block_threads != 256 && block_threads != 512 && block_threads != 1024)
    throw std::invalid_argument("radio workgroup size must be 256, 512 or 1024");
  if (chunk_tracks % (block_threads ? block_threads : kProjectionBlock) != 0)
    throw std::invalid_argument("radio chunk size must be a multiple of the workgroup size");
  return {chunk_tracks, tile_bins, target_workgroups, block_threads};
}

void shape_projection(ProjectionLaunch& L, bool coreas, bool zhs, bool fast, std::uint32_t observers,
                      std::uint64_t max_bins, std::uint64_t count, LaunchTuning const& tuning) {
  // Window tile: the whole waveform when it fits the preferred LDS size, else
  // equal tiles of at most that size (a tuning limit may ask for others up to
  // the LDS budget).
  // The fast form of both algorithms needs more than the 128 registers that 512
  // threads leave: 256 (three waves a SIMD). Measured with 3e4 tracks on 160 antennas
  // and 1024 bins, 262144 on 64 and 400, 5e5 on 100 and 2048: 0.20, 0.56 and 3.1 ms,
  // in the estimated shape of 512 or 1024 threads 0.24, 0.43 and 3.5.
  bool const fused = coreas && zhs;
  L.block_threads = tuning.block_threads ? tuning.block_threads : fast && fused ? 256u : kDefaultThreads;
  L.group = 1;
  if (fast && !fused && tuning.automatic() && observers != 0 && max_bins != 0 && count != 0) {
    shape_fast(L, zhs, observers, max_bins, count);
  } else {
    std::size_t const words = (fast ? std::min(kMaxDynamicLdsBytes, fast_dynamic_lds_limit(coreas, zhs, L.block_threads))
                                    : kMaxDynamicLdsBytes) / sizeof(long long);
    std::size_t const per_bin = (coreas ? 3u : 0u) + (zhs ? 3u : 0u);
    std::uint64_t capacity = default_tile_capacity(per_bin, zhs);
    if (tuning.tile_bins_limit != 0)
      capacity = std::min<std::uint64_t>((words - 3) / per_bin, tuning.tile_bins_limit);
    std::uint64_t const want = std::max<std::uint64_t>(max_bins, 1);
    std::uint64_t tile = std::min<std::uint64_t>(want, capacity);
    if (tuning.tile_bins_limit == 0) {  // equal tiles: a 4096-bin window as two 2048-bin tiles
      std::uint64_t const tiles = (want + capacity - 1) / capacity;
      tile = (want + tiles - 1) / tiles;
    }
    L.tile_bins = static_cast<std::uint32_t>(tile);
    L.bin_tiles = static_cast<std::uint32_t>((max_bins + tile - 1) / tile);
    if (L.bin_tiles == 0) L.bin_tiles = 1;
    std::uint64_t chunk = tuning.chunk_tracks;
    if (chunk == 0) {
      std::uint64_t const per_chunk = std::max<std::uint64_t>(1, std::uint64_t(observers) * L.bin_tiles);
      std::uint64_t const target = tuning.target_workgroups ? tuning.target_workgroups : kDefaultWorkgroups;
      std::uint64_t const chunks_wanted = std::max<std::uint64_t>(1, target / per_chunk);
      // a workgroup clears and flushes a whole window tile, so chunks of tens
      // of thousands of tracks pay (2^20 tracks on 160 antennas: 32768-track
      // chunks 1.2x faster than 16384, as fast as 65536)
      std::uint64_t chunks = std::min<std::uint64_t>(chunks_wanted, count / kMinimumDefaultChunk);
      // chunk c runs on XCD c % 8: a multiple of eight chunks keeps the XCDs
      // evenly loaded (50 chunks measured 12% slower than 48 or 64); a small
      // batch (a lepton front's tracks) still gets eight chunks, so every XCD
      // works on it (the EM + radio shower measured 10% faster than with
      // chunks of at least 8192 tracks)
      chunks = chunks >= kXcdCount ? chunks / kXcdCount * kXcdCount : kXcdCount;
      chunk = (count + chunks - 1) / chunks;
      std::uint64_t const block = L.block_threads;
      chunk = std::max<std::uint64_t>(block, (chunk + block - 1) / block * block);
    }
    chunk = std::min(chunk, kMaxChunkTracks);
    L.chunk_size = chunk;
  }
  std::uint64_t const chunks = (count + L.chunk_size - 1) / L.chunk_size;
  if (chunks > std::numeric_limits<std::uint32_t>::max())
    throw std::length_error("radio track batch too large for one launch");
  L.chunks = static_cast<std::uint32_t>(chunks);
  std::uint64_t const groups = (std::uint64_t(observers) + L.group - 1) / L.group;
  std::uint64_t const grid = (chunks + 7) / 8 * 8 * groups * L.bin_tiles;
  if (grid > std::numeric_limits<std::uint32_t>::max())
    throw std::length_error("radio projection grid too large");
}

}  // namespace c8mi::radio
