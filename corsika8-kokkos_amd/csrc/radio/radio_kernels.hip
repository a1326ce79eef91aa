// CoREAS / ZHS endpoint projection for gfx950.
//
// Physics: corsika/detail/kokkos/radio/algorithms/RadioProjection.inl (propagate
// :170-238, accumulate_co_reas :338-409, accumulate_zhs_segment :411-480,
// accumulate_zhs :482-529, add_sample :262-301). Every floating-point expression
// keeps the reference's operation order and the file is built without
// contraction, so the int64 fixed-point waveforms equal the FP64 restatement's.
//
// MI355X design (differs from the reference's track-tile x observer-tile teams,
// RadioAccumulator.inl:15-85):
//  * one workgroup = one observer x one chunk of tracks x one window tile; the
//    observer's whole waveform tile lives in LDS as int64 fixed point, so the
//    per-sample atomics are ds_add_u64, and HBM sees one flush per workgroup;
//  * ZHS middle bins all receive the same increment, so they are added to an
//    LDS difference array (two atomics per component instead of one per bin)
//    and recovered by a block prefix scan before the flush; integer addition
//    makes this bit-identical to the per-bin loop;
//  * threads stride over tracks (coalesced 9 x FP64 structure-of-arrays loads);
//  * blockIdx -> (chunk, observer) is XCD-aware: the eight XCDs take disjoint
//    chunk sets and walk all observers of a chunk back to back, so a chunk is
//    fetched from HBM once per XCD and re-read from that XCD's L2.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <stdexcept>
#include <type_traits>

#include "radio_block.hpp"
#include "radio_device.hpp"
#include "radio_launch.hpp"
#include "../runtime.hpp"

namespace c8mi::radio {
namespace {

constexpr double kC = 299792458.;
constexpr double kE = 1.6021766208e-19;
constexpr double kEps0 = 8.8541878128e-12;
constexpr double kPi = 3.141592653589793238462643383279502884;
constexpr double kEmConstant = 1. / (4. * kPi * kEps0 * kC);
constexpr double kChargeEm = kE * kEmConstant;
constexpr double kCoreasThreshold = 1.e-3;

struct V3 {
  double x, y, z;
};
__device__ __forceinline__ V3 vadd(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 vsub(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ V3 vmul(V3 a, double s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ V3 vdiv(V3 a, double s) { return {a.x / s, a.y / s, a.z / s}; }
__device__ __forceinline__ double vdot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 vcross(V3 a, V3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

__device__ __forceinline__ double nearest_bin(double scaled) {
  double const integral = floor(scaled);
  return integral + (scaled - integral >= 0.5 ? 1. : 0.);
}

// Device form of co_reas_doppler: error-free products and sums when the
// ordinary expression cancels to exactly zero.
__device__ __forceinline__ double doppler(double index, V3 beta, V3 emit) {
  double const ordinary = 1. - index * vdot(beta, emit);
  if (ordinary != 0.) return ordinary;
  double const px = beta.x * emit.x, py = beta.y * emit.y, pz = beta.z * emit.z;
  double const ex = fma(beta.x, emit.x, -px);
  double const ey = fma(beta.y, emit.y, -py);
  double const ez = fma(beta.z, emit.z, -pz);
  double const xy = px + py;
  double const xyv = xy - px;
  double const xye = (px - (xy - xyv)) + (py - xyv);
  double const xyz = xy + pz;
  double const xyzv = xyz - xy;
  double const xyze = (xy - (xyz - xyzv)) + (pz - xyzv);
  double const low = ex + ey + ez + xye + xyze;
  double const product = index * xyz;
  double const perr = fma(index, xyz, -product) + index * low;
  return (1. - product) - perr;
}

// ---- exact arithmetic ---------------------------------------------------------
//
// The reference's FP64 expressions in its operation order (correctly rounded
// IEEE division and square root, no contraction): the fixed-point waveforms
// equal the FP64 restatement's bit for bit. The fast form of the same updates
// is in radio_pair_fast.hpp.

struct Track {
  V3 start, end, disp, beta;
  double t0, t1, duration, length, beta_module, constant;
};

__device__ __forceinline__ bool load_track(double const* __restrict__ tracks,
                                           std::uint64_t stride, std::uint64_t i, Track& t) {
  t.start = {tracks[i], tracks[stride + i], tracks[2 * stride + i]};
  t.end = {tracks[3 * stride + i], tracks[4 * stride + i], tracks[5 * stride + i]};
  t.t0 = tracks[6 * stride + i];
  t.t1 = tracks[7 * stride + i];
  double const signed_weight = tracks[8 * stride + i];
  t.duration = t.t1 - t.t0;
  t.disp = vsub(t.end, t.start);
  t.length = sqrt(vdot(t.disp, t.disp));
  if (!(t.duration > 0.) || !(t.length > 0.)) return false;
  t.beta = vdiv(t.disp, kC * t.duration);
  t.beta_module = t.length / (kC * t.duration);
  t.constant = kChargeEm * signed_weight;
  return true;
}

// Observer quantities that do not depend on the track, evaluated once per
// thread with the same expressions propagate() and add_sample() use.
struct Obs {
  V3 position;
  double start, duration, rate, grid, wavelength;
  double nbins_d;
  std::int32_t nbins;
  std::uint64_t offset;
  double destination_height;
  std::uint64_t destination_index;
  double n_destination_table, integrated_destination;
};

struct Path {
  double time, n_source, n_destination, distance;
  V3 emit;
};

__device__ __forceinline__ Path propagate(PropagationDev const& p, V3 source, Obs const& o) {
  Path r;
  V3 const disp = vsub(o.position, source);
  r.distance = sqrt(vdot(disp, disp));
  r.emit = vdiv(disp, r.distance);
  double const distance = r.distance;
  if (p.homogeneous_index > 0.) {
    double const index = p.homogeneous_index;
    r.time = index * distance / kC;
    r.n_source = index;
    r.n_destination = index;
    return r;
  }
  double const source_height = (source.z - p.minimum_height) * p.inverse_step;
  double const destination_height = o.destination_height;
  std::uint64_t const last = p.table_size - 1;
  double n_source = 1.;
  double integrated_source = 1.;
  double n_destination = o.n_destination_table;
  double height = 1.;
  if (source_height + 0.5 >= static_cast<double>(last)) {
    n_source = p.refractivity[last] +
               p.slope_n_upper * fabs((source.z - p.maximum_height) * p.inverse_step) + 1.;
    integrated_source =
        p.integrated[last] + p.slope_i_upper * fabs(p.maximum_height - source.z);
    height = source_height - destination_height;
  } else if (source_height + 0.5 < static_cast<double>(last) && source_height > 0.) {
    // The table has fewer than 2^32 entries (checked on the host).
    std::uint32_t const source_index = static_cast<std::uint32_t>(source_height + 0.5);
    n_source = p.refractivity[source_index] + 1.;
    integrated_source = p.integrated[source_index];
    height = static_cast<double>(static_cast<std::int64_t>(source_index) -
                                 static_cast<std::int64_t>(o.destination_index)) *
             p.step;
    if (height == 0.) height = 1.;
  } else if (source_height == 0.) {
    n_source = 1.;
    n_destination = 1.;
    integrated_source = p.integrated[0];
    height = destination_height - source_height;
  } else {
    n_source = p.refractivity[0] + p.slope_n_lower * fabs(source_height) + 1.;
    integrated_source = p.integrated[0] + p.slope_i_lower * fabs(source_height);
    n_destination = 1.;
    height = destination_height - fabs(source_height);
  }
  r.time = (1. + (integrated_source - o.integrated_destination) / height) * distance / kC;
  r.n_source = n_source;
  r.n_destination = n_destination;
  return r;
}

// Per-thread tallies, folded into the block and then the global counters.
struct Tally {
  unsigned long long coreas = 0, zhs = 0, subtracks = 0, valid = 0, overflow = 0;
  double abs_sum = 0.;  // sum of |increments|, for kThreadLimit
};

// LDS accumulator for one mode: `Fixed` selects int64 fixed point (the
// production default) or FP64. The ZHS tile stores a difference array.
template <bool Fixed>
struct Tile {
  using Acc = std::conditional_t<Fixed, long long, double>;
  Acc* data;             // 3 components x stride
  std::uint32_t stride;  // bins per component row
  std::int32_t begin;    // first global bin of this tile
  std::int32_t bins;     // bins owned by this tile
  std::uint32_t observer;  // what contributions past the thread's limit need
  Budget* budgets;       // ZHS: of its ranges
};

// Below 2^51 (kThreadLimit) the round-to-nearest-even integer comes from adding
// 1.5 * 2^52 and reading the low mantissa bits: the same value as (long long) rint().
__device__ __forceinline__ long long fixed_increment(double scaled) {
  return __double_as_longlong(scaled + 6755399441055744.) - 0x4338000000000000LL;
}

template <class T>
__device__ __forceinline__ void lds_add(T* address, T value) {
  if constexpr (std::is_same_v<T, long long>)
    atomicAdd(reinterpret_cast<unsigned long long*>(address),
              static_cast<unsigned long long>(value));
  else
    atomicAdd(address, value);
}

// Bin of `time` per observer_nearest_bin; -1 when outside [0, nbins).
__device__ __forceinline__ std::int32_t sample_bin(Obs const& o, double time) {
  double const bin_value = nearest_bin((time - o.start) * o.rate);
  if (!(bin_value >= 0. && bin_value < o.nbins_d)) return -1;
  return static_cast<std::int32_t>(bin_value);
}

// CoREAS sample (add_sample with time gating, IsVectorPotential = false).
template <bool Fixed>
__device__ __forceinline__ void add_field_sample(Obs const& o, double scale,
                                                 Tile<Fixed> const& tile, double time, V3 c,
                                                 Tally& tally) {
  if (time < o.start || time > o.start + o.duration) return;
  std::int32_t const bin = sample_bin(o, time);
  if (bin < 0) return;
  std::int32_t const local = bin - tile.begin;
  if (local < 0 || local >= tile.bins) return;
  if constexpr (Fixed) {
    V3 const v = vmul(c, scale);
    double const magnitude = fabs(v.x) + fabs(v.y) + fabs(v.z);
    tally.abs_sum += magnitude;
    if (__builtin_expect(tally.abs_sum < kThreadLimit, 1)) {
      lds_add(tile.data + local, fixed_increment(v.x));
      lds_add(tile.data + tile.stride + local, fixed_increment(v.y));
      lds_add(tile.data + 2 * tile.stride + local, fixed_increment(v.z));
    } else {
      Rows const waves = waveform_rows<false>(tile.observer);
      double const vs[3] = {v.x, v.y, v.z};
      bool valid = true;
      unsigned long long overflows = 0;
      for (int k = 0; k < 3; ++k) {
        long long value = 0;
        if (!round_increment(vs[k], value)) valid = false;
        else if (magnitude < kThreadLimit)
          overflows += add_watched(tile.data + k * tile.stride + local, waves.row + k * waves.stride + bin, value);
        else overflows += checked_add(waves.row + k * waves.stride + bin, value);
      }
      // Counter updates are value selects: a branch between two tally fields
      // can become a store through a selected pointer, which pins the tally to
      // scratch memory.
      tally.overflow += overflows + (valid ? 0ull : 1ull);
      tally.coreas += valid ? 1ull : 0ull;
      return;
    }
  } else {
    lds_add(tile.data + local, c.x);
    lds_add(tile.data + tile.stride + local, c.y);
    lds_add(tile.data + 2 * tile.stride + local, c.z);
  }
  ++tally.coreas;
}

// Adds `c` to the ZHS bins [first, last] (inside [0, nbins)) through the
// difference array, clipped to the tile. Returns the number of this tile's
// bins that received it.
template <bool Fixed>
__device__ __forceinline__ std::int32_t add_potential_range(double scale,
                                                            Tile<Fixed> const& tile,
                                                            std::int32_t first,
                                                            std::int32_t last, V3 c,
                                                            Tally& tally, bool& valid) {
  std::int32_t const lo = (first > tile.begin ? first : tile.begin) - tile.begin;
  std::int32_t const hi =
      (last + 1 < tile.begin + tile.bins ? last + 1 : tile.begin + tile.bins) - tile.begin;
  valid = true;
  if (lo >= hi) return 0;
  if constexpr (Fixed) {
    V3 const v = vmul(c, scale);
    double const magnitude = fabs(v.x) + fabs(v.y) + fabs(v.z);
    tally.abs_sum += magnitude;
    double const vs[3] = {v.x, v.y, v.z};
    if (__builtin_expect(tally.abs_sum < kThreadLimit, 1)) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        long long const value = fixed_increment(vs[k]);
        lds_add(tile.data + k * tile.stride + lo, value);
        lds_add(tile.data + k * tile.stride + hi, -value);
      }
    } else {
      bool const in_tile = tile_takes(tile.budgets, static_cast<std::uint32_t>(lo), static_cast<std::uint32_t>(hi - 1),
                                      static_cast<std::uint32_t>(tile.bins), magnitude);
      Rows const waves = waveform_rows<true>(tile.observer);
      unsigned long long overflows = 0;
      for (int k = 0; k < 3; ++k) {
        long long value = 0;
        if (!round_increment(vs[k], value)) {
          valid = false;
        } else if (in_tile) {
          lds_add(tile.data + k * tile.stride + lo, value);
          lds_add(tile.data + k * tile.stride + hi, -value);
        } else {
          long long* const wave = waves.row + k * waves.stride + tile.begin;
          for (std::int32_t b = lo; b < hi; ++b) overflows += checked_add(wave + b, value);
        }
      }
      tally.overflow += overflows;
    }
  } else {
    lds_add(tile.data + lo, c.x);
    lds_add(tile.data + hi, -c.x);
    lds_add(tile.data + tile.stride + lo, c.y);
    lds_add(tile.data + tile.stride + hi, -c.y);
    lds_add(tile.data + 2 * tile.stride + lo, c.z);
    lds_add(tile.data + 2 * tile.stride + hi, -c.z);
  }
  return hi - lo;
}

// ZHS sample (add_sample with IsVectorPotential = true): no time gate.
template <bool Fixed>
__device__ __forceinline__ void add_potential_sample(Obs const& o, double scale,
                                                     Tile<Fixed> const& tile, double time, V3 c,
                                                     Tally& tally) {
  std::int32_t const bin = sample_bin(o, time);
  if (bin < 0) return;
  bool valid = true;
  std::int32_t const added = add_potential_range(scale, tile, bin, bin, c, tally, valid);
  unsigned long long const n = static_cast<unsigned long long>(added);
  tally.zhs += valid ? n : 0ull;
  tally.overflow += valid ? 0ull : n;
}

// separate_same_bin_endpoints (RadioProjection.inl:303-336).
__device__ __forceinline__ void separate_same_bin(double& start_time, double& end_time,
                                                  Obs const& o, bool signed_order) {
  double const s = start_time / o.grid;
  double const e = end_time / o.grid;
  if (static_cast<long long>(nearest_bin(s)) != static_cast<long long>(nearest_bin(e))) return;
  double const grid = o.grid;
  double const sf = s - floor(s);
  double const ef = e - floor(e);
  bool const forward = !signed_order || end_time >= start_time;
  if (forward) {
    if (sf >= 0.5 && ef >= 0.5) start_time -= grid;
    else if (sf < 0.5 && ef < 0.5) end_time += grid;
    else if (ef >= 1. - sf) end_time += grid;
    else start_time -= grid;
  } else {
    if (sf >= 0.5 && ef >= 0.5) end_time -= grid;
    else if (sf < 0.5 && ef < 0.5) start_time += grid;
    else if (sf >= 1. - ef) start_time += grid;
    else end_time -= grid;
  }
}

// t.constant * rate / (doppler * R)
__device__ __forceinline__ double field_scale(Track const& t, Obs const& o, double doppler_factor,
                                              Path const& path) {
  return t.constant * o.rate / (doppler_factor * path.distance);
}

template <bool Fixed>
__device__ __forceinline__ void coreas_pair(Track const& t, PropagationDev const& p, Obs const& o,
                            double scale, Tile<Fixed> const& tile, Tally& tally) {
  Path const ps = propagate(p, t.start, o);
  Path const pe = propagate(p, t.end, o);
  double const pre = doppler(ps.n_source, t.beta, ps.emit);
  double const post = doppler(pe.n_source, t.beta, pe.emit);
  double start_receive = t.t0 + ps.time;
  double end_receive = t.t1 + pe.time;
  if (ps.n_destination > 1. &&
      (fabs(pre) < kCoreasThreshold || fabs(post) < kCoreasThreshold)) {
    V3 const midpoint = vmul(vadd(t.start, t.end), 0.5);
    double const middle_time = (t.t0 + t.t1) * 0.5;
    Path const pm = propagate(p, midpoint, o);
    double const middle_receive = middle_time + pm.time;
    double const md = doppler(pm.n_source, t.beta, pm.emit);
    V3 field_start =
        vmul(vcross(pm.emit, vcross(pm.emit, t.beta)), field_scale(t, o, md, pm));
    V3 field_end = vmul(field_start, -1.);
    double delta;
    delta = t.length / (kC * t.beta_module) * fabs(md);
    if (start_receive < end_receive) {
      start_receive = middle_receive - 0.5 * delta;
      end_receive = middle_receive + 0.5 * delta;
    } else {
      start_receive = middle_receive + 0.5 * delta;
      end_receive = middle_receive - 0.5 * delta;
    }
    delta = end_receive - start_receive;
    if (fabs(delta) < o.grid) {
      double const shrink = fabs(delta / o.grid);
      field_start = vmul(field_start, shrink);
      field_end = vmul(field_end, shrink);
      separate_same_bin(start_receive, end_receive, o, true);
    }
    add_field_sample(o, scale, tile, start_receive, field_start, tally);
    add_field_sample(o, scale, tile, end_receive, field_end, tally);
    return;
  }
  V3 field_start =
      vmul(vcross(ps.emit, vcross(ps.emit, t.beta)), field_scale(t, o, pre, ps));
  V3 field_end =
      vmul(vcross(pe.emit, vcross(pe.emit, t.beta)), -field_scale(t, o, post, pe));
  if (pre < 1.e-9 || post < 1.e-9) {
    double const delta = end_receive - start_receive;
    if (fabs(delta) < o.grid) {
      double const shrink = fabs(delta / o.grid);
      field_start = vmul(field_start, shrink);
      field_end = vmul(field_end, shrink);
      separate_same_bin(start_receive, end_receive, o, false);
    }
  }
  add_field_sample(o, scale, tile, start_receive, field_start, tally);
  add_field_sample(o, scale, tile, end_receive, field_end, tally);
}

template <bool Fixed>
__device__ __forceinline__ void zhs_segment(V3 p1, V3 p2, double time1, double time2, Track const& t,
                            PropagationDev const& p, Obs const& o, double scale,
                            Tile<Fixed> const& tile, Tally& tally, bool subdivided,
                            bool use_cached, Path cached_midpoint_path) {
  // The cached path travels by value: a pointer to the caller's local would
  // pin it to scratch memory.
  Path const path = use_cached ? cached_midpoint_path
                               : propagate(p, vmul(vadd(p1, p2), 0.5), o);
  double const n_source = path.n_source;
  double const bk = vdot(t.beta, path.emit);
  double const middle_time = (time1 + time2) * 0.5;
  double d1 = time1 + path.time - n_source * bk * (time1 - middle_time);
  double d2 = time2 + path.time - n_source * bk * (time2 - middle_time);
  double sign = 1.;
  if (d1 > d2) {
    d1 = time2 + path.time - n_source * bk * (time2 - middle_time);
    d2 = time1 + path.time - n_source * bk * (time1 - middle_time);
    sign = -1.;
  }
  double const x1 = (d1 - o.start) * o.rate;
  double const start_bin = floor(x1 + 0.5);
  double const end_bin = floor((d2 - o.start) * o.rate + 0.5);
  V3 const bperp = vcross(path.emit, vcross(t.beta, path.emit));
  double const den = 1. - n_source * bk;
  V3 potential;  // of the last bin
  if (start_bin == end_bin) {
    if (fabs(den) > 1.e-15) {
      double const fraction = fabs(d2 * o.rate - d1 * o.rate);
      potential = vmul(bperp, sign * t.constant * fraction / (den * path.distance));
    } else {
      double const fraction = (time2 - time1) * o.rate;
      potential = vmul(bperp, sign * t.constant * fraction / path.distance);
    }
  } else {
    int const nb = static_cast<int>(end_bin - start_bin);
    double fraction = fabs(start_bin + 0.5 - x1);
    potential = vmul(bperp, sign * t.constant * fraction / (den * path.distance));
    add_potential_sample(o, scale, tile, d1, potential, tally);
    if (nb > 1) {
      V3 const middle = vmul(bperp, (subdivided ? 1. : sign) * t.constant / (den * path.distance));
      // Bins of the first and last middle sample, exactly as the per-bin loop
      // computes them; in between the bins are consecutive.
      double const b_first = nearest_bin((d1 + 1. / o.rate - o.start) * o.rate);
      double const b_last = nearest_bin((d1 + static_cast<double>(nb - 1) / o.rate - o.start) * o.rate);
      if (b_last - b_first == static_cast<double>(nb - 2)) {
        double const lo = b_first < 0. ? 0. : b_first;
        double const hi = b_last < o.nbins_d - 1. ? b_last : o.nbins_d - 1.;
        if (lo <= hi) {
          bool valid = true;
          std::int32_t const added =
              add_potential_range(scale, tile, static_cast<std::int32_t>(lo),
                                  static_cast<std::int32_t>(hi), middle, tally, valid);
          unsigned long long const n = static_cast<unsigned long long>(added);
          tally.zhs += valid ? n : 0ull;
          tally.overflow += valid ? 0ull : n;
        }
      } else {
        for (int index = 1; index < nb; ++index)
          add_potential_sample(o, scale, tile, d1 + static_cast<double>(index) / o.rate, middle,
                               tally);
      }
    }
    fraction = fabs((d2 - o.start) * o.rate + 0.5 - end_bin);
    potential = vmul(bperp, sign * t.constant * fraction / (den * path.distance));
  }
  add_potential_sample(o, scale, tile, d2, potential, tally);
}

template <bool Fixed>
__device__ __forceinline__ void zhs_pair(Track const& t, PropagationDev const& p, std::uint32_t refinement_u,
                         Obs const& o, double scale, Tile<Fixed> const& tile, Tally& tally,
                         bool count_subtracks) {
  V3 const midpoint = vmul(vadd(t.start, t.end), 0.5);
  Path const mp = propagate(p, midpoint, o);
  double const u_k = vdot(t.beta, mp.emit) / t.beta_module;
  double const sin2 = 1. - u_k * u_k;
  double const fraunhofer = sin2 * t.length * t.length / mp.distance / o.wavelength * 2. * kPi;
  double divisor = 1.;
  int nsub = 1;
  if (fraunhofer > 1.) {
    divisor = sqrt(fraunhofer) + 1.;
    nsub = static_cast<int>(ceil(divisor));
  }
  int const refinement = static_cast<int>(refinement_u);
  if (count_subtracks) {
    tally.subtracks += static_cast<unsigned long long>(nsub);
    if (refinement > 1)
      tally.subtracks += static_cast<unsigned long long>(nsub * (refinement - 1));
  }
  bool const subdivided = nsub > 1 || refinement > 1;
  // Unsubdivided, divisor == refinement == 1 and x / 1. is x exactly: the
  // single segment runs from start to start + displacement over the full
  // duration, so the divisions are skipped. Its midpoint is the track
  // midpoint whenever start + displacement == end bit for bit, and the
  // propagation above is then reused unchanged.
  V3 rs = t.disp;
  double rt = t.duration;
  bool use_cached = false;
  if (subdivided) {
    V3 const spatial_step = vdiv(t.disp, divisor);
    double const time_step = t.duration / divisor;
    rs = vdiv(spatial_step, static_cast<double>(refinement));
    rt = time_step / static_cast<double>(refinement);
  } else {
    V3 const p2 = vadd(t.start, t.disp);
    use_cached = __double_as_longlong(p2.x) == __double_as_longlong(t.end.x) &&
                 __double_as_longlong(p2.y) == __double_as_longlong(t.end.y) &&
                 __double_as_longlong(p2.z) == __double_as_longlong(t.end.z);
  }
  int const segments = nsub * refinement;
  V3 p1 = t.start;
  double time1 = t.t0;
  for (int i = 0; i < segments; ++i) {
    V3 const p2 = vadd(p1, rs);
    double const time2 = time1 + rt;
    zhs_segment(p1, p2, time1, time2, t, p, o, scale, tile, tally, subdivided, use_cached,
                       mp);
    p1 = p2;
    time1 = time2;
  }
}

__device__ __forceinline__ Obs make_obs(ObserverDev const& d, PropagationDev const& p) {
  Obs o;
  o.position = {d.position[0], d.position[1], d.position[2]};
  o.start = d.start_time;
  o.duration = d.duration;
  o.rate = d.sample_rate;
  o.grid = 1. / d.sample_rate;
  o.wavelength = kC / d.sample_rate;
  o.nbins = static_cast<std::int32_t>(d.number_of_bins);
  o.nbins_d = static_cast<double>(d.number_of_bins);
  o.offset = d.waveform_offset;
  if (p.homogeneous_index > 0.) {
    o.destination_height = 0.;
    o.destination_index = 0;
    o.n_destination_table = 1.;
    o.integrated_destination = 0.;
  } else {
    o.destination_height = (o.position.z - p.minimum_height) * p.inverse_step;
    o.destination_index = static_cast<std::uint64_t>(o.destination_height + 0.5);
    o.n_destination_table = p.refractivity[o.destination_index] + 1.;
    o.integrated_destination = p.integrated[o.destination_index];
  }
  return o;
}

template <bool Coreas, bool Zhs, bool Fixed, int Block>
__global__ void __launch_bounds__(Block, 4) radio_exact_kernel(ProjectionLaunch L) {
  using Acc = std::conditional_t<Fixed, long long, double>;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ Acc scan_scratch[Zhs ? Block / 64 : 1];
  __shared__ BlockTallies block;
  __shared__ Budget budgets[kRanges];

  std::uint32_t observer, bin_tile, within;
  std::uint64_t chunk_begin, chunk_end;
  CountersDev* counters = L.counters;
  bool first_observer_tile;
  if (L.segments == nullptr) {
    if (!decode_chunk(L, L.observer_count * L.bin_tiles, within, chunk_begin, chunk_end)) return;
    observer = within / L.bin_tiles;
    bin_tile = within % L.bin_tiles;
    first_observer_tile = L.count_valid && within == 0;
  } else {
    SegmentDev seg;
    std::uint64_t local;
    if (!decode_segment(L, seg, local)) return;
    std::uint64_t const per_chunk =
        static_cast<std::uint64_t>(L.slot_observer_counts[seg.slot]) * L.bin_tiles;
    std::uint64_t const chunk = local / per_chunk;
    within = static_cast<std::uint32_t>(local % per_chunk);
    observer = seg.slot * L.slot_observers + within / L.bin_tiles;
    bin_tile = within % L.bin_tiles;
    chunk_begin = seg.begin + chunk * L.chunk_size;
    chunk_end = chunk_begin + L.chunk_size < seg.end ? chunk_begin + L.chunk_size : seg.end;
    counters = L.counters + seg.slot;
    first_observer_tile = L.count_valid && within == 0;
  }

  std::uint32_t const W = L.tile_bins;
  Acc* const coreas_lds = reinterpret_cast<Acc*>(lds_raw);
  Acc* const zhs_lds = coreas_lds + (Coreas ? 3 * W : 0);
  std::uint32_t const lds_count = (Coreas ? 3 * W : 0) + (Zhs ? 3 * (W + 1) : 0);
  for (std::uint32_t i = threadIdx.x; i < lds_count; i += blockDim.x) coreas_lds[i] = 0;
  if (threadIdx.x < kRanges) budgets[threadIdx.x] = 0.;
  clear_tallies(block);
  __syncthreads();

  PropagationDev const prop = L.propagation;
  std::uint64_t const tile_begin = static_cast<std::uint64_t>(bin_tile) * W;
  // A fused launch has identical CoREAS and ZHS observers (position, window,
  // rate, bins and hence offsets); only their fixed-point scales differ.
  ObserverDev const& view = Coreas ? L.coreas_observers[observer] : L.zhs_observers[observer];
  Obs const o = make_obs(view, prop);
  double const coreas_scale = Coreas ? L.coreas_observers[observer].fixed_scale : 0.;
  double const zhs_scale = Zhs ? L.zhs_observers[observer].fixed_scale : 0.;
  std::uint64_t const nbins = static_cast<std::uint64_t>(o.nbins);
  std::uint32_t const tile_bins =
      tile_begin < nbins ? static_cast<std::uint32_t>(nbins - tile_begin < W ? nbins - tile_begin : W)
                         : 0u;
  Tile<Fixed> const ctile{coreas_lds, W, static_cast<std::int32_t>(tile_begin),
                          static_cast<std::int32_t>(tile_bins), observer, budgets};
  Tile<Fixed> const ztile{zhs_lds, W + 1, static_cast<std::int32_t>(tile_begin),
                          static_cast<std::int32_t>(tile_bins), observer, budgets};

  Tally ctally, ztally;
  for (std::uint64_t i = chunk_begin + threadIdx.x; i < chunk_end; i += blockDim.x) {
    Track t;
    if (!load_track(L.tracks, L.stride, i, t)) continue;
    if (first_observer_tile) ++ctally.valid;
    if constexpr (Coreas) {
      if (tile_bins) coreas_pair(t, prop, o, coreas_scale, ctile, ctally);
    }
    if constexpr (Zhs) {
      zhs_pair(t, prop, L.zhs_refinement, o, zhs_scale, ztile, ztally, bin_tile == 0);
    }
  }
  unsigned long long const counts[5] = {ctally.coreas, ztally.zhs, ztally.subtracks, ctally.valid,
                                        ctally.overflow + ztally.overflow};
  add_tallies<Coreas, Zhs>(block, counts);
  __syncthreads();

  if constexpr (Zhs) {
    for (int c = 0; c < 3; ++c) block_inclusive_scan(zhs_lds + c * (W + 1), W, scan_scratch);
  }
  unsigned long long overflows = 0;
  std::uint64_t const first = o.offset + tile_begin;
  if constexpr (Coreas)
    overflows += flush_tile<Fixed>(coreas_lds, W, tile_bins, L.coreas_waves, L.coreas_total_bins, first);
  if constexpr (Zhs) overflows += flush_tile<Fixed>(zhs_lds, W + 1, tile_bins, L.zhs_waves, L.zhs_total_bins, first);
  if (overflows) atomicAdd(&block.counts[4], overflows);
  __syncthreads();
  publish_tallies(block, counters);
}

// LeptonTransportRecord -> compact track (make_radio_track_kinematics input
// selection, RadioProjection.inl:145-168). Non-e+- records become zero-length
// tracks, which the projection rejects exactly as the reference does.
__global__ void __launch_bounds__(256)
    records_to_tracks_kernel(c8mi_lepton_transport_record const* __restrict__ records,
                             std::uint64_t count, double* __restrict__ tracks,
                             std::uint64_t stride) {
  std::uint64_t const i = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  c8mi_lepton_transport_record const& r = records[i];
  int const pid = r.start.pid;
  bool const lepton = pid == C8MI_PID_ELECTRON || pid == C8MI_PID_POSITRON;
  double const w = r.start.weight;
  tracks[i] = lepton ? r.start.position_m[0] : 0.;
  tracks[stride + i] = lepton ? r.start.position_m[1] : 0.;
  tracks[2 * stride + i] = lepton ? r.start.position_m[2] : 0.;
  tracks[3 * stride + i] = lepton ? r.end.position_m[0] : 0.;
  tracks[4 * stride + i] = lepton ? r.end.position_m[1] : 0.;
  tracks[5 * stride + i] = lepton ? r.end.position_m[2] : 0.;
  tracks[6 * stride + i] = lepton ? r.start.time_s : 0.;
  tracks[7 * stride + i] = lepton ? r.end.time_s : 0.;
  tracks[8 * stride + i] = pid == C8MI_PID_ELECTRON ? -w : w;
}

template <bool Coreas, bool Zhs, bool Fixed, int Block>
void launch_typed(ProjectionLaunch const& launch, hipStream_t stream, std::size_t lds_bytes,
                  std::uint32_t grid) {
  auto kernel = radio_exact_kernel<Coreas, Zhs, Fixed, Block>;
  static bool attribute_set = false;
  if (!attribute_set) {
    C8MI_HIP(hipFuncSetAttribute(reinterpret_cast<void const*>(kernel),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(kMaxDynamicLdsBytes)));
    attribute_set = true;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Block), lds_bytes, stream, launch);
  C8MI_HIP(hipGetLastError());
}

template <bool Coreas, bool Zhs, bool Fixed>
void launch_block(ProjectionLaunch const& launch, std::uint32_t block, hipStream_t stream,
                  std::size_t lds_bytes, std::uint32_t grid) {
  switch (block) {
    case 256: launch_typed<Coreas, Zhs, Fixed, 256>(launch, stream, lds_bytes, grid); break;
    case 512: launch_typed<Coreas, Zhs, Fixed, 512>(launch, stream, lds_bytes, grid); break;
    case 1024: launch_typed<Coreas, Zhs, Fixed, 1024>(launch, stream, lds_bytes, grid); break;
    default: throw std::invalid_argument("radio workgroup size must be 256, 512 or 1024");
  }
}

// CoREAS and ZHS in one exact kernel need more registers than four waves a SIMD
// leave, and a 2048-bin window two tiles: 6.1 ms against 3.3 for 5e5 tracks on 100
// antennas. So there is none.
template <bool Coreas, bool Zhs>
void launch_exact(ProjectionLaunch const& launch, std::uint32_t block, hipStream_t stream, std::size_t lds,
                  std::uint32_t grid) {
  if constexpr (Coreas && Zhs) throw std::logic_error("radio: an exact projection takes its algorithms one by one");
  else launch_block<Coreas, Zhs, true>(launch, block, stream, lds, grid);
}

template <bool Coreas, bool Zhs>
void launch_modes(ProjectionLaunch const& launch, bool fixed, bool exact, std::uint32_t block,
                  hipStream_t stream, std::size_t lds, std::uint32_t grid) {
  // FP64 (non-deterministic) accumulation is offered in the exact form only.
  if (!fixed) launch_block<Coreas, Zhs, false>(launch, block, stream, lds, grid);
  else if (exact) launch_exact<Coreas, Zhs>(launch, block, stream, lds, grid);
  else launch_fast(launch, Coreas, Zhs, block, grid, stream);
}

}  // namespace

std::size_t projection_lds_bytes(bool coreas, bool zhs, std::uint32_t tile_bins) {
  std::size_t const words = (coreas ? 3u * tile_bins : 0u) + (zhs ? 3u * (tile_bins + 1u) : 0u);
  return words * sizeof(long long);
}

std::uint32_t projection_grid(ProjectionLaunch const& launch) {
  std::uint64_t const groups = (launch.observer_count + launch.group - 1) / launch.group;
  std::uint64_t const chunk_rounds = (launch.chunks + kXcds - 1) / kXcds;
  return static_cast<std::uint32_t>(chunk_rounds * kXcds * groups * launch.bin_tiles);
}

void launch_projection(ProjectionLaunch const& launch, bool coreas, bool zhs, bool fixed,
                       bool exact, hipStream_t stream) {
  std::uint32_t const block = launch.block_threads;
  if (launch.track_count == 0 || launch.observer_count == 0) return;
  std::size_t const lds = projection_lds_bytes(coreas, zhs, launch.tile_bins);
  std::uint32_t const grid = projection_grid(launch);
  if (coreas && zhs) launch_modes<true, true>(launch, fixed, exact, block, stream, lds, grid);
  else if (coreas) launch_modes<true, false>(launch, fixed, exact, block, stream, lds, grid);
  else if (zhs) launch_modes<false, true>(launch, fixed, exact, block, stream, lds, grid);
}

void launch_pooled_projection(ProjectionLaunch const& launch, bool coreas, bool zhs, bool exact,
                              std::uint32_t grid, hipStream_t stream) {
  std::uint32_t const block = launch.block_threads;
  if (launch.track_count == 0 || grid == 0) return;
  std::size_t const lds = projection_lds_bytes(coreas, zhs, launch.tile_bins);
  if (coreas && zhs) launch_modes<true, true>(launch, true, exact, block, stream, lds, grid);
  else if (coreas) launch_modes<true, false>(launch, true, exact, block, stream, lds, grid);
  else if (zhs) launch_modes<false, true>(launch, true, exact, block, stream, lds, grid);
}

void launch_records_to_tracks(c8mi_lepton_transport_record const* records, std::uint64_t count,
                              double* tracks, std::uint64_t stride, hipStream_t stream) {
  if (count == 0) return;
  std::uint32_t const blocks = static_cast<std::uint32_t>((count + 255) / 256);
  hipLaunchKernelGGL(records_to_tracks_kernel, dim3(blocks), dim3(256), 0, stream, records,
                     count, tracks, stride);
  C8MI_HIP(hipGetLastError());
}

}  // namespace c8mi::radio
