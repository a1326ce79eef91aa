"""The measured workloads of c8mi: what a program around CORSIKA has it do, through the
public binding (`c8mi`, `c8mi.em`), over the sizes and options that are in use.

Two paths, EM transport (showers, a pool of showers, the serving stream, the host handoff,
the in-ice cascade) and the radio projection (standalone track lists and the tracks of the
showers above). Inputs follow `c8mi.workloads`, the generators of the benchmark and tests.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "corsika8-kokkos_amd"))

import c8mi  # noqa: E402
from c8mi import airtables, em, workloads  # noqa: E402

C = workloads.SPEED_OF_LIGHT
N_ICE = 1.78
START, DOWN = (0.0, 0.0, 112750.0), (0.0, 0.0, -1.0)
ICE_START = (0.0, 0.0, -100.0)
FIELD_T = (2.0e-5, 0.0, -4.0e-5)  # an Earth-like field


def listed():
    return [
        # -- EM transport -------------------------------------------------------------------
        # the smallest whole call: one 1 GeV photon, about a thousand steps in some hundred
        # fronts of a few particles each; a host that asks for single small showers
        {"name": "shower_1gev", "kind": "shower", "pid": 22, "energy": 1.0, "zenith": 0.0, "field": False,
         "thinning": 0.0, "moliere": "table"},
        # the benchmark's 100 GeV photon, one at a time: latency of a whole shower
        {"name": "shower_100gev", "kind": "shower", "pid": 22, "energy": 100.0, "zenith": 0.0, "field": False,
         "thinning": 0.0, "moliere": "table"},
        # an inclined 1 TeV positron in a magnetic field, thinned, analytical Moliere functions:
        # the curved-step branch and the options a production run switches on
        {"name": "shower_field_thinned", "kind": "shower", "pid": -11, "energy": 1000.0, "zenith": 40.0,
         "field": True, "thinning": 1e-4, "moliere": "analytic"},
        # the benchmark's EM throughput form, a pool of showers with their host prefixes
        {"name": "pool_100gev", "kind": "pool", "pid": 22, "energy": 100.0, "showers": 1000, "slots": 512},
        # the serving loop: mixed requests, each with its own axis and 40 antennas
        {"name": "stream_radio", "kind": "stream", "requests": 21, "low": 100.0, "high": 3000.0, "slots": 64,
         "arms": 8, "radii": 5, "bins": 1024},
        # a whole shower through the host handoff with 160 antennas, CoREAS and ZHS
        {"name": "handoff_radio_10tev", "kind": "handoff", "pid": 11, "energy": 1.0e4, "arms": 8, "radii": 20,
         "bins": 1024},
        # the in-ice cascade with ZHS on the Cherenkov ring
        {"name": "ice_zhs_10tev", "kind": "ice", "energy": 1.0e4, "antennas": 64, "bins": 4096},
        # -- radio projection alone ---------------------------------------------------------
        # a host that hands over a handful of 752-byte track records and reads the field back
        {"name": "radio_records_small", "kind": "radio", "api": "records", "tracks": 1500, "antennas": 24,
         "bins": 512, "rate": 1.0e9, "medium": "air", "mode": "both", "exact": False, "fixed": True,
         "refinement": 1},
        # the benchmark's headline list: 2^20 tracks on 160 antennas, 2048 bins at 0.2 ns
        {"name": "radio_standalone", "kind": "radio", "api": "tracks", "tracks": 1 << 20, "antennas": 160,
         "bins": 2048, "rate": 5.0e9, "medium": "air", "mode": "both", "exact": False, "fixed": True,
         "refinement": 1},
        # a lepton front's worth of in-ice tracks on a long window, ZHS only, ragged count
        {"name": "radio_ice_zhs", "kind": "radio", "api": "tracks", "tracks": 100003, "antennas": 64,
         "bins": 4096, "rate": 1.0e10, "medium": "ice", "mode": "zhs", "exact": False, "fixed": True,
         "refinement": 1},
        # the reference's campaign shape (79 antennas, 400 ns at 1 GHz) with its own FP64
        # operation order (exact) and refined ZHS tracks
        {"name": "radio_exact_refined", "kind": "radio", "api": "tracks", "tracks": 131077, "antennas": 79,
         "bins": 400, "rate": 1.0e9, "medium": "air", "mode": "both", "exact": True, "fixed": True,
         "refinement": 3},
        # the call without allocations, into device buffers that stay on the GPU
        {"name": "radio_device_buffers", "kind": "radio", "api": "noalloc", "tracks": 30000, "antennas": 160,
         "bins": 1024, "rate": 2.0e9, "medium": "air", "mode": "both", "exact": False, "fixed": True,
         "refinement": 1},
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    kind = rng.choice(("shower", "shower", "pool", "stream", "handoff", "ice", "radio", "radio", "radio", "radio"))
    if kind == "shower":
        field = rng.random() < 0.3
        energy = _log(rng, 1.0, 1000.0)
        return {"kind": kind, "pid": rng.choice((22, 11, -11)), "energy": round(energy, 3),
                "zenith": round(rng.uniform(0.0, 60.0), 2), "field": field,
                "thinning": 1e-4 if rng.random() < 0.4 else 0.0, "moliere": rng.choice(("table", "table", "analytic", "off"))}
    if kind == "pool":
        return {"kind": kind, "pid": rng.choice((22, 11)), "energy": round(_log(rng, 10.0, 100.0), 3),
                "showers": int(_log(rng, 16, 1000)), "slots": rng.choice((64, 200, 512))}
    if kind == "stream":
        return {"kind": kind, "requests": rng.randint(3, 20), "low": 100.0, "high": round(_log(rng, 300.0, 3000.0), 2),
                "slots": rng.choice((8, 64)), "arms": 8, "radii": rng.randint(1, 5), "bins": rng.choice((400, 777, 1024))}
    if kind == "handoff":
        return {"kind": kind, "pid": rng.choice((22, 11)), "energy": round(_log(rng, 100.0, 1.0e4), 2), "arms": 8,
                "radii": rng.randint(3, 20), "bins": rng.choice((512, 1000, 1024))}
    if kind == "ice":
        return {"kind": kind, "energy": round(_log(rng, 100.0, 1.0e4), 2), "antennas": rng.randint(8, 64),
                "bins": rng.choice((1024, 3001, 4096))}
    medium = rng.choice(("air", "air", "ice"))
    exact = rng.random() < 0.3
    api = rng.choice(("tracks", "tracks", "records", "noalloc"))
    fixed = api == "noalloc" or not exact or rng.random() < 0.7
    tracks = int(_log(rng, 500, 16384)) if api == "records" else int(_log(rng, 1000, 1 << 20))
    antennas = rng.randint(3, 160)
    antennas = max(3, min(antennas, int(1.6e8 / (4 if exact else 1) / tracks)))
    return {"kind": "radio", "api": api, "tracks": tracks, "antennas": antennas,
            "bins": rng.choice((333, 512, 1024, 2048, 4096)), "rate": rng.choice((1.0e9, 2.0e9, 5.0e9, 1.0e10)),
            "medium": medium, "mode": rng.choice(("both", "both", "coreas", "zhs")), "exact": exact, "fixed": fixed,
            "refinement": 1 if rng.random() < 0.8 else 2}


# ---- what a program builds once --------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _air_tables():
    return airtables.build_air_tables()


@functools.lru_cache(maxsize=None)
def _ice_tables():
    return airtables.build_ice_tables(cut_mev=0.1)


@functools.lru_cache(maxsize=None)
def _air_propagation(maximum_height):
    refractivity = workloads.exponential_refractivity(-1000.0, maximum_height, 1.0)
    return c8mi.Propagation(refractivity=refractivity, minimum_height_m=-1000.0, maximum_height_m=maximum_height,
                            step_m=1.0)


def _inclined(zenith_deg):
    th = math.radians(zenith_deg)
    d = np.array([math.sin(th), 0.0, -math.cos(th)])
    r, h, c = em.EARTH_RADIUS_M, START[2] - 750.0, math.cos(th)
    slant = -r * c + math.sqrt(r * r * c * c + h * h + 2.0 * r * h)
    return tuple(-slant * d), tuple(d)


def _ice_tracks(count, seed):
    """e+- steps of an in-ice cascade: a column of short steps along the axis around its
    maximum, most within a few centimetres of it, most nearly along it."""
    rng = np.random.default_rng(seed)
    along = rng.gamma(9.0, 0.45, count)
    lateral = rng.normal(0.0, 0.04, (2, count))
    start = np.stack([lateral[0], lateral[1], ICE_START[2] - along])
    tilt = rng.normal(0.0, 0.25, (2, count))
    d = np.stack([tilt[0], tilt[1], -np.ones(count)])
    d /= np.linalg.norm(d, axis=0)
    length = 10.0 ** rng.uniform(-4.0, -1.7, count)
    beta = rng.uniform(0.9, 1.0, count)
    out = np.empty((9, count))
    out[0:3] = start
    out[3:6] = start + length * d
    out[6] = along / C + rng.exponential(2e-11, count)
    out[7] = out[6] + length / (beta * C)
    out[8] = np.where(rng.random(count) < 0.6, -1.0, 1.0) * rng.choice((1.0, 1.0, 3.5), count)
    return out


def _radio_inputs(case, seed):
    """Track list [9][n], observers and the propagation of a standalone projection."""
    if case["medium"] == "ice":
        tracks = _ice_tracks(case["tracks"], seed)
        center = np.array(ICE_START) - np.array([0.0, 0.0, 4.0])
        observers = workloads.cherenkov_ring_observers(center, DOWN, 1000.0, N_ICE, count=case["antennas"],
                                                       sample_rate_hz=case["rate"], number_of_bins=case["bins"],
                                                       emission_time_s=4.0 / C,
                                                       pretrigger_s=min(100e-9, 0.25 * case["bins"] / case["rate"]))
        return tracks, observers, c8mi.Propagation(homogeneous_index=N_ICE)
    tracks = workloads.radio_config2_tracks(case["tracks"], seed)
    observers = workloads.star_observers(arms=8, radii=-(-case["antennas"] // 8), sample_rate_hz=case["rate"],
                                         number_of_bins=case["bins"])[:case["antennas"]].copy()
    observers["start_time_s"] = workloads.earliest_arrivals(tracks, observers) - 10.0e-9
    return tracks, observers, _air_propagation(110000.0)


def _accumulator(case, observers, propagation):
    return c8mi.RadioAccumulator(observers, propagation, coreas=case["mode"] != "zhs", zhs=case["mode"] != "coreas",
                                 deterministic=case["fixed"], zhs_refinement=case["refinement"], exact=case["exact"])


def _backend(seed, tables_module, tables, environment, start, direction, **kw):
    cfg = em.make_config(tables_module, seed=1 + seed, atmosphere=environment, start=start, direction=direction, **kw)
    return cfg, em.EmBackend(cfg, tables, environment)


# ---- the calls ---------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "seed": seed}
    if kind == "radio":
        tracks, observers, prop = _radio_inputs(case, seed)
        s.update(observers=observers, propagation=prop)
        if case["api"] == "records":
            s["records"] = workloads.tracks_to_records(tracks)
        else:
            s["tracks"] = torch.from_numpy(tracks).cuda()
        if case["api"] == "noalloc":
            total = int(observers["number_of_bins"].sum())
            s["buffers"] = [torch.empty((3, total), dtype=torch.int64, device="cuda") for _ in range(2)]
        else:
            s["accumulator"] = _accumulator(case, observers, prop)
        return s
    if kind == "shower":
        start, direction = _inclined(case["zenith"]) if case["zenith"] else (START, DOWN)
        air = em.Atmosphere(magnetic_field_t=FIELD_T if case["field"] else (0.0, 0.0, 0.0))
        thinning = (case["thinning"] * case["energy"], 1.0e3) if case["thinning"] else None
        s["config"], s["backend"] = _backend(
            seed, airtables, _air_tables(), air, start, direction, queue_capacity=1 << 20, observation_capacity=1 << 16,
            fallback_capacity=1 << 10, thinning=thinning, moliere=case["moliere"] != "off",
            moliere_table=True if case["moliere"] == "table" else None)
        s["primary"] = em.particle(case["pid"], case["energy"], start, direction, history_id=1)
        return s
    if kind == "pool":
        s["config"], s["backend"] = _backend(
            seed, airtables, _air_tables(), em.Atmosphere(), START, DOWN, slots=case["slots"], queue_capacity=1 << 22,
            observation_capacity=1 << 12, fallback_capacity=1 << 8, moliere=True, moliere_table=True,
            moliere_fast_iterations=5, resident_minimum_batch=16384)
        primary = em.particle(case["pid"], case["energy"], START, DOWN, history_id=1)
        s["requests"] = [dict(primary=primary, shower_id=1000 + k, arrival_s=0.0,
                              footprint=em.footprint_estimate(case["energy"])) for k in range(case["showers"])]
        return s
    if kind == "stream":
        air, prop = em.Atmosphere(), _air_propagation(113000.0)
        stream = workloads.serving_stream(case["requests"], 40.0, seed=seed + 7, e_min_gev=case["low"],
                                          e_max_gev=case["high"], arms=case["arms"], radii=case["radii"],
                                          bins=case["bins"])
        s["config"], s["backend"] = _backend(
            seed, airtables, _air_tables(), air, START, DOWN, slots=case["slots"], queue_capacity=1 << 22,
            observation_capacity=1 << 12, fallback_capacity=1 << 8, moliere=True, moliere_table=True)
        s["backend"].enable_slot_radio(case["arms"] * case["radii"], case["bins"], prop)
        s["requests"] = [dict(primary=em.particle(r["pid"], r["energy_gev"], tuple(r["start_m"]), tuple(r["direction"]),
                                                  history_id=1),
                              shower_id=100 + k, arrival_s=0.0, footprint=em.footprint_estimate(r["energy_gev"]),
                              axis=em.shower_axis(air, tuple(r["start_m"]), tuple(r["direction"])),
                              radio_observers=r["observers"]) for k, r in enumerate(stream)]
        return s
    if kind == "handoff":
        air, prop = em.Atmosphere(), _air_propagation(113000.0)
        observers = workloads.star_observers(arms=case["arms"], radii=case["radii"], sample_rate_hz=2.0e9,
                                             number_of_bins=case["bins"])
        workloads.plane_front_windows(observers, START, DOWN)
        s["config"], s["backend"] = _backend(
            seed, airtables, _air_tables(), air, START, DOWN, queue_capacity=1 << 21, observation_capacity=1 << 16,
            fallback_capacity=1 << 10, moliere=True, moliere_table=True)
        s["stepper"] = em.ScalarStepper(s["config"], _air_tables(), air)
        s["cascade"] = em.HybridCascade(s["backend"], s["stepper"])
        s["accumulator"] = c8mi.RadioAccumulator(observers, prop)
        s["backend"].attach_radio(s["accumulator"])
        s["cascade"].attach_radio(s["accumulator"])
        s["primary"] = em.particle(case["pid"], case["energy"], START, DOWN, history_id=1)
        return s
    e0 = case["energy"]
    ice = em.IceVolume()
    s["config"], s["backend"] = _backend(
        seed, airtables.IceMedium, _ice_tables(), ice, ICE_START, DOWN, cut_mev=0.1, thinning=(1.0e-6 * e0, 1.0e4),
        moliere=True, moliere_table=True, bins=256, queue_capacity=1 << 22, observation_capacity=1 << 10,
        fallback_capacity=1 << 14)
    depth = 36.08 / 0.92 / 100.0 * math.log(e0 * 1.0e3 / 78.0)
    observers = workloads.cherenkov_ring_observers(np.array(ICE_START) + depth * np.array(DOWN), DOWN, 1000.0, N_ICE,
                                                   count=case["antennas"], sample_rate_hz=1.0e10,
                                                   number_of_bins=case["bins"], emission_time_s=depth / C,
                                                   pretrigger_s=min(100e-9, 0.25 * case["bins"] / 1.0e10))
    s["accumulator"] = c8mi.RadioAccumulator(observers, c8mi.Propagation(homogeneous_index=N_ICE), coreas=False, zhs=True)
    s["backend"].attach_radio(s["accumulator"])
    s["primary"] = em.particle(11, e0, ICE_START, DOWN, history_id=1)
    return s


def _whole(values):
    out = []
    for v in values:
        out += list(v) if isinstance(v, (list, tuple)) else [v]
    return np.array(out, dtype=np.int64)


def _ledger(ledger):
    terms = [ledger[k] for k in em.LEDGER_ENERGY_TERMS]
    counts = [v for k, v in sorted(ledger.items()) if k not in em.LEDGER_ENERGY_TERMS]
    return np.array(terms), _whole(counts)


def _profile(handle):
    hist, ledger = handle.download_profile()
    terms, counts = _ledger(ledger)
    return {**hist, "ledger": terms, "counts": counts}


def _served(results, totals):
    """The results of a served list: every shower's ledger and counts."""
    rows = [r for r in results]
    ledgers = [_ledger(r["ledger"]) for r in rows]
    keys = ("photon_steps", "lepton_steps", "photon_interactions", "lepton_interactions", "secondaries",
            "next_history_id", "observations", "fallbacks")
    out = {"ledgers": np.stack([a for a, _ in ledgers]), "ledger_counts": np.stack([b for _, b in ledgers]),
           "showers": np.array([[r[k] for k in keys] for r in rows], dtype=np.int64),
           "totals": _whole([totals["photon_steps"], totals["lepton_steps"], totals["secondaries"]])}
    if "radio" in rows[0]:
        # raw fixed-point sums (2^62 over the limit of 1 V/m; ZHS times the sample rate)
        out["coreas"] = np.stack([r["radio"][0] for r in rows]) * 2.0 ** -62
        out["zhs"] = np.stack([r["radio"][1] for r in rows]) * (2.0 ** -62 / 2.0e9)
    return out


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "radio":
        modes = {"both": 3, "coreas": 1, "zhs": 2}[case["mode"]]
        if case["api"] == "noalloc":
            c, z = s["buffers"]
            c8mi.radio_project_fixed_noalloc(s["observers"], s["propagation"], s["tracks"].data_ptr(), case["tracks"],
                                             case["tracks"], c.data_ptr() if modes & 1 else None,
                                             z.data_ptr() if modes & 2 else None, coreas=bool(modes & 1),
                                             zhs=bool(modes & 2), zhs_refinement=case["refinement"],
                                             exact=case["exact"])
            out = {}
            if modes & 1:
                out["coreas"] = c * 2.0 ** -62
            if modes & 2:
                out["zhs"] = z * (2.0 ** -62 / case["rate"])
            return out
        acc = s["accumulator"]
        acc.reset()
        if case["api"] == "records":
            acc.enqueue_host_tracks(s["records"])
        else:
            acc.accumulate_tracks(s["tracks"].data_ptr(), case["tracks"], case["tracks"])
        coreas, zhs, _ = acc.download()
        return {k: v for k, v in (("coreas", coreas), ("zhs", zhs)) if v is not None}
    if kind == "shower":
        dev = s["backend"]
        dev.begin_shower(7, 2)
        dev.enqueue(s["primary"])
        totals = dev.run()
        return {**_profile(dev), "totals": _whole(totals.values())}
    if kind == "pool":
        requests = [dict(r) for r in s["requests"]]
        primaries = np.concatenate([r["primary"].reshape(1) for r in requests])
        batches, next_ids, _, _ = em.hybrid_prefixes(s["config"], _air_tables(), s["config"].atmosphere, primaries,
                                                     [r["shower_id"] for r in requests], threads=8,
                                                     hybrid=em.hybrid_config(minimum_batch=16384))
        for r, b, h in zip(requests, batches, next_ids):
            r["particles"], r["first_history_id"] = b, h
        return _served(*s["backend"].serve(requests, 0.4 * (1 << 22), realtime=False))
    if kind == "stream":
        return _served(*s["backend"].serve(s["requests"], 0.4 * (1 << 22), realtime=False))
    acc, dev = s["accumulator"], s["backend"]
    acc.reset()
    if kind == "handoff":
        totals = s["cascade"].run(s["primary"], 7, 2)
        out = {"totals": _whole(v for k, v in totals.items() if not k.endswith("seconds")),
               "host": _profile(s["stepper"])}
    else:
        dev.begin_shower(7, 2)
        dev.enqueue(s["primary"])
        out = {"totals": _whole(dev.run().values())}
    coreas, zhs, _ = acc.download()
    out.update(_profile(dev), zhs=zhs)
    if coreas is not None:
        out["coreas"] = coreas
    return out


# ---- costs and tolerances ----------------------------------------------------------------

STEPS_PER_GEV = 1070.0  # air showers at the 1 MeV cut
ICE_STEPS_PER_GEV = 7300.0  # in ice at the 100 keV cut, unthinned
OPS = {"coreas": 130.0, "zhs": 155.0}  # operations of one track on one antenna


def _steps(case):
    if case["kind"] == "pool":
        return STEPS_PER_GEV * case["energy"] * case["showers"]
    if case["kind"] == "stream":
        mean = (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
        return STEPS_PER_GEV * mean * case["requests"]
    if case["kind"] == "ice":
        return ICE_STEPS_PER_GEV * case["energy"] * 0.35  # the thinned share
    thinned = 0.25 if case.get("thinning") else 1.0
    return STEPS_PER_GEV * case["energy"] * thinned


def work(case):
    """A particle-step reads and writes a 120-byte state and takes about 300 operations of
    table queries, transport and scattering; a track's 72 bytes are read once and every
    waveform bin is written once; an update takes the operations of its formula."""
    kind = case["kind"]
    if kind == "radio":
        modes = ("coreas", "zhs") if case["mode"] == "both" else (case["mode"],)
        record = 752 if case["api"] == "records" else 72
        flops = sum(OPS[m] * (case["refinement"] if m == "zhs" else 1) for m in modes)
        return {"bytes": record * case["tracks"] + 24.0 * len(modes) * case["antennas"] * case["bins"],
                "flops": flops * case["tracks"] * case["antennas"]}
    steps = _steps(case)
    out = {"bytes": 240.0 * steps, "flops": 300.0 * steps}
    if kind in ("stream", "handoff", "ice"):
        antennas = case["antennas"] if kind == "ice" else case["arms"] * case["radii"]
        modes = ("zhs",) if kind == "ice" else ("coreas", "zhs")
        showers = case["requests"] if kind == "stream" else 1
        out["bytes"] += 72.0 * 0.9 * steps + 24.0 * len(modes) * antennas * case["bins"] * showers
        out["flops"] += sum(OPS[m] for m in modes) * 0.9 * steps * antennas
    return out


def tolerance(case):
    """EM: FP64 steps whose last-bit differences (another libm) travel through the shower, the
    parity bar of the tests (1e-9 of the primary's energy). Radio: FP64 with an int64
    fixed-point sum; an arrival time that rounds to the neighbouring bin moves one
    contribution, which is what the largest difference allows for."""
    if case["kind"] == "radio":
        return {"rel": 2e-4, "max": 0.5}
    if case["kind"] in ("shower", "pool"):
        return {"rel": 1e-8, "max": 1e-4, "differ": 0.0}
    return {"rel": 1e-4, "max": 0.5, "differ": 0.0}


# ---- the projection in plain FP64 -----------------------------------------------------

K_CHARGE = 1.6021766208e-19 / (4.0 * math.pi * 8.8541878128e-12 * C)


def _dot(a, b):
    return (a * b).sum(0)


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=0)


def _path(source, position, medium):
    """Straight path: (travel time, index at the source, index at the antenna, distance, direction)."""
    disp = position[:, None] - source
    r = disp.square().sum(0).sqrt()
    direction = disp / r
    if medium is None:
        n = torch.full_like(r, N_ICE)
        return N_ICE * r / C, n, N_ICE, r, direction
    refractivity, integrated, low = medium
    at = (source[2] - low + 0.5).floor().long()
    here = int(math.floor(float(position[2]) - low + 0.5))
    height = (at - here).double()
    height = torch.where(height == 0, torch.ones_like(height), height)
    mean = 1.0 + (integrated[at] - integrated[here]) / height
    return mean * r / C, 1.0 + refractivity[at], 1.0 + float(refractivity[here]), r, direction


def _nearest(x):
    return (x + 0.5).floor()


def _add(wave, bins, values, keep):
    """Adds values [3][n] to the bins [n] of wave [3][bins] where `keep`, as sorted segment sums."""
    n = wave.shape[1]
    at = torch.where(keep & (bins >= 0) & (bins < n), bins, torch.full_like(bins, float(n))).long()
    order = torch.argsort(at)
    sums = torch.cumsum(values[:, order], 1)
    sums = torch.cat([torch.zeros(3, 1, dtype=sums.dtype, device=sums.device), sums], 1)
    edges = torch.searchsorted(at[order], torch.arange(n + 1, device=at.device))
    wave += sums[:, edges[1:]] - sums[:, edges[:-1]]


def _separate(start, end, grid, which, signed):
    """Endpoints that fall into one bin move apart by one bin."""
    s, e = start / grid, end / grid
    which = which & (_nearest(s) == _nearest(e))
    sf, ef = s - s.floor(), e - e.floor()
    forward = (end >= start) if signed else torch.ones_like(which)
    both_high, both_low = (sf >= 0.5) & (ef >= 0.5), (sf < 0.5) & (ef < 0.5)
    ahead = both_low | (~both_high & torch.where(forward, ef >= 1.0 - sf, sf >= 1.0 - ef))
    start = torch.where(which & forward & ~ahead, start - grid, torch.where(which & ~forward & ahead, start + grid, start))
    end = torch.where(which & forward & ahead, end + grid, torch.where(which & ~forward & ~ahead, end - grid, end))
    return start, end


def _coreas(t, o, medium, wave):
    rate, grid = o["rate"], 1.0 / o["rate"]
    ts, ns, nd, rs, es = _path(t["start"], o["position"], medium)
    te, ne, _, re, ee = _path(t["end"], o["position"], medium)
    tm, nm, _, rm, emid = _path(0.5 * (t["start"] + t["end"]), o["position"], medium)
    beta = t["beta"]
    pre, post, mid = 1.0 - ns * _dot(beta, es), 1.0 - ne * _dot(beta, ee), 1.0 - nm * _dot(beta, emid)
    a, b = t["t0"] + ts, t["t1"] + te
    near = ((pre.abs() < 1e-3) | (post.abs() < 1e-3)) & (nd > 1.0)
    q = t["constant"] * rate
    fs = _cross(es, _cross(es, beta)) * (q / (pre * rs))
    fe = -_cross(ee, _cross(ee, beta)) * (q / (post * re))
    fm = _cross(emid, _cross(emid, beta)) * (q / (mid * rm))
    spread = t["duration"] * mid.abs()
    middle = 0.5 * (t["t0"] + t["t1"]) + tm
    side = torch.where(a < b, 1.0, -1.0)
    na, nb = middle - 0.5 * side * spread, middle + 0.5 * side * spread
    for low, x, y, f, g, signed in ((near, na, nb, fm, -fm, True), (~near, a, b, fs, fe, False)):
        delta = y - x
        close = low & (delta.abs() < grid)
        if not signed:
            close = close & ((pre < 1e-9) | (post < 1e-9))
        shrink = torch.where(close, delta.abs() / grid, torch.ones_like(delta))
        x, y = _separate(x, y, grid, close, signed)
        for time, field in ((x, f * shrink), (y, g * shrink)):
            inside = low & t["valid"] & (time >= o["begin"]) & (time <= o["begin"] + o["duration"])
            _add(wave, _nearest((time - o["begin"]) * rate), field, inside)


def _zhs(t, o, medium, wave, refinement):
    rate = o["rate"]
    n = wave.shape[1]
    _, _, _, rm, emid = _path(0.5 * (t["start"] + t["end"]), o["position"], medium)
    u = _dot(t["beta"], emid) / t["beta_module"]
    far = (1.0 - u * u) * t["length"].square() / rm * rate / C * 2.0 * math.pi
    divisor = torch.where(far > 1.0, far.clamp(min=0.0).sqrt() + 1.0, torch.ones_like(far))
    parts = torch.where(far > 1.0, divisor.ceil(), torch.ones_like(far)) * refinement
    step, dt = t["disp"] / (divisor * refinement), t["duration"] / (divisor * refinement)
    steps = torch.zeros(3, n + 1, dtype=wave.dtype, device=wave.device)
    p1, t1 = t["start"], t["t0"]
    for i in range(int(parts.max())):
        live = t["valid"] & (i < parts)
        p2, t2 = p1 + step, t1 + dt
        travel, index, _, r, e = _path(0.5 * (p1 + p2), o["position"], medium)
        bk = index * _dot(t["beta"], e)
        middle = 0.5 * (t1 + t2)
        d1, d2 = t1 + travel - bk * (t1 - middle), t2 + travel - bk * (t2 - middle)
        swap = d1 > d2
        d1, d2 = torch.where(swap, d2, d1), torch.where(swap, d1, d2)
        sign = torch.where(swap, -1.0, 1.0)
        x1, x2 = (d1 - o["begin"]) * rate, (d2 - o["begin"]) * rate
        b1, b2 = _nearest(x1), _nearest(x2)
        den = 1.0 - bk
        perp = _cross(e, _cross(t["beta"], e)) * (t["constant"] / r)
        one = b1 == b2
        flat = den.abs() <= 1e-15
        k = torch.where(flat, torch.ones_like(den), 1.0 / torch.where(flat, torch.ones_like(den), den))
        single = torch.where(flat, (t2 - t1) * rate, k * (d2 * rate - d1 * rate).abs())
        _add(wave, b2, perp * (sign * single), live & one)
        _add(wave, b1, perp * (sign * k * (b1 + 0.5 - x1).abs()), live & ~one)
        _add(wave, b2, perp * (sign * k * (x2 + 0.5 - b2).abs()), live & ~one)
        many = live & (b2 - b1 > 1.0)
        inner = perp * (torch.where(parts > 1, torch.ones_like(sign), sign) * k)
        first, last = (b1 + 1.0).clamp(0, n), b2.clamp(0, n)  # bins [first, last)
        some = many & (first < last)
        _add(steps, first, inner, some)
        _add(steps, last, -inner, some)
        p1, t1 = p2, t2
    wave += torch.cumsum(steps, 1)[:, :n]


def exact(case, seed):
    """The projection with CoREAS' and ZHS' formulas in FP64; none for the showers."""
    if case["kind"] != "radio":
        return None
    tracks, observers, prop = _radio_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["tracks"] * case["antennas"] > (2e8 if dev == "cuda" else 3e6):
        return None
    x = torch.from_numpy(tracks).to(dev)
    t = {"start": x[0:3], "end": x[3:6], "t0": x[6], "t1": x[7], "constant": K_CHARGE * x[8]}
    t["disp"], t["duration"] = t["end"] - t["start"], t["t1"] - t["t0"]
    t["length"] = t["disp"].square().sum(0).sqrt()
    t["beta"] = t["disp"] / (C * t["duration"])
    t["beta_module"] = t["length"] / (C * t["duration"])
    t["valid"] = (t["duration"] > 0) & (t["length"] > 0)
    medium = None
    if prop.refractivity is not None:
        medium = (torch.from_numpy(prop.refractivity).to(dev), torch.from_numpy(prop.integrated).to(dev),
                  float(prop.struct.minimum_height_m))
    out = {m: torch.zeros(case["antennas"], 3, case["bins"], dtype=torch.float64, device=dev)
           for m in ("coreas", "zhs") if case["mode"] in (m, "both")}
    for k, o in enumerate(observers):
        view = {"position": torch.tensor(o["position_m"], dtype=torch.float64, device=dev), "rate": float(o["sample_rate_hz"]),
                "begin": float(o["start_time_s"]), "duration": float(o["duration_s"])}
        if "coreas" in out:
            _coreas(t, view, medium, out["coreas"][k])
        if "zhs" in out:
            _zhs(t, view, medium, out["zhs"][k], case["refinement"])
    return {m: w.transpose(0, 1).reshape(3, -1).contiguous() for m, w in out.items()}
