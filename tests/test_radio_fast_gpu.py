"""The fast radio projection at the edges of its workgroups, waves, tiles and lists
against the FP64 oracle.

Track counts around a wave (64), a workgroup (512) and their remainders; tracks that all
take CoREAS's Cherenkov form (a wave lists them and runs 64 at a time), none, or a mix;
window tiles that cut segments of several bins; sources above, below and on the ends of
the propagation table; groups of observers and their remainders. The bar is the fast
form's: per observer a relative L2 error of 1e-6 (FP64 rounding of about ten operations per
sample is 1e-14 relative, 1e-11 near the Cherenkov angle, where 1 - n b.e >= 1e-9 cancels),
with a field limit of 1e-6 V/m, so that the int64 quantum (2^-62 of the limit per sample)
is below 1e-9 of the smallest field here. Counters equal the oracle's.
"""
import numpy as np
import pytest

import c8mi
import oracle_lib
from c8mi import workloads
from radio_cases import C, random_tracks, uniform_table, window_observers
from test_radio_gpu import POSITIONS, exponential_table, gpu_project

pytestmark = pytest.mark.gpu


LIMIT = 1.0e-6


def assert_close(tracks, obs, prop, refinement=1, tuning=None):
    ref = oracle_lib.radio_project(prop, obs, tracks, refinement=refinement, limit=LIMIT, threads=4)
    got = gpu_project(tracks, obs, prop, refinement=refinement, exact=False, limit=LIMIT, tuning=tuning)
    offsets = np.concatenate([[0], np.cumsum(obs["number_of_bins"].astype(np.int64))])
    for fixed, name in ((got[0], "coreas"), (got[1], "zhs")):
        field = oracle_lib.radio_decode(fixed, obs, limit=LIMIT, potential=name == "zhs")
        for k in range(obs.size):
            want = ref[name + "_float"][:, offsets[k]:offsets[k + 1]]
            error = np.linalg.norm(field[:, offsets[k]:offsets[k + 1]] - want)
            assert error <= 1e-6 * np.linalg.norm(want), (name, k)
    assert got[2] == ref["counters"]
    return ref["counters"]


def near_tracks(count, seed):
    """Tracks whose direction points at the antennas at beta ~ 1: small Doppler factors."""
    rng = np.random.default_rng(seed)
    tracks = random_tracks(count, seed, box=1.0, height=(900.0, 1400.0))
    length = rng.uniform(0.5, 3.0, count)
    tracks[3:6] = tracks[0:3] + np.stack([np.zeros(count), np.zeros(count), -length])
    tracks[7] = tracks[6] + length / (C * rng.uniform(0.9995, 1.0, count))
    return tracks


def mixed(count, seed, share):
    tracks = random_tracks(count, seed)
    near = np.random.default_rng(seed + 1).random(count) < share
    tracks[:, near] = near_tracks(count, seed + 2)[:, near]
    return tracks


@pytest.mark.parametrize("count", [1, 63, 64, 65, 511, 512, 513, 1300])
@pytest.mark.parametrize("share", [0.0, 0.4, 1.0])
def test_counts_and_cherenkov_lists(count, share):
    tracks = mixed(count, 11 + count, share)
    obs = window_observers(tracks, POSITIONS[:5], 2.0e9, 1024)
    for prop in (exponential_table(), c8mi.Propagation(homogeneous_index=1.0003)):
        assert_close(tracks, obs, prop)


@pytest.mark.parametrize("tile", [0, 5, 64, 333])
@pytest.mark.parametrize("refinement", [1, 3])
def test_segments_across_window_tiles(tile, refinement):
    tracks = mixed(700, 5, 0.2)
    tracks[3:6] += 3.0 * (tracks[3:6] - tracks[0:3])  # segments of several bins
    tracks[7] += 3.0 * (tracks[7] - tracks[6])
    obs = window_observers(tracks, POSITIONS[:4], 1.0e9, 120)
    prop = uniform_table(1.0003, upper=4000.0)
    tuning = dict(tile_bins=tile, chunk_tracks=512, block_threads=512) if tile else None
    counters = assert_close(tracks, obs, prop, refinement, tuning)
    assert counters["zhs_contributions"] > 1.5 * counters["zhs_subtracks"]


def test_sources_outside_the_table():
    tracks = random_tracks(600, 21, height=(-40.0, 300.0))
    tracks[2, :5] = tracks[5, :5] = 200.0  # the last table height
    tracks[2, 5:10] = 0.0  # the first
    obs = window_observers(tracks, ((3., 4., 50.), (-20., 60., 120.)), 2.0e9, 2048)
    prop = uniform_table(1.0003, lower=0.0, upper=200.0)
    assert_close(tracks, obs, prop)


def test_large_increments():
    """Components beyond 2^51 in fixed point take the rounding form."""
    tracks = mixed(200, 3, 0.3)
    obs = window_observers(tracks, POSITIONS[:3], 2.0e9, 512)
    prop = exponential_table()
    limit = 1.0e-9
    ref = oracle_lib.radio_project(prop, obs, tracks, limit=limit, threads=4)
    got = gpu_project(tracks, obs, prop, exact=False, limit=limit)
    for k, name in enumerate(("coreas", "zhs")):
        want = ref[name + "_fixed"].astype(np.float64)
        assert np.abs(want).max() > 2.0 ** 52
        assert np.linalg.norm(got[k] - want) <= 1e-6 * np.linalg.norm(want)


# The launch gives a workgroup more observers the more there are; 64-bin windows leave room
# for eight of them. Each observer has its own height, rate, bins and window here.
@pytest.mark.parametrize("observers,count", [(17, 9000), (33, 700), (65, 3001), (100, 9000), (66, 40000), (61, 40000)])
@pytest.mark.parametrize("mode", ["both", "coreas", "zhs"])
def test_groups_of_observers_and_their_remainders(observers, count, mode):
    rng = np.random.default_rng(observers)
    tracks = mixed(count, 100 + observers, 0.1)
    positions = np.stack([rng.uniform(-60, 60, observers), rng.uniform(-60, 60, observers), rng.uniform(0.0, 40.0, observers)], 1)
    obs = window_observers(tracks, [tuple(p) for p in positions], 1.0e9, 64)
    obs["sample_rate_hz"] = rng.choice((2.5e8, 5.0e8, 1.0e9), observers)
    obs["number_of_bins"] = rng.integers(2, 65, observers)
    obs["duration_s"] = (obs["number_of_bins"] - 1.0) / obs["sample_rate_hz"]
    prop = exponential_table()
    modes = dict(coreas=mode != "zhs", zhs=mode != "coreas")
    ref = oracle_lib.radio_project(prop, obs, tracks, limit=LIMIT, threads=4)
    got = gpu_project(tracks, obs, prop, exact=False, limit=LIMIT, **modes)
    ends = np.cumsum(obs["number_of_bins"].astype(np.int64))
    for fixed, name in ((got[0], "coreas"), (got[1], "zhs")):
        if not modes[name]:
            continue
        field = oracle_lib.radio_decode(fixed, obs, limit=LIMIT, potential=name == "zhs")
        want = ref[name + "_float"]
        for k, end in enumerate(ends):
            part = slice(int(end) - int(obs["number_of_bins"][k]), int(end))
            error = np.linalg.norm(field[:, part] - want[:, part])
            assert error <= 1e-6 * np.linalg.norm(want[:, part]), (name, k)
        assert got[2][name + "_contributions"] == ref["counters"][name + "_contributions"]


# Windows longer than a tile: groups of two to four observers with two or three tiles each, whose
# windows end in the first, the second or the last of them.
@pytest.mark.parametrize("observers,bins", [(40, 2500), (41, 5000), (61, 7000)])
@pytest.mark.parametrize("mode", ["coreas", "zhs"])
@pytest.mark.parametrize("index", [0.0, 1.0003])
def test_groups_of_observers_with_several_tiles(observers, bins, mode, index):
    count = 3000
    rng = np.random.default_rng(observers)
    tracks = mixed(count, 200 + observers, 0.1)
    tracks[3:6, ::5] += 20.0 * (tracks[3:6, ::5] - tracks[0:3, ::5])  # segments across tiles
    tracks[7, ::5] += 20.0 * (tracks[7, ::5] - tracks[6, ::5])
    positions = np.stack([rng.uniform(-60, 60, observers), rng.uniform(-60, 60, observers), rng.uniform(0.0, 40.0, observers)], 1)
    obs = window_observers(tracks, [tuple(p) for p in positions], 5.0e9, bins)
    obs["number_of_bins"] = rng.integers(2, bins + 1, observers)
    obs["number_of_bins"][:3] = (bins, bins // 2, bins // 3)
    obs["duration_s"] = (obs["number_of_bins"] - 1.0) / obs["sample_rate_hz"]
    prop = c8mi.Propagation(homogeneous_index=index) if index else exponential_table()
    ref = oracle_lib.radio_project(prop, obs, tracks, limit=LIMIT, threads=4)
    got = gpu_project(tracks, obs, prop, exact=False, limit=LIMIT, coreas=mode == "coreas", zhs=mode == "zhs")
    field = oracle_lib.radio_decode(got[0] if mode == "coreas" else got[1], obs, limit=LIMIT, potential=mode == "zhs")
    want = ref[mode + "_float"]
    ends = np.cumsum(obs["number_of_bins"].astype(np.int64))
    later = 0
    for k, end in enumerate(ends):
        part = slice(int(end) - int(obs["number_of_bins"][k]), int(end))
        assert np.linalg.norm(field[:, part] - want[:, part]) <= 1e-6 * np.linalg.norm(want[:, part]), k
        later += np.any(want[:, part][:, bins // 2:])
    assert later > 0
    assert got[2][mode + "_contributions"] == ref["counters"][mode + "_contributions"]


def test_arrival_times_round_as_the_oracles():
    """ZHS in ice, 1 km away: the two arrival times of a segment of 0.1 mm to 1 cm differ by 1e-16 s
    to 1e-12 s and are rounded to 8.5e-22 s each (2^-53 of 6e-6 s, half a unit), so a contribution
    carries a relative rounding of up to 1e-5. Evaluated in the oracle's order, fast times round
    as the oracle's unless the path's time, one square root apart, falls on the other side of a
    rounding boundary, and the contribution agrees to the errors of its other factors (ten operations
    of 1.1e-16, below 1e-12 over 1 - n e.b of more than 1e-3): 83.7% of the bins do. With the index
    multiplied after the division by c it was 81.5%, and 61% with a form that is equal in exact
    arithmetic only (midpoint and spread). One segment a nanosecond, so each has bins of its own."""
    count, rate = 400, 1.0e10
    obs = workloads.cherenkov_ring_observers(np.array([0.0, 0.0, -104.0]), (0.0, 0.0, -1.0), 1000.0, 1.78, count=8,
                                             sample_rate_hz=rate, number_of_bins=4096, pretrigger_s=2.0e-9)
    prop = c8mi.Propagation(homogeneous_index=1.78)
    errors = []
    for seed in (1, 2, 3):
        rng = np.random.default_rng(seed)
        tilt = rng.normal(0.0, 0.25, (2, count))
        d = np.stack([tilt[0], tilt[1], -np.ones(count)])
        d /= np.linalg.norm(d, axis=0)
        length = 10.0 ** rng.uniform(-4.0, -2.0, count)
        tracks = np.empty((9, count))
        tracks[0:3] = rng.normal(0.0, 0.003, (3, count)) + [[0.0], [0.0], [-104.0]]
        tracks[3:6] = tracks[0:3] + length * d
        tracks[6] = 1.0e-9 * np.arange(count)
        tracks[7] = tracks[6] + length / (rng.uniform(0.9, 1.0, count) * C)
        tracks[8] = np.where(rng.random(count) < 0.6, -1.0, 1.0)
        ref = oracle_lib.radio_project(prop, obs, tracks, coreas=False, threads=4)
        want = ref["zhs_float"].reshape(3, obs.size, 4096)
        limit = 1.0e3 * rate * np.abs(want).max()  # the int64 quantum is 2e-16 of the largest contribution
        got = gpu_project(tracks, obs, prop, coreas=False, exact=False, limit=limit)
        field = oracle_lib.radio_decode(got[1], obs, limit=limit, potential=True).reshape(want.shape)
        size = np.linalg.norm(want, axis=0)
        filled = size > 1e-6 * size.max()
        assert filled.sum() > 0.8 * count * obs.size
        errors.append(np.linalg.norm(field - want, axis=0)[filled] / size[filled])
    error = np.concatenate(errors)
    alike = float(np.mean(error <= 1e-12))
    print(f"{alike:.4f} of {error.size} bins alike, median error {np.median(error):.1e}, largest {error.max():.1e}", flush=True)
    assert alike > 0.828
