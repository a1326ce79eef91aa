"""Fixed-point sums of many large contributions that cancel: what is refused is a waveform
out of range, whatever the launch's shape.

Every track comes twice, with opposite charge, and 64 more come once: increments of a track
and of its mirror image are negatives of each other (rounding to nearest even is symmetric),
so the waveforms equal, bit for bit, those of the 64 alone, and no overflow is reported. The
sum of |increments| of an observer is `share` times 2^62, so that a workgroup's (up to eight
observers) passes 2^63, a thread's its limit for the tile (2^51), a bin its own (2^60) and a
range of bins its share (2^62).
"""
import numpy as np
import pytest

import oracle_lib
from radio_cases import random_tracks, window_observers
from test_radio_gpu import exponential_table, gpu_project

pytestmark = pytest.mark.gpu

PAIRS = 4096


def sum_of_magnitudes(tracks, obs, prop, refinement):
    """Largest of the observers' and algorithms' sums of |contribution|, in field units."""
    begin = np.concatenate([[0], np.cumsum(obs["number_of_bins"].astype(np.int64))])[:-1]
    total = np.zeros((2, obs.size))
    for k in range(tracks.shape[1]):
        ref = oracle_lib.radio_project(prop, obs, tracks[:, k:k + 1], refinement=refinement)
        total[0] += np.add.reduceat(np.abs(ref["coreas_float"]).sum(0), begin)
        total[1] += np.add.reduceat(np.abs(ref["zhs_float"]).sum(0), begin) * obs["sample_rate_hz"]
    return total.max()


@pytest.fixture(scope="module", params=[(1.0, 1), (12.0, 2)], ids=["short", "long_refined"])
def lists(request):
    """(tracks, the uncancelled 64, observers, propagation, sum of |contribution|, refinement)"""
    stretch, refinement = request.param
    base = random_tracks(64, 17, height=(400.0, 1500.0))
    base[3:6] += (stretch - 1.0) * (base[3:6] - base[0:3])
    base[7] += (stretch - 1.0) * (base[7] - base[6])
    rng = np.random.default_rng(3)
    positions = [tuple(p) for p in np.stack([rng.uniform(-80, 80, 40), rng.uniform(-80, 80, 40), rng.uniform(0, 30, 40)], 1)]
    obs = window_observers(base, positions, 1.0e9, 200)
    prop = exponential_table()
    twice = np.tile(np.repeat(base, 2, axis=1), (1, PAIRS // 64))
    twice[8, 1::2] *= -1.0
    total = sum_of_magnitudes(base, obs, prop, refinement) * twice.shape[1] / 64
    return np.concatenate([twice, base], axis=1), base, obs, prop, total, refinement


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("share", [0.05, 3.0, 12.0, 60.0])
@pytest.mark.parametrize("tuning", [None, dict(block_threads=256), dict(tile_bins=70, chunk_tracks=8192, block_threads=1024)],
                         ids=["automatic", "one_observer", "tiles"])
def test_cancelling_contributions(lists, exact, share, tuning):
    tracks, base, obs, prop, total, refinement = lists
    limit = total / share
    print(f"limit {limit:.3e}", flush=True)
    want = gpu_project(base, obs, prop, refinement=refinement, exact=exact, limit=limit)
    got = gpu_project(tracks, obs, prop, refinement=refinement, exact=exact, limit=limit, tuning=tuning)
    assert want[2]["fixed_point_overflows"] == got[2]["fixed_point_overflows"] == 0
    assert np.abs(want[0]).max() > 2 ** 40 and np.abs(want[1]).max() > 2 ** 40
    assert np.array_equal(got[0], want[0])
    assert np.array_equal(got[1], want[1])
    n = 2 * PAIRS // 64 + 1
    for k in ("coreas_contributions", "zhs_contributions", "zhs_subtracks", "valid_tracks"):
        assert got[2][k] == n * want[2][k], k


@pytest.mark.parametrize("exact", [False, True])
def test_sums_out_of_range_are_refused(lists, exact):
    """Without the mirror images the waveforms pass 2^63."""
    tracks, base, obs, prop, total, refinement = lists
    same = np.tile(base, (1, 2 * PAIRS // 64))
    got = gpu_project(same, obs, prop, refinement=refinement, exact=exact, limit=total / 3000.0)
    assert got[2]["fixed_point_overflows"] > 0
