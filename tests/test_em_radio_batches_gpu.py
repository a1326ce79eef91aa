"""Radio of showers whose e+- tracks fill several batches of the attached accumulator (2^20
tracks each; the two buffers take turns), against per-shower radio, which projects every
front by itself: the increments of a track don't depend on the launch, and integers add up in
any order, so the waveforms are equal bit for bit.
"""
import time

import numpy as np
import pytest

import c8mi
from c8mi import airtables, em, workloads
from test_em_front_edges_gpu import batch
from test_em_radio_gpu import DOWN, START, propagation

pytestmark = pytest.mark.gpu

BATCH = 1 << 20
COUNTERS = ("valid_tracks", "coreas_contributions", "zhs_contributions", "zhs_subtracks", "fixed_point_overflows")


@pytest.fixture(scope="module")
def tables():
    return airtables.build_air_tables()


def antennas(start, bins=512):
    observers = workloads.star_observers(arms=3, radii=3, sample_rate_hz=5.0e8, number_of_bins=bins)
    workloads.plane_front_windows(observers, start, DOWN)
    return observers


def electrons(count):
    """`count` electrons of 2 to 30 MeV, 500 m above the ground."""
    prim = np.tile(batch(3072, 5), -(-count // 3072))[:count].copy()
    prim["pid"] = np.where(np.arange(count) % 2, 11, -11)
    prim["energy_gev"] = np.random.default_rng(9).uniform(0.002, 0.03, count)
    prim["history_id"] = np.arange(1, count + 1)
    return prim


def attached(cfg, tables, atm, observers, prop, showers, exact, between=lambda radio, k: None):
    """One accumulator for all showers; `between` is called after each of them."""
    dev = em.EmBackend(cfg, tables, atm)
    radio = c8mi.RadioAccumulator(observers, prop, exact=exact)
    dev.attach_radio(radio)
    steps, fronts = [], []
    for k, (shower_id, prim) in enumerate(showers):
        dev.begin_shower(shower_id, int(np.max(np.atleast_1d(prim["history_id"]))) + 1)
        dev.enqueue(prim)
        totals = dev.run()
        steps.append(totals["lepton_steps"])
        fronts.append(totals["max_front"])
        between(radio, k)
    got = radio.download_fixed()
    dev.close()
    radio.close()
    return got, steps, fronts


def front_by_front(cfg, tables, atm, observers, prop, showers, exact):
    total = None
    dev = em.EmBackend(cfg, tables, atm)
    dev.enable_slot_radio(observers.size, int(observers["number_of_bins"].max()), prop, exact=exact)
    for shower_id, prim in showers:
        dev.slot_begin(0, shower_id, int(np.max(np.atleast_1d(prim["history_id"]))) + 1)
        dev.slot_set_radio(0, observers)
        dev.slot_enqueue(0, prim)
        dev.run_rounds(1 << 20)
        c, z, n = dev.slot_download_radio(0)
        n = np.array([n[k] for k in COUNTERS])
        total = [c, z, n] if total is None else [total[0] + c, total[1] + z, total[2] + n]
        dev.slot_end(0)
    dev.close()
    return total


def assert_equal(got, want):
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    assert [got[2][k] for k in COUNTERS] == want[2].tolist()
    assert want[2][0] > 0 and want[0].any() and want[1].any()


@pytest.mark.parametrize("exact", [False, True])
def test_many_batches(tables, exact):
    """A 10 TeV shower: the buffers are reused while the other is projected."""
    atm = em.Atmosphere()
    cfg = em.make_config(airtables, seed=3, atmosphere=atm, queue_capacity=1 << 21, moliere=True, moliere_table=True)
    showers = [(5, em.particle(11, 1.0e4, START, DOWN, history_id=1))]
    observers, prop = antennas(START), propagation()
    print("10 TeV attached", flush=True)
    got, steps, _ = attached(cfg, tables, atm, observers, prop, showers, exact)
    assert steps[0] > 3 * BATCH
    print("10 TeV front by front", flush=True)
    assert_equal(got, front_by_front(cfg, tables, atm, observers, prop, showers, exact))


def test_front_larger_than_a_batch(tables):
    """Fronts of 1.2e6 e+-: a started batch is projected, the next buffer grows."""
    atm = em.Atmosphere()
    start = (0.0, 0.0, 500.0)
    cfg = em.make_config(airtables, seed=4, atmosphere=atm, start=start, queue_capacity=1 << 22, moliere=True, moliere_table=True)
    showers = [(6, electrons(3000)), (7, electrons(1200000))]
    observers, prop = antennas(start), propagation()
    print("large front attached", flush=True)
    got, steps, fronts = attached(cfg, tables, atm, observers, prop, showers, False)
    assert steps[0] > 3000 and fronts[1] > BATCH
    print("large front front by front", flush=True)
    assert_equal(got, front_by_front(cfg, tables, atm, observers, prop, showers, False))


def test_reset_drops_tracks_not_projected_yet(tables):
    atm = em.Atmosphere()
    cfg = em.make_config(airtables, seed=5, atmosphere=atm, moliere=True, moliere_table=True)
    showers = [(8, em.particle(11, 5.0, START, DOWN, history_id=1)), (9, em.particle(22, 4.0, START, DOWN, history_id=1))]
    observers, prop = antennas(START), propagation()

    def between(radio, k):
        if k == 0:
            radio.reset()

    got, steps, _ = attached(cfg, tables, atm, observers, prop, showers, False, between)
    assert steps[0] > 100
    assert_equal(got, front_by_front(cfg, tables, atm, observers, prop, showers[1:], False))


def test_tuning_after_the_tracks(tables):
    """Knobs set after a run hold for later tracks: a shape that the tracks of the run together
    would be too many for (2^32 workgroups) neither refuses nor loses them."""
    atm = em.Atmosphere()
    cfg = em.make_config(airtables, seed=6, atmosphere=atm, moliere=True, moliere_table=True)
    prim = em.particle(22, 1000.0, START, DOWN, history_id=1)
    observers = antennas(START, 131072)
    observers = np.concatenate([observers] * 4)[:32]
    prop = propagation()
    downloads = []
    for tuned in (False, True):
        dev = em.EmBackend(cfg, tables, atm)
        radio = c8mi.RadioAccumulator(observers, prop, zhs=False)
        dev.attach_radio(radio)
        dev.begin_shower(10, 2)
        dev.enqueue(prim)
        steps = dev.run()["lepton_steps"]
        if tuned:
            assert -(-steps // 256) * observers.size * 131072 > 1 << 32
            radio.set_tuning(chunk_tracks=256, tile_bins=1)
        downloads.append(radio.download_fixed())
        dev.close()
        radio.close()
    assert downloads[0][2]["valid_tracks"] > 0 and downloads[0][0].any()
    assert downloads[0][2] == downloads[1][2]
    assert np.array_equal(downloads[0][0], downloads[1][0])


@pytest.mark.parametrize("call", ["run", "run_lepton_wavefront"])
def test_a_run_projects_its_tracks(tables, call):
    """The download reads waveforms back; the projection (here many times longer than that,
    64 segments a track) belongs to the run."""
    atm = em.Atmosphere()
    cfg = em.make_config(airtables, seed=7, atmosphere=atm, moliere=True, moliere_table=True)
    observers, prop = np.concatenate([antennas(START, 128)] * 18)[:160], propagation()
    dev = em.EmBackend(cfg, tables, atm)
    radio = c8mi.RadioAccumulator(observers, prop, coreas=False, zhs_refinement=64, exact=True)
    radio.enable_kernel_timing(True)
    dev.attach_radio(radio)
    if call == "run":
        dev.begin_shower(11, 2)
        dev.enqueue(em.particle(11, 100.0, START, DOWN, history_id=1))
        dev.run()
    else:
        prim = electrons(3000)
        prim["position_m"] = START
        dev.begin_shower(11, 3001)
        dev.run_lepton_wavefront(prim, 3001, 1 << 40, maximum_wavefronts=2)
    time.sleep(1.0)
    begin = time.perf_counter()
    _, _, counters = radio.download_fixed()
    seconds = time.perf_counter() - begin
    ms, launches = radio.kernel_time()["zhs"]
    dev.close()
    radio.close()
    print(f"{call}: {counters['valid_tracks']} tracks, projection {ms:.1f} ms, download {1e3 * seconds:.2f} ms", flush=True)
    assert counters["valid_tracks"] > 2000 and ms > 10.0
    assert 1e3 * seconds < 0.5 * ms
