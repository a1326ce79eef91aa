"""Front sizes at which the kernels of a front change, against the oracle's showers:
fronts of up to 1024 sources are compacted by one workgroup (edges of a wave and of the
workgroup, and of the several kernels above), fronts of up to 131072 e+- run the Moliere
tail in line and finish and vertices in one kernel. Counts, history IDs and ledger counts
are identical; energies and profile bins within 1e-9 of the primary energy (the bar of the
other shower tests).
"""
import numpy as np
import pytest

from c8mi import airtables, em
from test_em_gpu import STAT_KEYS, compare, run_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tables():
    return airtables.build_air_tables()


def batch(count, seed):
    """`count` low-energy particles 500 m above the ground, two in three of them e+-."""
    rng = np.random.default_rng(seed)
    out = np.zeros(count, dtype=em.PARTICLE_STATE_DTYPE)
    for k in range(count):
        pid = (11, -11, 22)[k % 3]
        tilt = rng.normal(0.0, 0.2, 2)
        d = np.array([tilt[0], tilt[1], -1.0])
        out[k] = em.particle(pid, float(rng.uniform(0.002, 0.03)), (rng.normal(0, 50.0), rng.normal(0, 50.0), 500.0),
                             d / np.linalg.norm(d), history_id=k + 1)
    return out


@pytest.mark.parametrize("lepton_count,table", [(1, True), (64, True), (65, True), (255, True), (1023, True), (1024, True),
                                                (1025, True), (1025, None), (8192, True), (8193, None)])
def test_front_sizes(tables, lepton_count, table):
    count = lepton_count * 3 // 2 + (1 if lepton_count * 3 % 2 else 0)
    prim = batch(count, lepton_count)
    leptons = int((prim["pid"] != 22).sum())
    assert abs(leptons - lepton_count) <= 1
    cfg, want, got = run_pair(tables, 0, 0, 3, primaries=prim, start=(0.0, 0.0, 500.0), moliere=True, moliere_table=table)
    assert got["stats"]["max_front"] >= leptons
    compare(cfg, want, got, float(prim["energy_gev"].sum()))


@pytest.mark.parametrize("lepton_count", [131072, 131074])
def test_finish_and_vertices_in_one_kernel_and_in_two(tables, lepton_count):
    """Counts only: over millions of steps an ulp of the device's exp or log that adds or
    saves a Moliere iteration (converged to 5e-5) moves an angle by up to 2.5e-9."""
    prim = batch(lepton_count * 3 // 2, lepton_count)
    assert int((prim["pid"] != 22).sum()) == lepton_count
    cfg, want, got = run_pair(tables, 0, 0, 3, primaries=prim, start=(0.0, 0.0, 500.0), moliere=True, moliere_table=True)
    for k in STAT_KEYS:
        assert got["stats"][k] == want["stats"][k], k
    ledger = em.decode_counters(want["counters"], cfg.struct.profile_energy_scale)
    for k in ("steps", "photon_cuts", "lepton_limits", "deposited_steps", "invalid_records", "fallback_reasons"):
        assert got["ledger"][k] == ledger[k], k


@pytest.mark.parametrize("count", [511, 512, 1024, 1025])
def test_photon_front_sizes(tables, count):
    prim = batch(count, 7 + count)
    prim["pid"] = 22
    cfg, want, got = run_pair(tables, 0, 0, 4, primaries=prim, start=(0.0, 0.0, 500.0))
    compare(cfg, want, got, float(prim["energy_gev"].sum()))
