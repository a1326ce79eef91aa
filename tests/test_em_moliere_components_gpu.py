"""Moliere scattering in media of one to four elements (the device has a kernel for each number
of components), interpolation table and analytical functions, against the oracle's showers.
Counts and history IDs are identical, energy sums within 1e-9 of the primary energy (the bar
of the other shower tests). Particles at the observation level agree to 1e-6: a sample
converges to 5e-5 of its angle, so an ulp of the device's exp or log that adds or saves an
iteration moves an angle by up to 2.5e-9; at a slope of up to 10 the last step's length moves by
10 times that, and the energy left, a tenth of what the step lost or more, by 100 times."""
import numpy as np
import pytest

import oracle_lib
from c8mi import airtables, em
from test_em_front_edges_gpu import batch
from test_em_gpu import STAT_KEYS, compare

pytestmark = pytest.mark.gpu

EXTRA = ("Xe", 54.0, 131.29, 0.02, 8.48, 0x5865000000000036)


class Elements:
    """airtables with the Moliere snapshot of the first `count` elements of air and xenon."""

    def __init__(self, count):
        elements = (airtables.AIR + [EXTRA])[:count]
        total = sum(e[3] for e in elements)
        elements = [(n, z, a, w / total, x0, h) for n, z, a, w, x0, h in elements]
        self.medium = airtables.Medium(elements, airtables.AIR_MEAN_EXCITATION_MEV, airtables.AIR_DENSITY_SEA_LEVEL, 28.96, 0xA1)

    def moliere_snapshot(self):
        return airtables.moliere_snapshot(medium=self.medium)

    def __getattr__(self, name):
        return getattr(airtables, name)


@pytest.mark.parametrize("count", [1, 2, 3, 4])
@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("fast", [0, 1])
def test_components(count, table, fast):
    module = Elements(count)
    snapshot = em.MoliereSnapshot.from_dict(module.moliere_snapshot())
    assert snapshot.component_count == count
    atm, start, tables = em.Atmosphere(), (0.0, 0.0, 500.0), airtables.build_air_tables()
    cfg = em.make_config(module, seed=3, atmosphere=atm, start=start, moliere=True,
                         moliere_table=em.MoliereInterpolation.build(snapshot) if table else None, moliere_fast_iterations=fast)
    prim = batch(600, count)
    want = oracle_lib.em_run_shower(cfg, tables, atm, prim, shower_id=1, first_history_id=2)
    dev = em.EmBackend(cfg, tables, atm)
    dev.begin_shower(1, 2)
    dev.enqueue(prim)
    stats = dev.run()
    hist, ledger = dev.download_profile()
    observed = dev.observations()[0]
    dev.close()
    assert want["stats"]["lepton_steps"] > 2000
    for k in STAT_KEYS:
        assert stats[k] == want["stats"][k], k
    energy = float(prim["energy_gev"].sum())
    expected = em.decode_counters(want["counters"], cfg.struct.profile_energy_scale)
    for k in ("steps", "lepton_limits", "deposited_steps", "invalid_records", "fallback_reasons"):
        assert ledger[k] == expected[k], k
    for k in em.LEDGER_ENERGY_TERMS:
        assert abs(ledger[k] - expected[k]) <= 1e-9 * energy, k
    deposits = want["hist"]["energy_loss"] / cfg.struct.profile_energy_scale
    assert np.max(np.abs(hist["energy_loss"] - deposits)) <= 1e-9 * energy
    ordered = [a[np.lexsort((a["step_id"], a["history_id"]))] for a in (observed, want["observations"])]
    assert ordered[0].size > 50 and np.array_equal(ordered[0]["history_id"], ordered[1]["history_id"])
    for f in ("energy_gev", "time_s"):
        np.testing.assert_allclose(ordered[0][f], ordered[1][f], rtol=1e-6, atol=0)
    np.testing.assert_allclose(ordered[0]["position_m"], ordered[1]["position_m"], rtol=0, atol=1e-4)


@pytest.mark.parametrize("moliere", [False, True])
def test_most_profile_bins(moliere):
    """1024 profile bins, the most: the step kernels hold two showers' histograms, the context and
    the small tables in 78 KB of LDS."""
    atm, start, tables = em.Atmosphere(), (0.0, 0.0, 500.0), airtables.build_air_tables()
    cfg = em.make_config(airtables, seed=4, atmosphere=atm, start=start, moliere=moliere, bins=1024)
    prim = batch(600, 9)
    want = oracle_lib.em_run_shower(cfg, tables, atm, prim, shower_id=1, first_history_id=2)
    dev = em.EmBackend(cfg, tables, atm)
    dev.begin_shower(1, 2)
    dev.enqueue(prim)
    got = {"stats": dev.run()}
    got["hist"], got["ledger"] = dev.download_profile()
    got["observations"], got["fallbacks"] = dev.observations()[0], dev.fallbacks()[0]
    dev.close()
    compare(cfg, want, got, float(prim["energy_gev"].sum()))
