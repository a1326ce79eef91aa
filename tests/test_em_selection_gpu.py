"""Column selection of photons and e+- over more process columns than the kernels keep the
rates of (16), fewer, and exactly as many, against the oracle's showers. Elements without
an LPM snapshot end in fallback records on both sides. Counts and ledger counts are
identical, energies and profile bins within 1e-9 of the primary energy.
"""
import pytest

from c8mi import airtables
from test_em_front_edges_gpu import batch
from test_em_gpu import compare, run_pair

pytestmark = pytest.mark.gpu


def medium(extra):
    """Air with `extra` further elements of oxygen's kind, 30% of the mass: photons have
    2 (3 + extra) + 1 columns."""
    elements = [(name, z, a, 0.7 * w, x0, h) for name, z, a, w, x0, h in airtables.AIR]
    elements += [(f"X{k}", 8.0 + k, 16.0 + 2 * k, 0.3 / extra, 34.0, 0x5800000000000000 + k) for k in range(extra)]
    return airtables.Medium(elements, airtables.AIR_MEAN_EXCITATION_MEV, airtables.AIR_DENSITY_SEA_LEVEL, 28.96, 0xA1)


@pytest.mark.parametrize("extra", [1, 4, 5, 6, 14])  # 9, 15, 17, 19, 35 columns of a photon
def test_columns_around_the_kept_rates(extra):
    tables = airtables.build_tables(medium(extra), 1.0)
    prim = batch(600, extra)
    cfg, want, got = run_pair(tables, 0, 0, 40 + extra, primaries=prim, start=(0.0, 0.0, 500.0))
    assert want["stats"]["photon_interactions"] > 300 and want["stats"]["lepton_interactions"] > 200
    compare(cfg, want, got, float(prim["energy_gev"].sum()))
