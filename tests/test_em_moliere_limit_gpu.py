"""Moliere samples whose Newton iteration never converges: the tail kernel ends them when
the iterates repeat, the oracle at the limit of 100 iterations. The same steps fail on both
sides (fallback records and reasons), all other results agree as in the other shower tests.
"""
import numpy as np
import pytest

from c8mi import airtables, em
from test_em_front_edges_gpu import batch
from test_em_gpu import compare, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("table", [True, None])
@pytest.mark.parametrize("fast", [0, 1])
def test_samples_that_never_converge(table, fast):
    prim = batch(30000, 77)
    prim["pid"][prim["pid"] == 22] = 11
    cfg, want, got = run_pair(airtables.build_air_tables(), 0, 0, 5, primaries=prim, start=(0.0, 0.0, 500.0), moliere=True,
                              moliere_table=table, fast_iterations=fast)
    failed = np.asarray(em.decode_counters(want["counters"], cfg.struct.profile_energy_scale)["fallback_reasons"])
    assert failed.sum() >= 3
    compare(cfg, want, got, float(prim["energy_gev"].sum()))
