"""Moliere samples whose Newton iteration never converges: the tail kernel ends them when
the iterates repeat, the oracle at the limit of 100 iterations. The same steps of the same
particles fail on both sides, and every count agrees. (Values are the business of the other
shower tests, on fewer steps: a converged sample stops within 5e-5 of its root, so an ulp of
the device's exp or log that adds or saves an iteration moves an angle by up to 2.5e-9.)
"""
import pytest

from c8mi import airtables, em
from test_em_front_edges_gpu import batch
from test_em_gpu import STAT_KEYS, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("table", [True, None])
@pytest.mark.parametrize("fast", [0, 1])
def test_samples_that_never_converge(table, fast):
    prim = batch(30000, 77)
    prim["pid"][prim["pid"] == 22] = 11
    cfg, want, got = run_pair(airtables.build_air_tables(), 0, 0, 5, primaries=prim, start=(0.0, 0.0, 500.0), moliere=True,
                              moliere_table=table, fast_iterations=fast)
    ledger = em.decode_counters(want["counters"], cfg.struct.profile_energy_scale)
    assert sum(ledger["fallback_reasons"]) >= 3
    assert got["ledger"]["fallback_reasons"] == ledger["fallback_reasons"]
    for k in STAT_KEYS:
        assert got["stats"][k] == want["stats"][k], k
    ids = [sorted(zip(side["fallbacks"]["particle"]["history_id"].tolist(), side["fallbacks"]["particle"]["step_id"].tolist(),
                      side["fallbacks"]["reason"].tolist())) for side in (want, got)]
    assert ids[0] == ids[1]
