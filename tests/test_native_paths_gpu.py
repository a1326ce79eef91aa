"""The paths of a loss query: the seven points of a Newton step in one cell polynomial of a
linear loss axis, in several cells, and one by one on other axes and without polynomials.
The bars are those of the other native query tests.
"""
import pytest

from c8mi import tables
from test_native_gpu import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [tables.AXIS_LINEAR, tables.AXIS_EXP, tables.AXIS_EXPM1])
@pytest.mark.parametrize("polynomial_every", [0, 1])
@pytest.mark.parametrize("seed,noise", [(21, 0.0), (22, 0.05)])
def test_loss_axes(monkeypatch, kind, polynomial_every, seed, noise):
    plain = tables.axis

    def axis(asked, low, high, nodes):
        if (asked, low, high) == (tables.AXIS_LINEAR, 0.0, 1.0) and kind != tables.AXIS_LINEAR:
            return plain(kind, 1e-3, high, nodes)
        return plain(asked, low, high, nodes)

    monkeypatch.setattr(tables, "axis", axis)
    got, want, q = _compare(seed, noise=noise, count=8000, polynomial_every=polynomial_every)
    loss = q["kind"] == tables.QUERY["loss_fraction"]
    assert (want["newton_iterations"][loss] > 0).sum() > 50
