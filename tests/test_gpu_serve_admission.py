"""Requests whose lattices are prepared ahead of admission: shared and distinct lattices, late
arrivals and small budgets give what each request gives alone; a bad request is refused."""
import numpy as np
import pytest

import sllg
from sllg import batch as SB

pytestmark = pytest.mark.gpu


def _reqs(late):
    out = []
    for k, (L, J, mu) in enumerate([(4, 3e-21, 1.5), (6, 3e-21, 1.5), (4, 3e-21, 2.0), (4, 2e-21, 1.5), (5, 3e-21, 1.5),
                                    (6, 3e-21, 1.5), (4, 3e-21, 1.5), (12, 3e-21, 1.5), (1, 3e-21, 1.5), (5, 1e-21, 1.5)]):
        out.append(dict(type=k % 3, L=L, J=J, mu=mu, steps=40 + 10 * (k % 2), update=10, T=20.0 * k, seed=k + 1,
                        arrival_s=0.002 * (k // 3) if late else 0.0, B0=(0.0, 0.0, -0.1), B1=(0.0, 0.0, 0.1)))
    return out


@pytest.mark.parametrize("late, kw", [(False, {}), (True, {}), (False, dict(max_members=2)),
                                      (False, dict(max_live_spins=300))])
def test_serve_equals_alone(gpu, late, kw):
    specs = _reqs(late)
    res, _, series = SB.serve(SB.make_requests(specs), want_series=True, **kw)
    for spec, r, m in zip(specs, res, series):
        one, _, ms = SB.serve(SB.make_requests([dict(spec, arrival_s=0.0)]), want_series=True)
        assert np.array_equal(m, ms[0])
        assert np.array_equal(r["m_final"], one[0]["m_final"])
        assert ("sq" in r) == ("sq" in one[0])
        if "sq" in r:
            assert np.array_equal(r["sq"], one[0]["sq"])


@pytest.mark.parametrize("bad", [dict(mu=-1.0), dict(mu=0.0), dict(L=0)])
def test_bad_request_is_refused(gpu, bad):
    specs = _reqs(False)
    specs[4].update(bad)
    with pytest.raises(Exception):
        SB.serve(SB.make_requests(specs))
    SB.serve(SB.make_requests(specs[:4]))  # the next run is unaffected
