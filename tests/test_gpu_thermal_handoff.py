"""A new handle hands the thermal field from predictor to corrector below 300,000 spins and draws it
twice above; the values, and so the bits, are the same either way."""
import numpy as np
import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(63, 66, 72), (50, 60, 100), (64, 75, 63)])  # below, at and above
def test_default_equals_both_forms(gpu, dims):
    s, s0 = W.sc_ferro(dims=dims, precision="fp32")[:2]
    out = []
    for thermal_cache in (None, 0, 1):
        with sllg.Context(s) as g:
            if thermal_cache is not None:
                g.set_launch(256, thermal_cache=thermal_cache)
            g.set_spins(s0)
            g.set_temperature(300.0)
            g.step(0, 4)
            g.set_temperature(0.0)
            g.step(4, 1)
            g.set_temperature(50.0)
            g.step(5, 2)
            out.append(g.get_spins())
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
