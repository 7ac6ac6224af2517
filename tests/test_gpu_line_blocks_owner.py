"""Line blocks are built where Heun steps of a handle can read them, and nowhere else."""
import numpy as np
import pytest

import sllg
from sllg import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["heun", "rk4", "rk5"])
def test_blocks_by_scheme(gpu, scheme):
    s = W.fcc_3shell(dims=(9, 10, 11), scheme=scheme)[0]
    with sllg.Context(s) as g:
        assert ("-blocks" in g.info()["exch_encoding"]) == (scheme == "heun")
        bytes_with = g.info()["device_bytes"]
        g.step(0, 2)
    s.flags = sllg.FLAG_NO_LINE_MODE  # packed entries alone
    with sllg.Context(s) as g:
        assert (g.info()["device_bytes"] < bytes_with) == (scheme == "heun")
        g.step(0, 2)
        assert np.all(np.isfinite(g.get_spins()))
