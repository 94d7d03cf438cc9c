"""GPU: fetched neighbour rows longer than the buffer that they pass through
(8,192 particles a group, 16,384 for the smallest clouds)."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [20, 130])
def test_rows_longer_than_the_buffer(n):
    """Standard SPH with one h that reaches every particle: the same rows whether
    they have room for 400 or for 50,002 particles."""
    from seren_amd.engine import ForceEngine
    pos, vel, mass, _ = cloud(n, "uniform", 95)
    rows = []
    for gather in (200, 25001):
        print(f"case {n} pp_gather {gather}", flush=True)
        eng = ForceEngine(multipole="quadrupole", mac="geometric", sound_speed=CS,
                          sph="standard", hmin=1.5, pp_gather=gather)
        try:
            eng.load(pos, vel, mass)
            eng.force_eval()
            d = eng.fetch()
            assert d["pplist"].shape == (n, 2 * gather)
            assert (d["pptot"] == n - 1).all()
            assert (d["pplist"][:, n - 1:] == 0).all()
            rows.append(d["pplist"][:, :n - 1])
        finally:
            eng.close()
    assert (rows[0] > 0).all()
    assert np.array_equal(rows[0], rows[1])
