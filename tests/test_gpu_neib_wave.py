"""GPU: neighbour rows from searches by whole waves against the per-particle
walks: the same rows in the same order, so everything is equal bit for bit.
Sizes around the eight particles of a wave, clouds that share a wave, and rows
above pp_limit (the Plummer sphere's outskirts)."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,profile", [([58], "uniform"), ([63], "uniform"), ([65], "r2"),
                                           ([71, 58, 61], "uniform"), ([2053], "plummer"),
                                           ([300, 2053, 59], "plummer")])
def test_rows_equal_the_walks(sizes, profile):
    from seren_amd.engine import TUNE_NEIB_GROUP, ForceEngine
    clouds = [cloud(n, profile, 60 + k) for k, n in enumerate(sizes)]
    got = []
    for group in (1, 0):
        print(f"case {sizes} {profile} group {group}", flush=True)
        eng = ForceEngine(multipole="quadrupole", mac="geometric", sound_speed=CS)
        try:
            eng.set_tuning(TUNE_NEIB_GROUP, group)
            eng.load_forest(clouds)
            eng.force_eval(hguess=True)
            got.append(eng.fetch())
        finally:
            eng.close()
    for key in got[0]:
        assert np.array_equal(got[0][key], got[1][key]), key
