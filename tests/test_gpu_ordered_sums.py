"""GPU: small clouds, whose gravity terms are added in the walk's order.

A group whose near-field list was not stored walks the tree again and one wave
adds its pair terms, leaf by leaf; a stored list is gone through by all the
block's waves, which pass their terms on in list order.  Both add the same terms
in the same order, so with room for 4 leaves a group (nearly every list dropped)
the state is the default's bit for bit, also where the second evaluation's MAC
reads the |a| that the pair phase writes, and beside a larger cloud.
"""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu

KEYS = ("porig", "pos", "h", "a", "gpot", "agravmag", "pptot")


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes,profile", [([65], "uniform"), ([2053], "plummer"),
                                           ([6144], "r2"), ([59, 4099, 7001], "uniform")])
def test_dropped_near_lists_change_nothing(precision, sizes, profile):
    from seren_amd.engine import TUNE_NEAR_CAP, ForceEngine
    print(f"case {precision} {sizes} {profile}", flush=True)
    clouds = [cloud(n, profile, 70 + k) for k, n in enumerate(sizes)]
    out = []
    for cap in (None, 4):
        eng = ForceEngine(multipole="octupole", mac="gadget2", precision=precision,
                          abserror=1e-4, sound_speed=CS)
        try:
            if cap is not None:
                eng.set_tuning(TUNE_NEAR_CAP, cap)
            eng.load_forest(clouds)
            for k in range(3):
                eng.force_eval(hguess=k == 0)
            out.append(eng.fetch(neighbours=False))
        finally:
            eng.close()
    for key in KEYS:
        assert np.array_equal(out[0][key], out[1][key]), key
