"""GPU: a forest of more than 25,600 groups takes its walks in tree order instead
of longest first; every cloud's results are those of the cloud alone."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_clouds_of_a_large_forest_equal_themselves_alone(precision):
    kinds = [cloud(6209, "uniform", 99), cloud(2053, "plummer", 100)]
    clouds = kinds * 200   # 98 + 33 groups each
    out = []
    for load in (clouds, kinds[:1], kinds[1:]):
        print(f"case {precision} {len(load)} clouds", flush=True)
        from seren_amd.engine import ForceEngine
        eng = ForceEngine(multipole="octupole", mac="gadget2", precision=precision,
                          abserror=1e-4, sound_speed=CS)
        try:
            off = eng.load_forest(load)
            for k in range(2):
                eng.force_eval(hguess=k == 0)
            out.append((off, eng.fetch(neighbours=False)))
        finally:
            eng.close()
    off, forest = out[0]
    for k in (0, 1, 198, 199, 398, 399):
        alone = out[1 + k % 2][1]
        for key in ("pos", "h", "a", "gpot", "agravmag", "pptot"):
            assert np.array_equal(forest[key][off[k]:off[k + 1]], alone[key]), (k, key)
