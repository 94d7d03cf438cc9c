"""GPU: hydro forces with eight lanes per particle at sizes around their
waves and rows of one term to hundreds: mixed precision (whose lanes add FP32
terms in list order through LDS) against FP64 (whose lanes add in a tree), at
the bars that the mixed kernel holds against FP64 elsewhere: 1e-5 rms and 1e-3
of the rms acceleration at most."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,profile", [(58, "uniform"), (63, "uniform"), (65, "uniform"),
                                       (71, "r2"), (2053, "plummer")])
def test_mixed_against_fp64(n, profile):
    from seren_amd.engine import ForceEngine
    got = []
    for precision in ("fp64", "mixed"):
        print(f"case {n} {profile} {precision}", flush=True)
        eng = ForceEngine(multipole="quadrupole", mac="geometric", sound_speed=CS,
                          precision=precision)
        try:
            eng.load(*cloud(n, profile, 70))
            eng.force_eval(hguess=True, grav=False)
            got.append(eng.fetch(neighbours=False))
        finally:
            eng.close()
    assert np.array_equal(got[0]["pptot"], got[1]["pptot"])
    d = np.linalg.norm(got[1]["a"] - got[0]["a"], axis=1)
    scale = np.sqrt((got[0]["a"]**2).sum(1).mean())
    assert np.sqrt((d**2).mean()) <= 1e-5 * scale
    assert d.max() <= 1e-3 * scale
