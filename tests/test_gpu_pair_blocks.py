"""GPU: blocks of four waves in the mixed pair phase (3 blocks per CU beside a
cloud of more than 393,216 particles) against blocks of eight: each wave takes
two of a list's eight shares, so the sums are the same bit for bit, with stored
lists and with lists that are walked again, in the large cloud and in one beside
it whose terms are added in list order."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("near_cap", [None, 4])
def test_half_blocks_change_nothing(near_cap):
    from seren_amd.engine import TUNE_NEAR_CAP, TUNE_PAIR_BLOCKS, ForceEngine
    clouds = [cloud(2503, "plummer", 90), cloud(393217, "uniform", 91)]
    out = []
    for blocks in (0, 3):
        print(f"case near cap {near_cap} pair blocks {blocks}", flush=True)
        eng = ForceEngine(multipole="octupole", mac="gadget2", precision="mixed",
                          abserror=1e-3, sound_speed=CS)
        try:
            eng.set_tuning(TUNE_PAIR_BLOCKS, blocks)
            if near_cap is not None:
                eng.set_tuning(TUNE_NEAR_CAP, near_cap)
            eng.load_forest(clouds)
            for k in range(2):
                eng.force_eval(hguess=k == 0)
            out.append(eng.fetch(neighbours=False))
        finally:
            eng.close()
    for key in ("porig", "h", "a", "gpot", "agravmag", "pptot"):
        assert np.array_equal(out[0][key], out[1][key]), key
