"""GPU: the gravity walk's split of a group over lanes and waves, at group
sizes around the edges of its parts.

With a vanishing opening angle no cell is accepted, so the walk's near lists
hold every leaf and its pair phase is the direct sum.  Both sum the same FP64
terms in different orders: at most n additions of relative error 2^-53 each,
on sums whose terms exceed the result by less than 1e3 here, so 1e-10 of the
largest acceleration bounds the difference for n < 1e3.
"""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("near_cap", [4096, 4])
@pytest.mark.parametrize("n", [58, 63, 64, 65, 79, 81, 128, 191, 700])
def test_pair_phase_is_the_direct_sum(n, near_cap):
    from seren_amd.engine import TUNE_NEAR_CAP, ForceEngine
    print(f"case n {n} near_cap {near_cap}", flush=True)
    eng = ForceEngine(multipole="quadrupole", mac="geometric", thetamaxsqd=1e-12, sound_speed=CS)
    try:
        eng.set_tuning(TUNE_NEAR_CAP, near_cap)
        eng.load(*cloud(n, "r2", 40 + n))
        eng.force_eval(hguess=True, hydro=False)
        d = eng.fetch(neighbours=False)
        a, pot = eng.direct_gravity(np.arange(n, dtype=np.int32))
    finally:
        eng.close()
    assert np.abs(d["a"] - a).max() <= 1e-10 * np.abs(a).max()
    assert np.abs(d["gpot"] - pot).max() <= 1e-10 * np.abs(pot).max()
