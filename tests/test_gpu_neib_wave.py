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


@pytest.mark.parametrize("n,profile", [(58, "uniform"), (71, "r2"), (2053, "plummer")])
def test_rows_equal_the_walks_on_a_tree_stocked_before(n, profile):
    """The drop-in drivers cannot know whether the host moved its particles since
    the tree was stocked: there each particle's own sphere test decides."""
    from seren_amd import engine as sx
    pos, vel, mass, h = cloud(n, profile, 80)
    got = []
    for group in (1, 0):
        print(f"case {n} {profile} group {group}", flush=True)
        eng = sx.ForceEngine(multipole="quadrupole", mac="geometric", sound_speed=CS)
        try:
            eng.set_tuning(sx.TUNE_NEIB_GROUP, group)
            st = sx.SerenState(pos, vel, mass, np.full(n, 0.2) if h is None else h, eng.pp_limit)
            sx.tree_update(eng, st)
            st.parray[:, :3] += 1e-3 * np.random.default_rng(1).standard_normal((n, 3))
            sx.sph_update(eng, st)
            got.append((st.parray.copy(), st.pptot.copy(), st.pplist.copy(), st.rho.copy()))
        finally:
            eng.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
