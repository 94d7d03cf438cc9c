"""GPU: neighbour rows above pp_limit, and the lane h solve's occupancy modes,
each against a route of its own.

Rows above pp_limit are searched by whole waves; with SERENX_TUNE_NEIB_GROUP 0
every particle walks the tree alone, for its count and for its row.  The rows --
and so every force, evaluation and step -- are the same bit for bit: at sizes
whose first pass eight particles share, and above 262,144 particles, where one
walk per wave of 64 counts them.
"""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu

KEYS = ("porig", "pos", "v", "h", "rho", "omega", "div_v", "a", "pptot", "pplist")


@pytest.mark.parametrize("precision,thermal", [("fp64", "energy"), ("mixed", "isothermal")])
@pytest.mark.parametrize("n,steps", [(2053, 6), (20000, 6), (262147, 0)])
def test_overflow_rows_equal_the_particles_own_walks(n, steps, precision, thermal):
    from seren_amd.engine import TUNE_NEIB_GROUP, ForceEngine
    pos, vel, mass, _ = cloud(n, "plummer", 47)
    out = []
    for group in (1, 0):
        print(f"case plummer {n} {precision} {thermal} group {group}", flush=True)
        eng = ForceEngine(multipole="quadrupole", mac="geometric", precision=precision,
                          sound_speed=CS, thermal=thermal)
        try:
            eng.set_tuning(TUNE_NEIB_GROUP, group)
            eng.load(pos, vel, mass)
            if thermal == "energy":
                eng.set_energy(np.full(n, CS * CS / 0.4))
            eng.force_eval(hguess=True)
            eng.force_eval()
            d = eng.fetch()
            assert (d["pptot"] > eng.pp_limit).sum() > 0
            d = {key: d[key] for key in KEYS}
            if thermal == "energy":
                d["dudt"] = eng.fetch_energy()[1]
            if steps:
                eng.step_begin("lfkdk", nlevels=3, nbuildstep=4)
                eng.step(steps)
                st = eng.fetch()
                d.update({"step " + key: st[key] for key in KEYS})
            out.append(d)
        finally:
            eng.close()
    for key in out[0]:
        assert np.array_equal(out[0][key], out[1][key]), key


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lane_hsolve_occupancy_modes_agree(precision):
    """SERENX_TUNE_HSOLVE_WAVES chooses between two builds of the lane kernel,
    which solves contexts of more than 65,536 particles: the same h, rho, Omega
    and neighbour lists bit for bit."""
    from seren_amd.engine import TUNE_HSOLVE_WAVES, ForceEngine
    pos, vel, mass, _ = cloud(65601, "r2", 78)
    out = []
    for waves in (0, 8, -1):
        print(f"case {precision} waves {waves}", flush=True)
        eng = ForceEngine(multipole="octupole", mac="gadget2", precision=precision,
                          abserror=1e-4, sound_speed=CS)
        try:
            eng.set_tuning(TUNE_HSOLVE_WAVES, waves)
            eng.load(pos, vel, mass)
            eng.force_eval(hguess=True)
            eng.force_eval()
            out.append(eng.fetch())
        finally:
            eng.close()
    for d in out[1:]:
        for key in ("h", "rho", "omega", "zeta", "pptot", "pplist", "a", "gpot"):
            assert np.array_equal(out[0][key], d[key]), key
