"""GPU: the FP64 walk by blocks with fewer registers (from as many groups as the
device has CUs on, 16,384 particles) against the one with more: a cloud's walk is
the same bit for bit alone and beside one that takes the launch past the line."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,profile,multipole,mac", [(6145, "uniform", "octupole", "gadget2"),
                                                     (9001, "plummer", "quadrupole", "geometric"),
                                                     (16001, "r2", "octupole", "eigen")])
def test_cloud_alone_equals_cloud_in_a_launch_of_many_groups(n, profile, multipole, mac):
    from seren_amd.engine import ForceEngine
    small, other = cloud(n, profile, 97), cloud(16385, "uniform", 98)
    out = []
    for clouds in ([small], [small, other]):
        print(f"case {n} {profile} {multipole} {mac} of {len(clouds)}", flush=True)
        eng = ForceEngine(multipole=multipole, mac=mac, abserror=1e-4, sound_speed=CS)
        try:
            eng.load_forest(clouds)
            for k in range(2):
                eng.force_eval(hguess=k == 0)
            out.append(eng.fetch(neighbours=False))
        finally:
            eng.close()
    for key in ("pos", "h", "a", "gpot", "agravmag"):
        assert np.array_equal(out[0][key], out[1][key][:n]), key
