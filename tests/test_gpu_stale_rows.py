"""GPU: neighbour rows on a tree that was stocked before the particles moved.

The drop-in drivers search with the bounding spheres of the last stock.  A
moved particle can lie outside them, so its list is what its own walk opens,
and a leaf can pass the walk's test where one of its ancestors fails it (its
sphere need not lie within theirs).  Rows from searches that eight particles
share, rows above pp_limit (searched one by one) and the particles' own walks
must agree all the same, in the counts, the lists and the forces summed over
them, bit for bit.

Short filaments give flat leaves that stick out of their branches: in a model
of these clouds on the CPU, 15 to 17 rows above pp_limit per cloud hold fewer
particles by the own walk than by tests of the leaves alone.
"""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from helpers import CS, cloud  # noqa: E402

pytestmark = pytest.mark.gpu


def _filaments(n, seed, length):
    """Groups of eight points on a line along one axis, in the unit cube."""
    rng = np.random.default_rng(seed)
    k = n // 8 + 1
    centre, axis = rng.uniform(-1, 1, (k, 3)), rng.integers(0, 3, k)
    pos = np.repeat(centre, 8, 0)
    pos[np.arange(8 * k), np.repeat(axis, 8)] += rng.uniform(-length, length, (k, 8)).ravel()
    return pos[:n], 0.1 * rng.standard_normal((n, 3)), np.full(n, 1.0 / n), np.full(n, 0.1)


def _rows(group, ics, move, **kw):
    from seren_amd import engine as sx
    pos, vel, mass, h = ics
    eng = sx.ForceEngine(multipole="quadrupole", mac="geometric", sound_speed=CS, **kw)
    try:
        eng.set_tuning(sx.TUNE_NEIB_GROUP, group)
        st = sx.SerenState(pos, vel, mass, h, eng.pp_limit)
        sx.tree_update(eng, st)
        st.parray[:, :3] = move(st.parray[:, :3])
        sx.sph_update(eng, st)
        sx.update_thermal_properties_isothermal(st, CS)
        sx.sph_hydro_forces(eng, st)
        return eng.pp_limit, dict(parray=st.parray.copy(), pptot=st.pptot.copy(),
                                  pplist=st.pplist.copy(), rho=st.rho.copy(), a=st.a.copy())
    finally:
        eng.close()


def _compare(ics, move, **kw):
    limit, waves = _rows(1, ics, move, **kw)
    _, walks = _rows(0, ics, move, **kw)
    assert (walks["pptot"] > limit).sum() > 0
    for key in walks:
        assert np.array_equal(waves[key], walks[key]), key


@pytest.mark.parametrize("length,hmin,amount", [(0.2, 0.1, 0.06), (0.2, 0.1, 0.1),
                                                (0.1, 0.1, 0.06), (0.05, 0.06, 0.15)])
def test_constant_h(length, hmin, amount):
    """Standard SPH with one h for all and rows of four, so nearly every row is
    searched by both passes; noise, or (the last) a shift of the whole cloud."""
    print(f"case filaments {length} h {hmin} moved by {amount}", flush=True)

    def move(x):
        if length == 0.05:
            return x + amount * np.array([0.6, 0.64, 0.48])
        return x + amount * np.random.default_rng(5).standard_normal(x.shape)
    _compare(_filaments(2053, 3, length), move, sph="standard", hmin=hmin, pp_gather=2)


@pytest.mark.parametrize("n,seed,amount", [(2053, 83, 0.02), (2053, 85, 0.005), (20011, 86, 0.01)])
def test_gradh(n, seed, amount):
    """Plummer spheres, whose outskirts have rows above pp_limit."""
    print(f"case plummer {n} {seed} moved by {amount}", flush=True)
    pos, vel, mass, _ = cloud(n, "plummer", seed)
    _compare((pos, vel, mass, np.full(n, 0.05)),
             lambda x: x + amount * np.random.default_rng(1).standard_normal(x.shape))
