"""Slabs of more than 512 particles (512 threads, the cells' candidates taken
in windows of one wavefront, the particles that reach a wall flown from a
list) against the captured step graph, bit for bit: many and few candidates
per cell, one cell and many cells per slab, rare and frequent acceptances, and
a wall cell with more particles headed for the wall than the list takes at a
time."""
import numpy as np
import pytest

import helpers
from test_gpu_slab import _assert_same, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cells,ppc,dt,sgwm_mult,steps,shape", [
    (50, 1000, 2.6e-9, 1.0, 60, (0, 0)), (12, 1300, 2e-9, 20.0, 12, (1, 8)), (24, 500, 1e-9, 3.0, 40, (1, 4)),
    (40, 60, 5e-10, 5.0, 60, (20, 8)), (20, 30, 2e-10, 1.0, 60, (10, 4)), (3, 900, 2e-9, 1.0, 30, (1, 8))])
def test_large_slabs_equal_graph(hip, mzo, n_cells, ppc, dt, sgwm_mult, steps, shape):
    case = helpers.couette_case(mzo, n_cells=n_cells, ppc=ppc, seed=n_cells, dt=dt, sgwm_mult=sgwm_mult, dx=1e-5)
    a, b = helpers.store_from_case(hip, case), helpers.store_from_case(hip, case)
    b.set_slab_shape(*shape)
    assert hip.couette_steps(a, steps, 3, dt, props_every=1, mode="graph") == "graph"
    assert hip.couette_steps(b, steps, 3, dt, props_every=1, mode="slab") == "slab", b.slab_info()
    assert b.slab_info()[0] >= 4
    _assert_same(_state(hip, a, n_cells), _state(hip, b, n_cells))
    assert a.collision_factors(1, 1)["n_coll"].sum() > 0
    a.close()
    b.close()


def test_more_wall_hits_than_the_list_holds(hip, mzo):
    """Every particle of both wall cells starts next to its wall and flies
    into it in the first step: 1,200 hits a slab, 512 listed at a time."""
    case = helpers.couette_case(mzo, n_cells=6, ppc=1200, seed=4, dt=2e-10, dx=1e-5)
    pv, n = case["pv"], 7200
    ids = pv.index[:n]
    for cells, x0, v0 in ((ids[:1200], 1e-9, -300.0), (ids[-1200:], 6e-5 - 1e-9, 300.0)):
        pv.x[cells - 1, 0] = x0
        pv.v[cells - 1, 0] = v0
    a, b = helpers.store_from_case(hip, case), helpers.store_from_case(hip, case)
    b.set_slab_shape(1, 8)
    for st, mode in ((a, "graph"), (b, "slab")):
        assert hip.couette_steps(st, 3, 1, case["dt"], props_every=1, mode=mode) == mode
    sa, sb = _state(hip, a, 6), _state(hip, b, 6)
    _assert_same(sa, sb)
    assert np.all(sa[0]["v"][:1200, 0] > -300.0)
    a.close()
    b.close()


@pytest.mark.parametrize("n_cells,ppc,shape", [(7, 250, (1, 4)), (7, 600, (1, 8)), (9, 200, (2, 4)), (9, 400, (2, 8))])
def test_flights_through_a_wall_slab_to_the_wall(hip, mzo, n_cells, ppc, shape):
    """Eight particles next to each wall's slab fly through the whole of it in
    one step (two cells a slab: the last slab is one cell), reach the wall and
    are reflected: an interior slab's flight, with its own wall draws, which
    ends in the neighbour slab."""
    dx, dt, spc = 1e-5, 2e-9, shape[0]
    case = helpers.couette_case(mzo, n_cells=n_cells, ppc=ppc, seed=9, dt=dt, dx=dx)
    pv, last = case["pv"], n_cells - spc * ((n_cells - 1) // spc)
    ids = pv.index[:n_cells * ppc]
    left, right = ids[spc * ppc:spc * ppc + 8], ids[(n_cells - last - 1) * ppc:(n_cells - last - 1) * ppc + 8]
    pv.x[left - 1, 0], pv.v[left - 1, 0] = (spc + 0.3) * dx, -(spc + 0.8) * dx / dt
    pv.x[right - 1, 0], pv.v[right - 1, 0] = (n_cells - last - 0.3) * dx, (last + 0.8) * dx / dt
    one, a, b = (helpers.store_from_case(hip, case) for _ in range(3))
    assert hip.couette_steps(one, 1, 1, dt, props_every=1, mode="graph") == "graph"
    d = one.download_species(1)
    one.close()
    vx = dict(zip(d["index"], d["v"][:, 0]))
    assert sum(0 < vx[i] < 3000 for i in left) >= 5 and sum(-3000 < vx[i] < 0 for i in right) >= 5   # few collided
    assert hip.couette_steps(a, 3, 1, dt, props_every=1, mode="graph") == "graph"
    b.set_slab_shape(*shape)
    assert hip.couette_steps(b, 3, 1, dt, props_every=1, mode="slab") == "slab", b.slab_info()
    assert b.slab_info()[:2] == (shape[1], spc)
    _assert_same(_state(hip, a, n_cells), _state(hip, b, n_cells))
    a.close()
    b.close()


def test_thermal_flights_through_the_last_slab(hip, mzo):
    """401 cells of 400 particles on the shape the library picks, two cells a
    slab and one in the last, 200 steps of 0.33 thermal cell widths (dt * sqrt(k
    T / m) / dx): now and then a particle of the last slab but one reaches the
    wall in one step."""
    n_cells, steps, dx = 401, 200, 1e-6
    dt = 0.33 * dx / np.sqrt(helpers.KB * 300.0 / helpers.MASS_AR)
    case = helpers.couette_case(mzo, n_cells=n_cells, ppc=400, seed=2, dt=dt, dx=dx)
    a, b = helpers.store_from_case(hip, case), helpers.store_from_case(hip, case)
    through = 0
    d = a.download_species(1)
    for t in range(1, 1 + steps):
        before = d
        assert hip.couette_steps(a, 1, t, dt, props_every=1, mode="graph") == "graph"
        d = a.download_species(1)
        n = d["n_total"]
        hit = (before["x"][:n, 0] < (n_cells - 1) * dx) & (before["x"][:n, 0] + before["v"][:n, 0] * dt >= case["L"])
        now = dict(zip(d["index"][:n], d["v"][:n, 0])) if hit.any() else {}
        through += sum(now[i] < 0 for i in before["index"][:n][hit])
    assert through > 0
    assert hip.couette_steps(b, steps, 1, dt, props_every=1, mode="slab") == "slab", b.slab_info()
    assert b.slab_info()[0] >= 4 and b.slab_info()[1] == 2
    _assert_same(_state(hip, a, n_cells), _state(hip, b, n_cells))
    a.close()
    b.close()
