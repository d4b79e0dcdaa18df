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
