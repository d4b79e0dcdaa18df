"""The captured step graph over several calls on one store, with what its
launches hold changed between them: the current buffer (odd numbers of steps, a
sort, a split's squash), the seed, walls, grid, interaction, time step and
volumes.  Every call against the same step launched kernel by kernel, bit for
bit."""
import numpy as np
import pytest

import helpers
from test_gpu_slab import _assert_same, _state

pytestmark = pytest.mark.gpu
NC = 12


def _walls(hip, st, case):
    st.set_walls(hip.MaxwellWalls1D(case["species"], 500.0, 200.0, -100.0, 800.0, 1.0, 0.5))


def _interaction(hip, st, case):
    it = case["it"]
    st.set_interactions([[type("I", (), dict(mu1=it.mu1, mu2=it.mu2, vhs_factor=5.0 * it.vhs_factor,
                                             vhs_o=it.vhs_o))()]])


def _split(hip, st, case):
    # unequal weights, so the collisions split: group 2, then a squash
    hip.ntc(st, 1, 1, case["dt"], tag=(900 << 4) | 1)
    assert st.scalars(1)["n_total"] > NC * 80


CHANGES = {
    "none": lambda hip, st, case: None,
    "sort": lambda hip, st, case: hip.sort_particles(st, 1),
    "split": _split,
    "seed": lambda hip, st, case: st.set_seed(123),
    "walls": _walls,
    "grid": lambda hip, st, case: st.set_grid(hip.Grid1DUniform(case["L"], NC, wall_offset=1e-3)),
    "interaction": _interaction,
}


@pytest.mark.parametrize("avg", [False, True])
@pytest.mark.parametrize("change", CHANGES)
@pytest.mark.parametrize("counts", [(1, 2, 5), (4, 4, 3), (3, 1, 6)])
def test_graph_calls_equal_eager_calls(hip, mzo, counts, change, avg):
    case = helpers.couette_case(mzo, n_cells=NC, ppc=80, seed=4, dt=5e-10, sgwm_mult=20.0,
                                weights=(lambda r, n: r.uniform(0.5, 2.0, n)) if change == "split" else None)
    out = []
    for mode in ("eager", "graph"):
        st = helpers.store_from_case(hip, case, capacity=NC * 80 * 12)
        st.surf_clear(1)
        st.props_avg_clear()
        step, dt = 1, case["dt"]
        for i, n in enumerate(counts):
            if i:
                CHANGES[change](hip, st, case)
            if avg:
                path = hip.couette_avg_steps(st, n, step, dt, 10, species_data=case["species"], mode=mode)
            else:
                path = hip.couette_steps(st, n, step, dt, species_data=case["species"], props_every=1, mode=mode)
            assert path == mode
            step += n
        out.append((_state(hip, st, NC), hip.PhysProps(NC, 1).fetch_avg(st), hip.SurfProps.grid1d(1).fetch(st, 1)._to_device()))
        st.close()
    _assert_same(out[0][0], out[1][0])
    for k in ("np", "n", "v", "T"):
        assert np.array_equal(getattr(out[0][1], k), getattr(out[1][1], k)), k
    assert np.array_equal(out[0][2], out[1][2])


def test_graph_calls_with_other_steps_and_volumes(hip, mzo):
    """The time step, the cell volumes and the interval of the properties change
    from call to call and back."""
    case = helpers.couette_case(mzo, n_cells=NC, ppc=80, seed=6, dt=5e-10, sgwm_mult=20.0)
    dx = case["L"] / NC
    out = []
    for mode in ("eager", "graph"):
        st = helpers.store_from_case(hip, case)
        step = 1
        for n, dt, V, every in ((3, 5e-10, None, 1), (2, 2e-10, None, 1), (5, 2e-10, 3 * dx, 1), (4, 2e-10, 2 * dx, 0),
                                (3, 5e-10, None, 1)):
            assert hip.couette_steps(st, n, step, dt, species_data=case["species"], props_every=every,
                                     V=None if V is None else np.full(NC, V), mode=mode) == mode
            step += n
        out.append(_state(hip, st, NC))
        st.close()
    _assert_same(*out)
