"""Uploads behind queued steps: a call that replaces what the steps still read
(collision factors, volumes, mass, grid, particles) acts after them, as if the
program had waited in between.  Against the same calls with a wait, bit for
bit."""
import numpy as np
import pytest

import helpers
from test_gpu_slab import _assert_same, _state

pytestmark = pytest.mark.gpu
NC, PPC, STEPS = 200, 100, 400


@pytest.mark.parametrize("what", ["sigma", "grid", "volumes", "mass", "particles", "batch"])
def test_upload_acts_after_queued_steps(hip, mzo, what):
    case = helpers.couette_case(mzo, n_cells=NC, ppc=PPC, seed=2, dt=2e-10)
    dt, dx = case["dt"], case["L"] / NC
    out = []
    for wait in (True, False):
        st = helpers.store_from_case(hip, case)
        sp = case["species"]
        V = np.full(NC, dx)
        hip.couette_steps(st, 2, 1, dt, species_data=sp, V=V, mode="graph")   # captures
        st.sync()
        hip.couette_steps(st, STEPS, 3, dt, species_data=sp, V=V if what == "volumes" else None, mode="graph")
        if wait:
            st.sync()
        if what == "sigma":
            st.set_sigma_g_w_max(1, 1, 50.0 * case["sgwm"])
        elif what == "grid":
            st.set_grid(hip.Grid1DUniform(case["L"] * 0.5, NC))
            st.sync()
            st.set_grid(hip.Grid1DUniform(case["L"], NC))
        elif what == "volumes":
            hip.couette_steps(st, 2, 3 + STEPS, dt, species_data=sp, V=0.1 * V, mode="graph")
        elif what == "mass":
            hip.couette_steps(st, 2, 3 + STEPS, dt, species_data=[hip.Species("Ar", 2 * case["mass"])], mode="graph")
        elif what == "particles":
            helpers.upload_from_oracle(st, mzo, case["pv"], case["pia"])
            hip.couette_steps(st, 2, 1, dt, species_data=sp, mode="graph")
        else:
            hip.batch0d_steps(st, 1, 3 + STEPS, dt, [hip.Species("Ar", 2 * case["mass"])], V=0.2 * V)
        out.append(_state(hip, st, NC))
        st.close()
    _assert_same(*out)
