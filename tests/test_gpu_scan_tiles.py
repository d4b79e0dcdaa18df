"""The scan that places created particles, over numbers of cells around its
tiles of 4,096: NTC with splitting against the oracle's per-cell calls, ids,
free ids and the cell table bit for bit."""
import ctypes as C

import numpy as np
import pytest

import helpers
from test_gpu_configs import _batched_0d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [1, 3, 4095, 4096, 4097, 8193])
def test_split_over_scan_tiles_vs_oracle(hip, mzo, nc):
    counts = [40] + [4] * (nc - 1)
    b = _batched_0d(hip, mzo, nc, 0, seed=29, counts=counts, cap_mult=12)
    st, pv, pia = b["st"], b["pv"], b["pia"]
    V = np.minimum(1.0, np.asarray(counts) / 200.0)
    r = mzo.RNG(seed=7, tag=17)
    hip.ntc(st, 1, 1, 4 * b["dt"], V=V, equal_weight=False, tag=17)
    for c in range(1, nc + 1):
        mzo.lib().mzo_ntc_single(r.ref, C.byref(b["cfs"][c - 1]), C.byref(b["it"]), pv.p, pia.p, c, 1, 4 * b["dt"],
                                 V[c - 1], 1e-16, 0)
    got = st.download_species(1)
    assert got["err"] == 0 and got["n_total"] > sum(counts)
    helpers.assert_state_matches(mzo, got, pv, pia, rtol=1e-11)   # the windows' bound
    st.close()
