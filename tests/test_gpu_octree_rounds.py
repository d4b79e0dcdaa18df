"""The octree merge's splits worked out ahead of the refine order, where the
order is hard: equal weights (ties everywhere, broken by the bin ids), weights
over many decades (a child nearly as heavy as its parent, so the order dives),
velocities on a coarse lattice (bins that cannot be told apart split to the
depth limit), zero weights, targets from a few bins to nearly the cell, bins
that run out; in LDS and on the device-memory path, against the oracle's
sequential merge: ids, cell table and free ids bit for bit, values to 1e-12 as
in the other octree tests."""
import numpy as np
import pytest

import helpers

pytestmark = pytest.mark.gpu


def _cells(mzo, counts, weights, lattice, seed):
    rng = np.random.default_rng(seed)
    n, nc = sum(counts), len(counts)
    pv, pia = mzo.ParticleVector(n), mzo.PIA(nc, 1)
    for i in range(1, n + 1):
        pv.pop_to(i)
    v = rng.normal(0.0, 300.0, size=(n, 3))
    pv.v[:n] = np.round(v / 150.0) * 150.0 if lattice else v
    pv.x[:n] = rng.uniform(0.01, 0.99, size=(n, 3))
    pv.x[:n, 0] += np.repeat(np.arange(nc), counts)
    pv.w[:n] = {"equal": np.ones(n), "decades": 10.0 ** rng.uniform(-12, 0, n),
                "zeros": np.where(rng.random(n) < 0.6, 0.0, rng.uniform(0.5, 2, n))}[weights]
    pos = 1
    for c, k in enumerate(counts, start=1):
        pia.set(c, 1, k, pos, pos + k - 1, k)
        pos += k
    pia.set_n_total(1, n)
    return pv, pia


@pytest.mark.parametrize("weights", ["equal", "decades", "zeros"])
@pytest.mark.parametrize("lattice", [False, True])
@pytest.mark.parametrize("counts,targets,max_nbins,max_depth", [
    ([64, 65, 500, 1300, 2048], [16, 63, 40, 1000, 2000], 512, 10),
    ([2049, 3000, 5000, 700], [400, 2900, 3000, 690], 16384, 10),
    ([900, 4000], [800, 3900], 60, 4), ([3, 17, 40], [2, 16, 39], 512, 10),
    ([24000, 2100], [23000, 1500], 32768, 10),   # a list of bins larger than LDS
    ([2060] * 300, [150] * 300, 512, 10)])       # more large cells than CUs
def test_octree_rounds_vs_oracle(hip, mzo, weights, lattice, counts, targets, max_nbins, max_depth):
    nc = len(counts)
    pv, pia = _cells(mzo, counts, weights, lattice, seed=sum(counts))
    st = hip.DeviceStore(nc, 1, sum(counts) + 512)
    helpers.upload_from_oracle(st, mzo, pv, pia)
    st.set_grid(hip.Grid1DUniform(float(nc), nc))
    st.set_seed(99)
    tag = (4 << 4) | 3
    thresholds = np.array(targets, dtype=np.int32)
    merged = hip.merge_octree_targets(st, 1, thresholds, thresholds, max_Nbins=max_nbins, max_depth=max_depth,
                                      squash=False, tag=tag)
    assert merged == nc
    r = mzo.RNG(seed=99, tag=tag)
    for c in range(1, nc + 1):
        oc = mzo.Octree(max_Nbins=max_nbins, max_depth=max_depth)
        mzo.lib().mzo_merge_octree_N2_based(r.ref, oc.p, pv.p, pia.p, c, 1, int(targets[c - 1]), None)
    got = st.download_species(1)
    assert got["err"] == 0
    helpers.assert_state_matches(mzo, got, pv, pia, rtol=1e-12)
    st.close()
