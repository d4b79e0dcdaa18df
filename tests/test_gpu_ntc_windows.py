"""The candidate windows of NTC and SWPM (one wavefront per cell, candidates
evaluated ahead) against the oracle's sequential loops, where the windows can
go wrong: cells of two to five particles (redrawn pairs, particles met twice
in a window), rare acceptances (one long track), frequent ones (several
tracks), splits on every collision, calls of few cells and of more than the
4,096 that run the small cells one lane each.  Counts, ids and the cell table
bit for bit; values to 1e-11, which leaves 1e4 ulp for the ulp or two per
collision by which the device's pow, sin and cos differ from the C library's
over the few hundred collisions of a particle."""
import ctypes as C

import numpy as np
import pytest

import helpers
from test_gpu_configs import _batched_0d

pytestmark = pytest.mark.gpu
RTOL = 1e-11


@pytest.mark.parametrize("method", ["equal", "split", "swpm"])
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("slack,dt_mult", [(1.0, 4.0), (8.0, 2.0), (60.0, 1.0)])
def test_windows_vs_oracle(hip, mzo, method, many, slack, dt_mult):
    counts = [2, 3, 5, 1, 64, 65, 300, 900] + ([12] * 4100 if many else [30] * 6)
    b = _batched_0d(hip, mzo, len(counts), 0, seed=17, counts=counts, cap_mult=12)
    st, pv, pia, it, nc = b["st"], b["pv"], b["pia"], b["it"], len(counts)
    # small cells hardly ever collide at the flow's time step: their volume shrinks
    V = np.minimum(1.0, np.asarray(counts) / 40.0)
    dt = b["dt"] * dt_mult
    sg = np.array([b["cfs"][c].sigma_g_w_max for c in range(nc)]) * slack
    if method == "swpm":
        sg /= 1e23 / np.asarray(counts)
    st.set_sigma_g_w_max(1, 1, sg)
    cfs = (mzo.CFSwpm * nc)() if method == "swpm" else b["cfs"]
    for c in range(nc):
        if method == "swpm":
            cfs[c].sigma_g_max = sg[c]
        else:
            cfs[c].sigma_g_w_max = sg[c]
    for step in (1, 2):
        tag = (step << 4) | 1
        r = mzo.RNG(seed=7, tag=tag)
        if method == "swpm":
            hip.swpm(st, 1, 1.0, dt, V=V, tag=tag)
            for c in range(1, nc + 1):
                mzo.lib().mzo_swpm(r.ref, C.byref(cfs[c - 1]), C.byref(it), pv.p, pia.p, c, 1, 1.0, dt, V[c - 1])
        else:
            hip.ntc(st, 1, 1, dt, V=V, equal_weight=method == "equal", tag=tag)
            for c in range(1, nc + 1):
                mzo.lib().mzo_ntc_single(r.ref, C.byref(cfs[c - 1]), C.byref(it), pv.p, pia.p, c, 1, dt, V[c - 1],
                                         1e-16, 1 if method == "equal" else 0)
        cf = st.collision_factors(1, 1)
        assert np.array_equal(cf["n_coll"], [cfs[c].n_coll for c in range(nc)])
        assert np.array_equal(cf["n_coll_performed"], [cfs[c].n_coll_performed for c in range(nc)])
        got = st.download_species(1)
        assert got["err"] == 0
        helpers.assert_state_matches(mzo, got, pv, pia, rtol=RTOL)
        hip.sort_particles(st, 1)
        mzo.lib().mzo_sort_particles(C.byref(b["grid"]), pv.p, pia.p, 1)
    assert cf["n_coll"].max() > 40 and cf["n_coll_performed"].sum() > 20
    st.close()


@pytest.mark.parametrize("nc", [3, 4200])
def test_two_species_windows_vs_oracle(hip, mzo, nc):
    """Two species of unequal weights: a split lands in either species, which
    ends the window whichever it is."""
    rng = np.random.default_rng(5)
    na, nb = (60, 200) if nc < 100 else (6, 9)
    m = [66.3e-27, 6.65e-27]
    pvs, pia = [mzo.ParticleVector(nc * na), mzo.ParticleVector(nc * nb)], mzo.PIA(nc, 2)
    for s, (pv, n) in enumerate(zip(pvs, (na, nb)), start=1):
        for i in range(1, nc * n + 1):
            pv.pop_to(i)
            pv.set(i, 1e12 * rng.lognormal(), rng.normal(0, np.sqrt(helpers.KB * 300.0 / m[s - 1]), 3),
                   list(rng.uniform(size=3)))
        for c in range(1, nc + 1):
            pia.set(c, s, n, (c - 1) * n + 1, c * n, n)
        pia.set_n_total(s, nc * n)
    its = mzo.interactions(["Ar", "He"])
    st = hip.DeviceStore(nc, 2, [8 * nc * na, 8 * nc * nb])
    for s in (1, 2):
        helpers.upload_from_oracle(st, mzo, pvs[s - 1], pia, species=s)
    st.set_interactions([[type("I", (), dict(mu1=its[i][k].mu1, mu2=its[i][k].mu2, vhs_factor=its[i][k].vhs_factor,
                                             vhs_o=its[i][k].vhs_o))() for k in range(2)] for i in range(2)])
    sg = mzo.lib().mzo_estimate_sigma_g_w_max(C.byref(its[0][1]), m[0], m[1], 300.0, 300.0, 4e12, 1.0)
    st.set_sigma_g_w_max(1, 2, np.full(nc, sg))
    st.set_seed(11)
    cfs = (mzo.CF * nc)()
    for c in range(nc):
        cfs[c].sigma_g_w_max = sg
    dt = 50.0 / (na * nb * sg)
    tag = (3 << 4) | 2
    hip.ntc(st, 1, 2, dt, V=1.0, tag=tag)
    r = mzo.RNG(seed=11, tag=tag)
    for c in range(1, nc + 1):
        mzo.lib().mzo_ntc_two(r.ref, C.byref(cfs[c - 1]), C.byref(its[0][1]), pvs[0].p, pvs[1].p, pia.p, c, 1, 2, dt,
                              1.0, 1e-16, 0)
    cf = st.collision_factors(1, 2)
    assert np.array_equal(cf["n_coll_performed"], [cfs[c].n_coll_performed for c in range(nc)])
    for s in (1, 2):
        got = st.download_species(s)
        assert got["err"] == 0 and got["n_total"] > nc * (na, nb)[s - 1]
        helpers.assert_state_matches(mzo, got, pvs[s - 1], pia, species=s, rtol=RTOL)
    st.close()


@pytest.mark.parametrize("two", [False, True])
def test_equal_weights_without_tolerance_vs_oracle(hip, mzo, two):
    """dw_tol = 0 with equal weights: no pair counts as equal, so a collision
    of two of them leaves a copy of weight 0 of the second, at its position."""
    nc, n = 6, 40
    rng = np.random.default_rng(8)
    names, m = (["Ar", "He"], [66.3e-27, 6.65e-27]) if two else (["Ar"], [66.3e-27])
    ns = len(names)
    pvs, pia = [mzo.ParticleVector(nc * n) for _ in names], mzo.PIA(nc, ns)
    for s, pv in enumerate(pvs, start=1):
        for i in range(1, nc * n + 1):
            pv.pop_to(i)
            pv.set(i, 1e12, rng.normal(0, np.sqrt(helpers.KB * 300.0 / m[s - 1]), 3),
                   [(i - 1) // n + rng.uniform(0.1, 0.9), *rng.uniform(size=2)])
        for c in range(1, nc + 1):
            pia.set(c, s, n, (c - 1) * n + 1, c * n, n)
        pia.set_n_total(s, nc * n)
    its = mzo.interactions(names)
    st = hip.DeviceStore(nc, ns, [8 * nc * n] * ns)
    for s in range(1, ns + 1):
        helpers.upload_from_oracle(st, mzo, pvs[s - 1], pia, species=s)
    st.set_interactions([[type("I", (), dict(mu1=its[i][k].mu1, mu2=its[i][k].mu2, vhs_factor=its[i][k].vhs_factor,
                                             vhs_o=its[i][k].vhs_o))() for k in range(ns)] for i in range(ns)])
    it, b = its[0][ns - 1], ns
    sg = mzo.lib().mzo_estimate_sigma_g_w_max(C.byref(it), m[0], m[-1], 300.0, 300.0, 1e12, 1.0)
    st.set_sigma_g_w_max(1, b, np.full(nc, sg))
    st.set_seed(12)
    cfs = (mzo.CF * nc)()
    for c in range(nc):
        cfs[c].sigma_g_w_max = sg
    dt = 30.0 / (n * n * sg)
    tag = (2 << 4) | 1
    hip.ntc(st, 1, b, dt, V=1.0, dw_tol=0.0, tag=tag)
    r = mzo.RNG(seed=12, tag=tag)
    for c in range(1, nc + 1):
        if two:
            mzo.lib().mzo_ntc_two(r.ref, C.byref(cfs[c - 1]), C.byref(it), pvs[0].p, pvs[1].p, pia.p, c, 1, 2, dt, 1.0,
                                  0.0, 0)
        else:
            mzo.lib().mzo_ntc_single(r.ref, C.byref(cfs[c - 1]), C.byref(it), pvs[0].p, pia.p, c, 1, dt, 1.0, 0.0, 0)
    cf = st.collision_factors(1, b)
    assert np.array_equal(cf["n_coll_performed"], [cfs[c].n_coll_performed for c in range(nc)])
    assert not np.any(cf["n_eq_w_coll_performed"]) and cf["n_coll_performed"].sum() > 20
    got = [st.download_species(s) for s in range(1, ns + 1)]
    assert sum(g["n_total"] for g in got) == ns * nc * n + cf["n_coll_performed"].sum()
    for s, g in enumerate(got, start=1):
        assert g["err"] == 0
        helpers.assert_state_matches(mzo, g, pvs[s - 1], pia, species=s, rtol=RTOL)
    st.close()


@pytest.mark.parametrize("method", ["equal", "split", "swpm"])
@pytest.mark.parametrize("nc", [4097, 8200, 17000])
def test_lanes_and_wavefronts_of_one_call_vs_oracle(hip, mzo, method, nc):
    """Calls of a pass of lanes and a pass of wavefronts over the cells it
    leaves, where those passes' shapes change: groups of 64 cells with no, some and
    only long candidate loops, a last group of one cell, groups of empty cells."""
    rng = np.random.default_rng(nc)
    counts = rng.integers(2, 7, nc)
    counts[64:128] = 30
    counts[128:1024:7] = 60
    counts[2000:2100] = 1
    counts[-1] = 50
    b = _batched_0d(hip, mzo, nc, 0, seed=31, counts=counts, cap_mult=12)
    st, pv, pia, it = b["st"], b["pv"], b["pia"], b["it"]
    sg = np.array([b["cfs"][c].sigma_g_w_max for c in range(nc)]) * 2.0
    if method == "swpm":
        sg /= 1e23 / counts
    st.set_sigma_g_w_max(1, 1, sg)
    cfs = (mzo.CFSwpm * nc)() if method == "swpm" else b["cfs"]
    for c in range(nc):
        if method == "swpm":
            cfs[c].sigma_g_max = sg[c]
        else:
            cfs[c].sigma_g_w_max = sg[c]
    V = counts / np.where(counts > 6, 250.0, 12.0)   # about 40 candidates in the large cells, one in the others
    dt, tag = (1.2 if method == "swpm" else 4.0) * b["dt"], (5 << 4) | 1
    r = mzo.RNG(seed=7, tag=tag)
    if method == "swpm":
        hip.swpm(st, 1, 1.0, dt, V=V, tag=tag)
        for c in range(1, nc + 1):
            mzo.lib().mzo_swpm(r.ref, C.byref(cfs[c - 1]), C.byref(it), pv.p, pia.p, c, 1, 1.0, dt, V[c - 1])
    else:
        hip.ntc(st, 1, 1, dt, V=V, equal_weight=method == "equal", tag=tag)
        for c in range(1, nc + 1):
            mzo.lib().mzo_ntc_single(r.ref, C.byref(cfs[c - 1]), C.byref(it), pv.p, pia.p, c, 1, dt, V[c - 1], 1e-16,
                                     1 if method == "equal" else 0)
    cf = st.collision_factors(1, 1)
    assert np.array_equal(cf["n_coll"], [cfs[c].n_coll for c in range(nc)])
    assert np.array_equal(cf["n_coll_performed"], [cfs[c].n_coll_performed for c in range(nc)])
    assert cf["n_coll"].max() > 20 and np.median(cf["n_coll"]) <= 4
    got = st.download_species(1)
    assert got["err"] == 0
    helpers.assert_state_matches(mzo, got, pv, pia, rtol=RTOL)
    st.close()
