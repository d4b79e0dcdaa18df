"""compute_props! on one wave per cell with eight loads of a lane in flight:
cell sizes around the borders of its two loops (64 particles a pass, 512 a
block of loads), one and two groups, against numpy in long double.  A sum of N
terms is off by at most N 2^-53 of the sum of magnitudes: 1e-12 for 5,000."""
import numpy as np
import pytest

import helpers

pytestmark = pytest.mark.gpu


def test_props_sizes_vs_numpy(hip):
    counts = np.array([1, 63, 64, 65, 448, 449, 511, 512, 513, 575, 576, 960, 961, 1024, 1025, 5000])
    n, nc = int(counts.sum()), len(counts)
    rng = np.random.default_rng(3)
    v = rng.normal(50.0, 300.0, size=(n, 3))
    w = rng.uniform(0.5, 2.0, n)
    first = np.cumsum(counts) - counts
    pia = np.zeros((nc, 7), dtype=np.int64)
    pia[:, 0] = pia[:, 3] = counts
    pia[:, 1], pia[:, 2], pia[:, 5] = first + 1, first + counts, -1
    st = hip.DeviceStore(nc, 1, n)
    st.upload_species(1, np.full((n, 3), 0.5), v, w, np.arange(1, n + 1), pia, n, True, None, n)
    sp = [hip.Species("Ar", helpers.MASS_AR)]
    st.set_species_data(sp)
    pp = hip.compute_props(st, sp)
    for c in range(nc):
        s = slice(first[c], first[c] + counts[c])
        wl, vl = w[s].astype(np.longdouble), v[s].astype(np.longdouble)
        mean = (wl[:, None] * vl).sum(0) / wl.sum()
        T = (wl * ((vl - mean) ** 2).sum(1)).sum() * helpers.MASS_AR / (3 * wl.sum() * helpers.KB)
        assert pp.np[0, c] == counts[c]
        assert abs(pp.n[0, c] / wl.sum() - 1) < 1e-12
        assert np.all(np.abs(pp.v[0, c] - mean) < 1e-12 * 1500.0)
        if counts[c] > 1:
            assert abs(pp.T[0, c] / T - 1) < 1e-11
    st.close()


def test_moments_wave_and_workgroup_per_cell(hip):
    """The same cells alone (a workgroup a cell) and in front of 4,100 more (a
    wave a cell): sums of up to 3,000 positive terms in two orders."""
    counts = np.array([1, 2, 63, 64, 65, 255, 256, 257, 3000, 0, 7] + [3] * 4100)
    rng = np.random.default_rng(4)
    n_all = int(counts.sum())
    v, w = rng.normal(50.0, 300.0, size=(n_all, 3)), rng.uniform(0.5, 2.0, n_all)
    out = []
    for nc in (11, len(counts)):
        k = counts[:nc]
        n = int(k.sum())
        first = np.cumsum(k) - k
        pia = np.zeros((nc, 7), dtype=np.int64)
        pia[:, 0] = pia[:, 3] = k
        pia[:, 1], pia[:, 2], pia[:, 5] = first + 1, first + k, -1
        st = hip.DeviceStore(nc, 1, n)
        st.upload_species(1, np.full((n, 3), 0.5), v[:n], w[:n], np.arange(1, n + 1), pia, n, True, None, n)
        pp = hip.PhysProps(nc, 1, [4, 6, 8], Tref=300.0)
        hip.compute_props_with_total_moments(st, [hip.Species("Ar", helpers.MASS_AR)], pp)
        out.append((pp.n[0, :11], pp.v[0, :11], pp.T[0, :11], pp.moments[0, :11]))
        st.close()
    for a, b, atol in zip(*out, (0.0, 1e-12 * 1500.0, 0.0, 0.0)):
        assert np.allclose(a, b, rtol=1e-12, atol=atol, equal_nan=True)


@pytest.mark.parametrize("more", [0, 1012])
def test_moments_of_cells_on_one_and_all_waves_of_a_workgroup(hip, more):
    """1,020 cells, and 8, a workgroup each, of which those of more than 512 (256)
    particles use all its waves, against numpy in long double: sums of up to 1,500
    positive terms, and a power of a ulp or two each."""
    counts = np.array([256, 257, 1500, 512, 513, 0, 1, 255] + [9] * more)
    nc, n = len(counts), int(counts.sum())
    rng = np.random.default_rng(6)
    v, w = rng.normal(50.0, 300.0, size=(n, 3)), rng.uniform(0.5, 2.0, n)
    first = np.cumsum(counts) - counts
    pia = np.zeros((nc, 7), dtype=np.int64)
    pia[:, 0] = pia[:, 3] = counts
    pia[:, 1], pia[:, 2], pia[:, 5] = first + 1, first + counts, -1
    st = hip.DeviceStore(nc, 1, n)
    st.upload_species(1, np.full((n, 3), 0.5), v, w, np.arange(1, n + 1), pia, n, True, None, n)
    pp = hip.PhysProps(nc, 1, [4, 6], Tref=300.0)
    hip.compute_props_with_total_moments(st, [hip.Species("Ar", helpers.MASS_AR)], pp)
    ratio = []
    for c in range(nc):
        s = slice(first[c], first[c] + counts[c])
        wl, vl = w[s].astype(np.longdouble), v[s].astype(np.longdouble)
        assert pp.np[0, c] == counts[c]
        if counts[c] < 3:
            continue
        mean = (wl[:, None] * vl).sum(0) / wl.sum()
        speed = np.sqrt(((vl - mean) ** 2).sum(1))
        assert abs(pp.n[0, c] / wl.sum() - 1) < 1e-13
        assert np.all(np.abs(pp.v[0, c] - mean) < 1e-12 * 1500.0)
        assert abs(pp.T[0, c] / ((wl * speed ** 2).sum() * helpers.MASS_AR / (3 * wl.sum() * helpers.KB)) - 1) < 1e-12
        ratio.append([pp.moments[0, c, j] / ((wl * speed ** p).sum() / wl.sum()) for j, p in enumerate((4, 6))])
    assert np.allclose(ratio, ratio[0], rtol=1e-12, atol=0)   # the scaling is the same for every cell
    st.close()
