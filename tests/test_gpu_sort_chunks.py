"""The count-matrix sort where its chunks can go wrong: particle counts about
the ends of chunks of 1,024 and 4,096 and of a wavefront, key ranges wider
than the 4,096 keys counted or ranked at once, capacities that change the
chunk, empty stores; index, PIA and keys bit for bit against the oracle's
counting sort, on computed cells and on stored keys (which lie in the former
order, so a chunk then spans many cells), and again on the sorted state."""
import ctypes as C

import numpy as np
import pytest

import helpers
from test_gpu_parity import _store
from test_gpu_sort_radix import _scattered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nc,cap,nearly", [
    (1, 1, 1, False), (63, 5, 64, False), (1024, 3, 1024, True), (1025, 700, 4000, False),
    (4095, 4096, 8192, False), (9000, 4097, 20000, False), (4097, 9000, 4097, True),
    (70001, 16384, 70001, False), (70001, 16385, 70001, False), (12289, 500, (1 << 21) + 1, True),
    (40000, 6000, (1 << 21) + 1, False), (0, 7, 100, False)])
def test_sort_chunks_vs_oracle(hip, mzo, n, nc, cap, nearly):
    if n == 0:
        pv, pia = mzo.ParticleVector(1), mzo.PIA(nc, 1)
    else:
        pv, pia = _scattered(mzo, n, nc, seed=n + nc, nearly_sorted=nearly)
    grid = mzo.grid1d(1.0, nc)
    st = _store(hip, mzo, pv, pia, nc, cap=cap)
    st.set_grid(hip.Grid1DUniform(1.0, nc))
    for stored in (False, True, False):
        hip.sort_particles(st, 1, compute_cells=not stored)
        if stored:
            mzo.lib().mzo_sort_particles_precomputed(pv.p, pia.p, 1)
        else:
            mzo.lib().mzo_sort_particles(C.byref(grid), pv.p, pia.p, 1)
        got = st.download_species(1)
        assert got["err"] == 0 and got["contiguous"] and got["n_total"] == n
        if n == 0:
            assert np.all(got["pia"] == [0, 0, -1, 0, 0, -1, 0])
            continue
        helpers.assert_state_matches(mzo, got, pv, pia, rtol=0.0, check_buffer=False)
        assert np.array_equal(got["cell"], pv.cell[:n])
    st.close()


def test_forced_matrix_refuses_more_cells_than_it_states(hip):
    """14,336 cells at most where a caller asks for the count matrix, with and
    without allocating."""
    for nc in (14336, 14337):
        st = hip.DeviceStore(nc, 1, 64)
        pia = np.zeros((nc, 7), dtype=np.int64)
        pia[:, 2] = pia[:, 5] = -1
        pia[0] = [3, 1, 3, 3, 0, -1, 0]
        x = np.array([[nc - 0.5, 0, 0], [0.5, 0, 0], [7.5, 0, 0]])
        st.upload_species(1, x, np.zeros((3, 3)), np.ones(3), np.arange(1, 4), pia, 3, True, None, 3)
        st.set_grid(hip.Grid1DUniform(float(nc), nc))
        st.set_sort_path("matrix")
        for sort in (hip.sort_particles, hip.sort_particles_noalloc):
            if nc > 14336:
                with pytest.raises(hip.MzError):
                    sort(st, 1)
            else:
                sort(st, 1)
                assert list(st.download_species(1)["index"]) == [2, 3, 1]
        st.close()
