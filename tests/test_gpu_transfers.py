"""Host transfers around the sizes where their route changes: computeFlux batches
through the context's pinned staging, the runtime's copies and the transfer
threads' chunks, and field round trips below and above the threaded size.  The
same kernel runs behind every route, so results are compared bit for bit."""
import threading

import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from fvmhd3d_amd import mesh as M
from fvmhd3d_amd.state import global_step_state
from tests.test_zz_no_alloc import _faces

pytestmark = pytest.mark.gpu

PIN = (1 << 20) // 308
CHUNK = 16384


@pytest.mark.parametrize("n", [1, 255, PIN, PIN + 1, 2 * CHUNK - 1, 2 * CHUNK, 3 * CHUNK + 1, 9 * CHUNK - 7])
def test_flux_batch_routes_agree(n):
    faces = _faces(n, n)
    ctx = G.Context()
    got = ctx.compute_flux(*faces)
    for a in range(0, n, 3000):  # 3000 faces at a time: the pinned staging
        part = ctx.compute_flux(*[x[a:a + 3000] for x in faces])
        for x, y in zip(got, part):
            assert np.array_equal(x[a:a + 3000].view(np.uint64), y.view(np.uint64)), a
    ctx.close()


def test_concurrent_contexts():
    """Two threads with a context each: the second finds the slots in use and takes
    the runtime's copies."""
    faces = _faces(6 * CHUNK, 5)
    ref = None
    out = [None] * 4

    def work(i):
        ctx = G.Context()
        for _ in range(3):
            out[i] = ctx.compute_flux(*faces)
        ctx.close()

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(out))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for o in out:
        ref = ref or o
        assert all(np.array_equal(a.view(np.uint64), b.view(np.uint64)) for a, b in zip(o, ref))


@pytest.mark.parametrize("n", [46, 47, 61])
def test_field_round_trip(n):
    """A ten-wide field of n^3 cells is 7.8, 8.3 and 18 MB: below and above 8 MiB,
    and several slots of 5 MiB with a remainder."""
    m = M.workload_mesh("lattice", n)
    st = global_step_state(m, M.ic_orszag_tang(m.pos), dt=0.0)
    ctx = G.Context()
    ctx.upload_mesh(m.ncell, m.ncell, 0, m.faces, m.cell_off, m.cell_face, m.volume)
    w = np.random.default_rng(n).standard_normal(st.w.shape)
    ctx.upload("w", w)
    assert np.array_equal(ctx.download("w"), w)
    ctx.substep_setup(m.faces, m.cell_off, m.cell_face, m.volume)
    ctx.substep_upload("U", w)
    assert np.array_equal(ctx.substep_download("U"), w)
    ctx.close()
