"""Cells with more faces than the 16-lanes-per-cell kernels stage at once, and
active lists around the size where their sort changes.

The reconstruction and the slope limiter stage 24 faces of a cell at a time: a
cell inside a shell of generators has one face per shell generator, here on
both sides of one and two chunks.  Everything is compared with the oracle at the
bar of the parity tests (1e-12 of a component's largest value); the total cell
count is no multiple of the four cells of a wavefront.  Lists of more than 64
faces are ranked without LDS (cell lists of an uploaded face list, face-end
lists)."""
import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from fvmhd3d_amd import mesh as M
from fvmhd3d_amd.state import global_step_state
from tests.helpers import perturb_gradients
from tests.test_gpu_parity import _run_pipeline

pytestmark = pytest.mark.gpu


def shell_mesh(nshell):
    """A cell with nshell faces: its generator at the centre of a Fibonacci shell."""
    k = np.arange(nshell) + 0.5
    th, ph = np.arccos(1.0 - 2.0 * k / nshell), np.pi * (1.0 + 5.0 ** 0.5) * k
    shell = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], 1)
    rng = np.random.default_rng(nshell)
    shell *= 1.0 + 0.01 * rng.standard_normal((nshell, 1))
    far = rng.uniform(0.0, 1.0, (400, 3))
    far = far[np.linalg.norm(far - 0.5, axis=1) > 0.3]
    m = M.build_periodic(np.concatenate([[[0.5, 0.5, 0.5]], 0.5 + 0.2 * shell, far[:183]]))
    assert m.cell_off[1] == nshell
    return m


@pytest.mark.parametrize("limiter", [G.LIMITER_SHIPPED, G.LIMITER_MINMOD, G.LIMITER_SMOOTH])
@pytest.mark.parametrize("nshell", [23, 24, 25, 48, 49, 70])
def test_many_faced_cells(nshell, limiter):
    m = shell_mesh(nshell)
    st = global_step_state(m, M.ic_orszag_tang(m.pos), dt=1e-3)
    _run_pipeline("f64", limiter, perturb_gradients(st, scale=0.2))


@pytest.mark.parametrize("nshell", [63, 64, 65, 70])
def test_uploaded_face_lists_of_many_faced_cells(nshell):
    """Cell lists built on the device equal the mesh builder's exactly."""
    m = shell_mesh(nshell)
    ctx = G.Context()
    ctx.upload_faces(m.ncell, m.ncell, 0, m.faces, m.volume)
    off, cf = ctx.cell_faces()
    ctx.close()
    assert np.array_equal(off, m.cell_off) and np.array_equal(cf, m.cell_face)


@pytest.mark.parametrize("case", ["shell", "lattice"])
def test_substep_lists_match_host_layouts(case):
    """The substep layout's face-end lists (from the cells' global lists) against
    the host driver, whose layouts count over the active faces: a cell with 70
    faces; and 17^3 cells, so that active lists on both sides of 4096 cells (the
    ranked and the radix-sorted order) occur.  Same bits."""
    from fvmhd3d_amd.substep import DeviceSubstepper, GpuBackend, Substepper, ic_thin_disk
    m = shell_mesh(70) if case == "shell" else M.workload_mesh("lattice", 17)
    W = ic_thin_disk(m.pos)
    Sh = Substepper(m, W, dtmax=0.125, limiter=G.LIMITER_SMOOTH)
    Bh = GpuBackend(Sh.gamma, Sh.courant, tuple(m.box), limiter=G.LIMITER_SMOOTH)
    Sd = DeviceSubstepper(m, W, dtmax=0.125, limiter=G.LIMITER_SMOOTH)
    Sh.init_rungs(Bh)
    Sd.init_rungs()
    n = []
    for k in range(33):
        a, b = Sh.substep(Bh), Sd.substep()
        assert a == b, (k, a, b)
        n.append(a[0])
    if case == "lattice":
        assert min(n) <= 4096 < max(n)
    for f in ("W", "U", "dU", "tend", "dt_new"):
        ref = np.asarray(getattr(Sh, f), dtype=np.float64)
        assert np.array_equal(ref.view(np.uint64), Sd.state(f).reshape(ref.shape).view(np.uint64)), f
