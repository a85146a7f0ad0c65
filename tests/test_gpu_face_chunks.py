"""Cells with more faces than the 16-lanes-per-cell kernels stage at once.

The reconstruction and the slope limiter stage 24 faces of a cell at a time: a
cell inside a shell of generators has one face per shell generator, here on
both sides of one and two chunks.  Everything is compared with the oracle at the
bar of the parity tests (1e-12 of a component's largest value); the total cell
count is no multiple of the four cells of a wavefront."""
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
