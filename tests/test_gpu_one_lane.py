"""The one-lane kernels of the device-resident path, which meshes past 32768 (FP64)
and 49152 (FP32) cells run: on small meshes, where FVM_FUSED_ONE_LANE (read at every
launch) selects them, against the quad kernels bit for bit.

Every sum of a quad kernel is formed in the order of the one-lane kernel, so the
two agree in every bit, for each limiter, static and moving, at cell counts that
leave a wavefront part empty."""
import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from fvmhd3d_amd import mesh as M
from fvmhd3d_amd.state import global_step_state

pytestmark = pytest.mark.gpu


def _state(n, moving):
    pos = M.uniform_random(n, seed=7)
    m = M.build_periodic(pos[M.morton_order(pos, (1, 1, 1))])
    W = M.ic_orszag_tang(m.pos)
    vel = None
    if moving:
        vel = W[:, 1:4] + 0.01 * np.random.default_rng(n).standard_normal((n, 3))
    return global_step_state(m, W, dt=0.0, vel=vel)


def _run(st, lim, precision, moving, nsteps=3):
    ctx = G.Context(gamma=st.gamma, courant=st.courant, box=st.box, limiter=lim)
    ctx.upload_state(st.copy())
    ctx.fused_setup(precision, moving=moving)
    ctx.fused_run(nsteps, 1.0)
    ctx.fused_sync()
    out = [ctx.fused_dt_history(nsteps)] + [ctx.download(f) for f in ("w", "U", "x", "y", "z", "t", "dt_new")]
    ctx.close()
    return out


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("lim", [G.LIMITER_SHIPPED, G.LIMITER_MINMOD, G.LIMITER_SMOOTH])
@pytest.mark.parametrize("precision", [G.FUSED_FP64, G.FUSED_FP32])
@pytest.mark.parametrize("n", [67, 1003])
def test_quads_have_the_bits_of_one_lane(monkeypatch, n, precision, lim, moving):
    st = _state(n, moving)
    monkeypatch.delenv("FVM_FUSED_ADDR64", raising=False)
    monkeypatch.delenv("FVM_FUSED_ONE_LANE", raising=False)
    quads = _run(st, lim, precision, moving)
    monkeypatch.setenv("FVM_FUSED_ONE_LANE", "1")
    for a, b in zip(quads, _run(st, lim, precision, moving)):
        assert np.all(np.isfinite(b)) and np.array_equal(a, b)
