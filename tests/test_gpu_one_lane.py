"""The one-lane kernels of the device-resident path, which meshes past 32768 (FP64)
and 49152 (FP32) cells run: on small meshes, where FVM_FUSED_ONE_LANE (read at every
launch) selects them, against the quad kernels bit for bit and against the
oracle; and moving meshes just past those sizes.

Every sum of a quad kernel is formed in the order of the one-lane kernel, so the
two agree in every bit, for each limiter, static and moving, at cell counts that
leave a wavefront part empty."""
import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from fvmhd3d_amd import mesh as M
from fvmhd3d_amd.state import global_step_state
from oracle.oracle import Oracle

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


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("n", [12 ** 3, 13 ** 3])
def test_one_lane_addressing_variants_agree(monkeypatch, n, moving):
    """The FP32 flux kernel with 32-bit record offsets (up to 2^24 cells) and with
    64-bit addresses: 27 whole wavefronts, and a last one partly past the last cell,
    whose block read of its own records runs past the array."""
    st = _state(n, moving)
    monkeypatch.setenv("FVM_FUSED_ONE_LANE", "1")
    monkeypatch.delenv("FVM_FUSED_ADDR64", raising=False)
    a = _run(st, G.LIMITER_SMOOTH, G.FUSED_FP32, moving)
    monkeypatch.setenv("FVM_FUSED_ADDR64", "1")
    for x, y in zip(a, _run(st, G.LIMITER_SMOOTH, G.FUSED_FP32, moving)):
        assert np.array_equal(x, y)


def _against_oracle(st, lim, moving, nsteps):
    ref = st.copy()
    o = Oracle("f64", limiter=lim)
    o.get_active_faces(ref)
    dts = np.asarray(o.step_global(ref, 1.0, nsteps))
    out = _run(st, lim, G.FUSED_FP64, moving, nsteps)
    assert np.array_equal(dts, out[0])
    for a, b in ((out[1], ref.w), (out[2], ref.U)):
        assert (np.abs(a - b) / (np.abs(b).max(axis=0) + 1e-300)).max() <= 1e-12
    return out


def _fp32_near(st, lim, moving, nsteps, f64):
    out = _run(st, lim, G.FUSED_FP32, moving, nsteps)
    assert np.array_equal(out[0], f64[0])
    for a, b in ((out[1][:, 0], f64[1][:, 0]), (out[2][:, 4], f64[2][:, 4])):
        assert np.abs(a - b).sum() / np.abs(b).sum() <= 1e-4


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("lim", [G.LIMITER_SHIPPED, G.LIMITER_MINMOD, G.LIMITER_SMOOTH])
def test_one_lane_matches_oracle(monkeypatch, lim, moving):
    """FP64 to 1e-12 of the component's largest magnitude, FP32 to 1e-4 in the relative
    L1 error of density and total energy (the bars of the other fused tests)."""
    st = _state(1003, moving)
    monkeypatch.delenv("FVM_FUSED_ADDR64", raising=False)
    monkeypatch.setenv("FVM_FUSED_ONE_LANE", "1")
    _fp32_near(st, lim, moving, 3, _against_oracle(st, lim, moving, 3))


@pytest.mark.parametrize("n", [32768, 32769, 49152, 49153])
def test_moving_mesh_past_the_quads(monkeypatch, n):
    monkeypatch.delenv("FVM_FUSED_ADDR64", raising=False)
    monkeypatch.delenv("FVM_FUSED_ONE_LANE", raising=False)
    st = _state(n, True)
    f64 = _against_oracle(st, G.LIMITER_MINMOD, True, 2) if n < 40000 else _run(st, G.LIMITER_MINMOD, G.FUSED_FP64, True, 2)
    _fp32_near(st, G.LIMITER_MINMOD, True, 2, f64)
