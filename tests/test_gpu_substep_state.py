"""What a substep leaves behind, and what it starts from: the layout in the
context after fvm_substep_run stays usable through the other entry points."""
import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from fvmhd3d_amd import mesh as M
from fvmhd3d_amd.substep import DeviceSubstepper, GpuBackend, Substepper, ic_disk, ic_thin_disk
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _mesh(n, seed):
    pos = M.uniform_random(n, seed=seed)
    return M.build_periodic(pos[M.morton_order(pos, (1, 1, 1))])


def _partial_substep(m, ic=ic_disk, dtmax=0.25):
    """A device substepper just after a substep with inactive neighbours, the host
    driver of the same substeps, and that substep's layout (state, perm)."""
    W = ic(m.pos)
    D = DeviceSubstepper(m, W, dtmax=dtmax, limiter=G.LIMITER_SMOOTH)
    H = Substepper(m, W, dtmax=dtmax, limiter=G.LIMITER_SMOOTH)
    B = GpuBackend(H.gamma, H.courant, tuple(float(b) for b in m.box), limiter=G.LIMITER_SMOOTH)
    D.init_rungs()
    H.init_rungs(B)
    for k in range(16):
        assert D.substep() == H.substep(B)
        nact, _, nimp, _ = D.local_counts[-1]
        if k > 2 and 0 < nact < m.ncell // 2 and nimp > 0:
            break
    else:
        raise AssertionError("no partial substep")
    active = np.zeros(m.ncell, dtype=bool)
    active[H.last_active] = True
    st, perm = H._state(active, H.last_active)
    D.ctx.np = len(perm)
    return D, H, st, perm


def _lists_and_results(ctx, st):
    for name in G.FIELDS:
        ctx.upload(name, getattr(st, name))
    ctx.set_time(st.t_global)
    fa = ctx.get_active_faces()
    ctx.compute_reconstruction()
    ctx.slope_limiter()
    ctx.compute_fluid_update(False)
    return [fa] + [ctx.download(f) for f in ("x", "y", "z", "t", "lim", "dU", "dgp", "ddivB")]


def test_layout_with_boundary_flags_lists_its_active_faces():
    """Boundary flags uploaded to a substep's layout, then the active faces asked for
    again: the list is that of the flags in the layout (the oracle's, on the same
    layout), whatever flags the global state has had uploaded; the face-end lists
    agree with those of a context that was given the layout as a mesh."""
    m = _mesh(10 ** 3, 9)
    D, H, st, perm = _partial_substep(m)
    assert len(D.ctx.get_active_faces()) == len(st.faces)
    rng = np.random.default_rng(2)
    st.bnd[rng.choice(st.np, size=st.np // 3, replace=False)] = G.OUTFLOW
    want = np.asarray(Oracle("f64", limiter=G.LIMITER_SMOOTH).get_active_faces(st.copy()))
    assert 0 < len(want) < len(st.faces)
    P = G.Context(gamma=H.gamma, courant=H.courant, box=st.box, limiter=G.LIMITER_SMOOTH)
    P.upload_state(st)
    ref = _lists_and_results(P, st)
    assert np.array_equal(ref[0], want)
    flags = np.zeros(m.ncell, np.int32)
    for some in (0, 1, 0):
        flags[:5] = some
        D.ctx.substep_upload("bnd", flags)
        for a, b in zip(_lists_and_results(D.ctx, st), ref):
            assert np.array_equal(a, b)
    P.close()
    D.ctx.close()


def test_refused_substep_leaves_the_layout_before_it():
    """A substep refused because its active cells do not end their step now: the
    layout of the substep before it still gives its face lists and results (those
    of a context that was given it as a mesh), and the substeps go on."""
    m = _mesh(10 ** 3, 9)
    D, H, st, perm = _partial_substep(m)
    for every in (0xFFFFFFFF, 1 << D.max_rung()):  # every cell; the cells of the finest rung
        with pytest.raises(G.FvmError) as e:
            D.ctx.substep_run(every, -1.0, 0.25, 0, 6)
        assert e.value.code == G.FVM_ESTATE
    P = G.Context(gamma=H.gamma, courant=H.courant, box=st.box, limiter=G.LIMITER_SMOOTH)
    P.upload_state(st)
    for a, b in zip(_lists_and_results(D.ctx, st), _lists_and_results(P, st)):
        assert np.array_equal(a, b)
    B = GpuBackend(H.gamma, H.courant, st.box, limiter=G.LIMITER_SMOOTH)
    for _ in range(3):
        assert D.substep() == H.substep(B)
    assert np.array_equal(D.state("W"), H.W)
    P.close()
    D.ctx.close()


@pytest.mark.parametrize("case", ["disk_random_12", "thin_disk_lattice_17"])
def test_uploaded_state_runs_in_index_order(case):
    """A state taken between two substeps (fields, times and rungs) uploaded into a new
    context and run on without fvm_substep_init_rungs: its cells count as pushed in
    index order, and the substeps equal the host driver's with those stamps, bit for
    bit.  17^3 = 4913 cells: active lists on both sides of 4096 cells, whose orders
    come from two sorts."""
    if case == "disk_random_12":
        m, ic, dtmax = _mesh(12 ** 3, 9), ic_disk, 0.25
    else:
        m, ic, dtmax = M.workload_mesh("lattice", 17), ic_thin_disk, 0.125
    _, H, _, _ = _partial_substep(m, ic, dtmax)
    H.seq[:] = np.arange(m.ncell)
    H.next_seq = m.ncell
    D = DeviceSubstepper(m, H.W, dtmax=dtmax, limiter=G.LIMITER_SMOOTH)
    for name in ("U", "x", "y", "z", "t", "mm_lo", "mm_hi", "J", "dU", "dgp", "ddivB", "mvol", "bnd", "tbeg", "tend",
                 "dt_new", "rung"):
        D.ctx.substep_upload(name, getattr(H, name))
    D.clock.tsysU, D.clock.min_rung = H.clock.tsysU, H.clock.min_rung
    D.hist = np.bincount(H.rung, minlength=32).astype(np.int32)
    B = GpuBackend(H.gamma, H.courant, tuple(float(b) for b in m.box), limiter=G.LIMITER_SMOOTH)
    nact = []
    for k in range(32):
        a, b = H.substep(B), D.substep()
        assert a == b, k
        nact.append(a[0])
    assert np.all(np.isfinite(H.dU))
    for name in ("W", "U", "dU", "t", "tend", "dt_new"):
        assert np.array_equal(getattr(H, name), D.state(name).reshape(getattr(H, name).shape)), name
    assert np.array_equal(H.rung, D.state("rung"))
    assert m.ncell < 4096 or min(nact) <= 4096 < max(nact)
    D.ctx.close()
