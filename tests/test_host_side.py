"""The library's host side without a device: what it allocates and when it waits.

libfvm_gpu.so runs in a process of its own over tests/hip_stub.c, which stands in
for the HIP runtime (allocations from a budget on the host, kernels that do
nothing), so device memory can be short at any chosen point."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROW = 448  # bytes of a cell's row for the face flux kernel


@pytest.fixture(scope="session")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip_stub") / "libamdhip64.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-I/opt/rocm/include", "-Wl,-soname,libamdhip64.so.7", "-o", so,
                    os.path.join(HERE, "hip_stub.c")], check=True)
    return so


def _apart(stub, case):
    """Run a function of this file in a process that has the stub for a HIP runtime."""
    code = (f"import sys; sys.path.insert(0, {ROOT!r})\n"
            f"from tests import test_host_side as t\n"
            f"t.{case}(t.Stub({stub!r}))\nprint('case done')\n")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("case done\n"), r.stdout + r.stderr


class Stub:
    def __init__(self, so):
        self.L = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)  # found by its name when the library asks for HIP
        self.L.stub_used.restype = ctypes.c_size_t
        self.L.stub_budget.argtypes = [ctypes.c_size_t]
        self.L.stub_waits.restype = self.L.stub_launches.restype = self.L.stub_copies.restype = ctypes.c_long
        self.L.hipHostMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_uint]

    def used(self):
        return self.L.stub_used()

    def budget(self, n=None):
        self.L.stub_budget(ctypes.c_size_t(-1).value if n is None else n)

    def waits(self):
        return self.L.stub_waits()

    def copies(self):
        return self.L.stub_copies()

    def pinned(self, shape, dtype=np.float64):
        n, p = int(np.prod(shape)) * np.dtype(dtype).itemsize, ctypes.c_void_p()
        assert self.L.hipHostMalloc(ctypes.byref(p), n, 0) == 0
        return np.frombuffer((ctypes.c_char * n).from_address(p.value), dtype=dtype).reshape(shape)


def _random_mesh(n, nface, seed=1):
    """Faces between random pairs of cells (no geometry) and complete cell lists."""
    from fvmhd3d_amd.mesh import FACE_DTYPE
    rng = np.random.default_rng(seed)
    faces = np.zeros(nface, dtype=FACE_DTYPE)
    assert faces.itemsize == 56
    faces["s1"] = rng.integers(0, n, nface)
    faces["s2"] = (faces["s1"] + rng.integers(1, n, nface)) % n
    cell = np.concatenate([faces["s1"], faces["s2"]])
    order = np.argsort(cell, kind="stable")
    off = np.zeros(n + 1, np.int32)
    off[1:] = np.cumsum(np.bincount(cell, minlength=n))
    return faces, off, (order % nface).astype(np.int32), np.ones(n)


def case_rows_come_last(S):
    from fvmhd3d_amd import gpu as G
    n = 20000
    mesh = _random_mesh(n, 150000)

    def setup(budget=None):
        S.budget()
        ctx = G.Context()
        S.budget(budget)
        ctx.substep_setup(*mesh)
        return ctx

    ctx = setup()
    full = S.used()
    ctx.close()
    assert S.used() == 0
    # room for everything but the rows: the setup goes without them
    ctx = setup(full - ROW * n)
    assert S.used() == full - ROW * n
    ctx.close()
    with pytest.raises(G.FvmError):
        setup(full - ROW * n - 1)


def case_rows_are_given_back(S):
    from fvmhd3d_amd import gpu as G
    n = 20000
    ctx = G.Context()
    ctx.substep_setup(*_random_mesh(n, 150000))
    full = S.used()
    S.budget(full + (1 << 20))
    ctx.upload_mesh(n, n, 0, *_random_mesh(n, 150000))  # stages its face records: 56 bytes a face
    assert abs(S.used() - (full - ROW * n + 56 * 150000)) < 256
    ctx.close()


@pytest.mark.parametrize("case", ["case_rows_come_last", "case_rows_are_given_back"])
def test_optional_rows_yield_to_what_a_call_needs(stub, case):
    """The face flux kernel reads its cells from rows where there is memory for them
    (448 bytes a cell); without them it reads the fields.  fvm_substep_setup needs
    no more memory than its other buffers, and a later allocation that fails gets
    the rows' memory."""
    _apart(stub, case)


def case_setup_of_a_larger_mesh(S):
    from fvmhd3d_amd import gpu as G
    n = 20000
    mesh = _random_mesh(n, 150000)
    ctx = G.Context()
    ctx.upload_mesh(n, n, 0, *mesh)
    ctx.substep_setup(*mesh)
    assert ctx.L.fvm_compute_reconstruction(ctx.h) == G.FVM_OK  # every buffer is where it was
    before, full = S.used(), None
    for short in (False, True):
        c = G.Context()
        c.upload_mesh(1000, 1000, 0, *_random_mesh(1000, 8000))
        if short:  # for the last of the buffers that the path cannot do without
            S.budget(full - ROW * n - 1)
            with pytest.raises(G.FvmError):
                c.substep_setup(*mesh)
        else:
            c.substep_setup(*mesh)
            full = S.used()
        assert c.L.fvm_compute_reconstruction(c.h) == G.FVM_ESTATE
        c.close()
        assert S.used() == before
    ctx.close()


def test_setup_of_a_larger_mesh_ends_the_one_before(stub):
    """fvm_substep_setup makes room for its mesh in the context's buffers: where one of
    them moves, or cannot be had, the mesh uploaded before is gone."""
    _apart(stub, "case_setup_of_a_larger_mesh")


def case_one_wait_a_field(S):
    from fvmhd3d_amd import gpu as G
    n = 20000
    ctx = G.Context()
    ctx.upload_mesh(n, n, 0, *_random_mesh(n, 150000))
    ctx.substep_setup(*_random_mesh(n, 150000))
    for name, (_, width, kind) in G.FIELDS.items():
        a = np.zeros((n, width), np.int32 if kind == "i" else np.float64)
        for call in (ctx.upload, ctx.download, ctx.substep_upload):
            if call == ctx.substep_upload and name not in ("w", "U", "pos", "tend", "bnd"):
                continue
            before = S.waits()
            call(name, a) if call != ctx.download else call(name)
            assert S.waits() == before + 1, (name, call.__name__)
    ctx.close()


def test_field_transfers_wait_once(stub):
    """A field of less than 8 MiB goes up or down with one wait for the stream."""
    _apart(stub, "case_one_wait_a_field")


def case_pinned_arrays_are_not_staged(S):
    from fvmhd3d_amd import gpu as G
    n = 120000  # a ten-wide field: 9.6 MB, two slots
    ctx = G.Context()
    ctx.upload_mesh(n, n, 0, *_random_mesh(n, 130000))
    for new, copies in ((np.zeros, 2), (S.pinned, 1)):
        a = new((n, 10))
        for call in (ctx.L.fvm_upload_field, ctx.L.fvm_download_field):
            before = S.copies()
            ctx._chk(call(ctx.h, G.FIELDS["w"][0], a.ctypes.data, n))
            assert S.copies() == before + copies
    n = 40000  # faces: three chunks of three copies each, or the eight arrays
    shapes = [((n, 3), float), ((n, 10), float), ((n, 10), float), (n, np.int32), ((n, 3), float), (n, float), (n, float),
              ((n, 10), float)]
    for new, copies in ((np.zeros, 9), (S.pinned, 8)):
        arrays = [new(*s) for s in shapes]
        before = S.copies()
        ctx._chk(ctx.L.fvm_compute_flux(ctx.h, n, *[a.ctypes.data for a in arrays]))
        assert S.copies() == before + copies
    ctx.close()


def test_pinned_arrays_are_copied_directly(stub):
    """Arrays that are pinned themselves go to and from the device in one copy each,
    not through the pinned slots."""
    _apart(stub, "case_pinned_arrays_are_not_staged")


def case_flux_without_staging(S):
    from fvmhd3d_amd import gpu as G
    ctx = G.Context()

    def arrays(n):
        return [np.zeros((n, 3)), np.zeros((n, 10)), np.zeros((n, 10)), np.zeros(n, np.int32), np.zeros((n, 3)), np.zeros(n),
                np.zeros(n), np.zeros((n, 10))]

    def run(a):
        ctx._chk(ctx.L.fvm_compute_flux(ctx.h, len(a[0]), *[x.ctypes.data for x in a]))

    before = S.used()
    for n in (300, 5000, 32767):
        run(arrays(n))
    assert S.used() == before  # these routes have no device staging
    S.budget(before)
    for n in (32768, 100000):
        run(arrays(n))
    assert S.used() == before
    a = arrays(40000)
    a[7] = a[1]  # the flux in Wi
    with pytest.raises(G.FvmError):
        run(a)
    S.budget()
    run(a)
    assert S.used() == before + 308 * 40000
    ctx.close()


def test_flux_batches_without_device_memory(stub):
    """computeFlux allocates device staging for the routes that use it only, and takes
    a batch in pieces where there is no memory for it; a batch computed in its
    inputs' memory needs it and is refused."""
    _apart(stub, "case_flux_without_staging")
