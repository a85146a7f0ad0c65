"""Callers' arrays in pinned memory: computeFlux batches and field transfers give
what pageable arrays give, bit for bit, at the sizes of every route."""
import ctypes

import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from tests.helpers import workload_mesh
from tests.test_zz_no_alloc import _faces

pytestmark = pytest.mark.gpu


@pytest.fixture
def pinned():
    G.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the library's own
    hip.hipHostMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_uint]
    hip.hipHostFree.argtypes = [ctypes.c_void_p]
    held = []

    def copy(a):
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), a.nbytes, 0) == 0
        held.append(p)
        b = np.frombuffer((ctypes.c_char * a.nbytes).from_address(p.value), dtype=a.dtype).reshape(a.shape)
        b[...] = a
        return b

    yield copy
    for p in held:
        hip.hipHostFree(p)


@pytest.mark.parametrize("n", [3000, 16383, 16384, 32768, 70001])
def test_flux_batches_in_pinned_arrays(pinned, n):
    faces = _faces(n, n)
    ctx = G.Context()
    want = ctx.compute_flux(*faces)
    arrays = [pinned(a) for a in (*faces, np.zeros(n), np.zeros(n), np.zeros((n, 10)))]
    ctx._chk(ctx.L.fvm_compute_flux(ctx.h, n, *[a.ctypes.data for a in arrays]))
    for x, y in zip(arrays[5:], want):
        assert np.array_equal(x, y)
    mixed = [a.copy() if k % 2 else pinned(a) for k, a in enumerate((*faces, np.zeros(n), np.zeros(n), np.zeros((n, 10))))]
    ctx._chk(ctx.L.fvm_compute_flux(ctx.h, n, *[a.ctypes.data for a in mixed]))
    for x, y in zip(mixed[5:], want):
        assert np.array_equal(x, y)
    ctx.close()


@pytest.mark.parametrize("n", [12, 49])
def test_fields_in_pinned_arrays(pinned, n):
    m = workload_mesh("lattice", n)
    ctx = G.Context()
    ctx.upload_mesh(m.ncell, m.ncell, 0, m.faces, m.cell_off, m.cell_face, m.volume)
    w = np.random.default_rng(n).standard_normal((m.ncell, 10))
    a, b = pinned(w), pinned(np.zeros_like(w))
    ctx._chk(ctx.L.fvm_upload_field(ctx.h, G.FIELDS["w"][0], a.ctypes.data, m.ncell))
    ctx._chk(ctx.L.fvm_download_field(ctx.h, G.FIELDS["w"][0], b.ctypes.data, m.ncell))
    assert np.array_equal(b, w) and np.array_equal(ctx.download("w"), w)
    ctx.close()
