"""computeFlux batches whose outputs lie in the memory of their inputs, at the
sizes of every route: the results are those of separate arrays, bit for bit."""
import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from tests.test_zz_no_alloc import _faces

pytestmark = pytest.mark.gpu

PIN = (1 << 20) // 308
CHUNK = 16384


@pytest.mark.parametrize("n,noalloc", [(300, False), (PIN + 1, False), (2 * CHUNK - 1, False), (9 * CHUNK - 7, False),
                                       (300, True), (2 * CHUNK - 1, True)])
def test_outputs_in_input_memory(n, noalloc):
    faces = _faces(n, n)
    ctx = G.Context()
    want = ctx.compute_flux(*faces)
    fn = ctx.L.fvm_compute_flux_noalloc if noalloc else ctx.L.fvm_compute_flux
    for case in ("narrow outputs in wij and normal", "flux in Wi", "flux across Wi and Wj"):
        wij, Wi, Wj, jbnd, nrm = [a.copy() for a in faces]
        both = np.concatenate([Wi, Wj])
        Wi, Wj = both[:n], both[n:]
        psi, Bn, flux = np.empty(n), np.empty(n), np.empty((n, 10))
        if case == "narrow outputs in wij and normal":
            psi, Bn = wij.reshape(-1)[n:2 * n], nrm.reshape(-1)[2 * n:]
        elif case == "flux in Wi":
            flux = Wi
        else:
            flux = both[n // 2:n // 2 + n]
        ctx._chk(fn(ctx.h, n, *[a.ctypes.data for a in (wij, Wi, Wj, jbnd, nrm, psi, Bn, flux)]))
        for x, y in zip((psi, Bn, flux), want):
            assert np.array_equal(x, y), case
    ctx.close()
