"""The face flux kernel reads its cells from rows from 131072 active faces on:
both sides of that size, cell counts that leave a block of 64 rows part empty,
moving faces, boundary cells of every kind on either side of a face, and both
storage types, against the oracle at the bar of the parity tests."""
import numpy as np
import pytest

from fvmhd3d_amd import gpu as G
from tests.helpers import alfven_state, perturb_gradients
from tests.test_gpu_parity import _run_pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows,storage", [(25, False, "f64"), (26, True, "f64"), (26, True, "shipped"), (27, True, "f64")])
def test_face_flux_from_rows(n, rows, storage):
    st = perturb_gradients(alfven_state(n, moving=True))
    assert (len(st.faces) >= 131072) == rows
    if n != 27:
        idx = np.random.default_rng(11).choice(st.np, size=400, replace=False)
        st.bnd[idx] = np.tile(np.array([1, 2, 3, 4], dtype=np.int32), 100)
    _run_pipeline(storage, G.LIMITER_SHIPPED, st)
