"""GPU: the context-free transform on both sides of its rule for short y sides with a
factor of 11 or 13 (dense below 56) against the oracle, at the transform tests' bound."""
import ctypes

import numpy as np
import pytest

from tests.helpers import max_rel
from tertia_amd.params import small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,ny", [(22, 22), (52, 52), (64, 26), (26, 64), (128, 44), (256, 52),
                                   (48, 66), (35, 22)])
def test_short_rows_of_large_radix(oracle_mod, nz, ny):
    from tertia_amd.mesh import Mesh
    m = Mesh(small(ny=ny, nz=nz, nslices=1), history=())
    try:
        x = np.random.default_rng(nz + 1000 * ny).standard_normal((nz, ny))
        for kz in (0, 1):
            for ky in (0, 1):
                ref = 0.25 * oracle_mod.transform2d(x, kz, ky, use_fft=False, nthreads=4)
                m.set_field("Rho", x)
                for dst in ("Jx", "Rho"):
                    assert m.L.qss_transform2d_noalloc(ny, nz, kz, ky, m.layer_ptr("Rho"),
                                                       m.layer_ptr(dst), 0.25,
                                                       ctypes.c_void_p(m.stream)) == 0
                got = m.get_field("Jx")
                assert max_rel(got, ref) < 1e-13, (kz, ky)
                assert np.array_equal(m.get_field("Rho"), got)
    finally:
        m.close()
