"""GPU: where a grid's line transforms lose to the GEMMs, the GEMMs run: the bits are
then those of the context with a GEMM method set."""
import ctypes

import numpy as np
import pytest

from tests.helpers import max_rel
from tertia_amd.params import small

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")


@pytest.mark.parametrize("ny,nz,n,lines", [
    (352, 352, 1, False), (352, 352, 2, False), (352, 352, 3, True),     # full tiles
    (352, 64, 3, False), (64, 352, 1, True),     # such a chain along z costs nothing
    (198, 198, 1, False), (198, 198, 6, True),
    (288, 288, 1, True), (200, 312, 1, True)])
def test_rows_of_large_radix(oracle_mod, ny, nz, n, lines):
    from tertia_amd import _lib
    from tertia_amd.mesh import Mesh
    m = Mesh(small(ny=ny, nz=nz, nslices=1, ppc_y=1, ppc_z=1), history=())
    try:
        rng = np.random.default_rng(ny + nz + n)
        x = [rng.standard_normal((nz, ny)) for _ in range(n)]
        kinds = (ctypes.c_int * n)(*[q % 2 for q in range(n)])

        def batch():
            for f, a in zip(FIELDS, x):
                m.set_field(f, a)
            _lib.check(m.L.qss_transform2d_batched(
                m.h, n, kinds, kinds,
                ctypes.cast((ctypes.c_void_p * n)(*[m.layer_ptr(f) for f in FIELDS[:n]]), _lib._dpp),
                ctypes.cast((ctypes.c_void_p * n)(*[m.layer_ptr(f, "P") for f in FIELDS[:n]]),
                            _lib._dpp), 1.0), "qss_transform2d_batched")
            return [m.get_field(f, "P") for f in FIELDS[:n]]
        got = batch()
        ref = oracle_mod.transform2d(x[-1], kinds[n - 1], kinds[n - 1], use_fft=False, nthreads=4)
        assert max_rel(got[-1], ref) < 1e-13
        m.transform_method = m.transform_method   # the GEMM form
        same = all(np.array_equal(a, b) for a, b in zip(got, batch()))
        assert same != lines
    finally:
        m.close()


@pytest.mark.parametrize("ny,nz,lines", [
    (64, 179, True), (64, 181, False), (100, 255, False), (126, 201, False),   # y a chain
    (320, 255, True), (121, 143, True), (121, 145, False),                     # a long one; dense
    (129, 97, False)])
def test_dense_columns_in_layer_steps(oracle_mod, ny, nz, lines):
    """Layers of a grid whose z side has no chain: lines on one side of the rule, the
    GEMMs' bits on the other."""
    from tertia_amd.mesh import Mesh
    p = small(ny=ny, nz=nz, nslices=4)
    m, o = Mesh(p, history=("Ex",)), oracle_mod.Oracle(p, history=("Ex",))
    try:
        runs = []
        for _ in range(2):
            m.MoveAllSplitLayers()
            runs.append(np.stack([m.history("Ex", s) for s in range(p.nslices)]))
            m.transform_method = m.transform_method   # the GEMM form
        o.sweep()
        ref = np.stack([o.history("Ex", s) for s in range(p.nslices)])
        assert np.linalg.norm(runs[0] - ref) <= 1e-10 * np.linalg.norm(ref)
        assert np.array_equal(*runs) != lines
    finally:
        m.close()
        o.close()
