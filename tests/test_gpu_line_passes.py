"""GPU: runtime chains of three and four passes of the line transforms (the middle
passes trade the exchange's sides), with radices up to 8 and above, on either axis.

Transforms, one plane and eight at a time, against the oracle at the transform tests'
bound (1e-13 of the largest result); sweeps, which run the rows with the Guess and
Iterate maps and the columns with their epilogues, against the oracle at the small
sweeps' bound (rel-L2 1e-10)."""
import ctypes

import numpy as np
import pytest

from tests.helpers import max_rel
from tertia_amd.params import small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,ny", [
    (224, 400), (400, 224), (480, 288), (288, 504),     # three passes of at most 8
    (270, 378), (378, 324), (324, 270),                 # four
    (352, 440), (416, 450), (500, 352), (440, 416), (450, 500),   # three with 9, 10, 11, 13
    (208, 286), (312, 198)])                            # two with those
def test_long_chains_vs_oracle(oracle_mod, nz, ny):
    from tertia_amd import _lib
    from tertia_amd.mesh import Mesh
    fields = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "Jx", "Jy")
    m = Mesh(small(ny=ny, nz=nz, nslices=1, ppc_y=1, ppc_z=1), history=())
    try:
        x = np.random.default_rng(ny + 1000 * nz).standard_normal((nz, ny))
        kinds = [(kz, ky) for kz in (0, 1) for ky in (0, 1)]
        ref = {k: oracle_mod.transform2d(x, *k, use_fft=False, nthreads=4) for k in kinds}
        for k in kinds:
            assert max_rel(m.transform2d(x, *k, 0.25), 0.25 * ref[k]) < 1e-13, k
        for f in fields:
            m.set_field(f, x)
        kk = [kinds[q % 4] for q in range(8)]
        _lib.check(m.L.qss_transform2d_batched(
            m.h, 8, (ctypes.c_int * 8)(*[k[0] for k in kk]), (ctypes.c_int * 8)(*[k[1] for k in kk]),
            ctypes.cast((ctypes.c_void_p * 8)(*[m.layer_ptr(f) for f in fields]), _lib._dpp),
            ctypes.cast((ctypes.c_void_p * 8)(*[m.layer_ptr(f, "P") for f in fields]), _lib._dpp),
            1.0), "qss_transform2d_batched")
        for f, k in zip(fields, kk):
            assert max_rel(m.get_field(f, "P"), ref[k]) < 1e-13, (f, k)
    finally:
        m.close()


@pytest.mark.parametrize("ny,nz,kw", [
    (224, 30, {}), (30, 224, {"n_iter": 1}), (480, 20, {}), (20, 480, {}), (288, 18, {}),
    (162, 24, {}), (24, 162, {}), (270, 16, {"n_iter": 0}), (16, 378, {}),   # four passes
    (352, 16, {}), (16, 352, {}), (450, 16, {}), (16, 440, {}), (26, 44, {})])   # 9, 11, 13
def test_sweep_on_long_chains_vs_oracle(oracle_mod, ny, nz, kw):
    from tertia_amd.mesh import Mesh
    p = small(ny=ny, nz=nz, nslices=8, **kw)
    fields = ("Ex", "Ey", "Ez", "By", "Psi")
    m = Mesh(p, history=fields)
    o = oracle_mod.Oracle(p, use_fft=False, nthreads=8, history=fields)
    try:
        rg = m.MoveAllSplitLayers()
        st, ro = o.sweep()
        assert st == 0
        assert np.abs(rg - ro).max() < 1e-9
        for f in fields:
            G = np.stack([m.history(f, s) for s in range(p.nslices)])
            R = np.stack([o.history(f, s) for s in range(p.nslices)])
            e = float(np.linalg.norm(G - R) / np.linalg.norm(R))
            assert e <= 1e-10, (f, e)
    finally:
        m.close()
        o.close()
