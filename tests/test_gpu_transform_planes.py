"""GPU: a batch of transforms whose outputs are other entries' inputs.  Each result is
that of the inputs as they were before the call, on grids small enough for the
one-launch form and on larger ones, for line transforms, dense tables and the
mixed modes, and for planes that overlap in part."""
import ctypes

import numpy as np
import pytest

from tests.helpers import max_rel
from tertia_amd.params import PRECISIONS, small

pytestmark = pytest.mark.gpu

NAMES = ("Ex", "Ey", "Ez", "Bx", "By")


@pytest.mark.parametrize("prec", ["fp64", "mixed32"])
@pytest.mark.parametrize("ny,nz", [(32, 32), (64, 48), (64, 64), (80, 64), (128, 96)])
@pytest.mark.parametrize("to", [(1, 0), (1, 2, 3, 4, 0), (0, 2, 1)])
def test_outputs_on_other_inputs(ny, nz, prec, to):
    from tertia_amd import _lib
    from tertia_amd.mesh import Mesh
    n = len(to)
    rng = np.random.default_rng(ny + nz + n)
    x = [rng.standard_normal((nz, ny)) for _ in range(n)]
    kz, ky = [q % 2 for q in range(n)], [q // 2 % 2 for q in range(n)]
    m = Mesh(small(ny=ny, nz=nz, nslices=1, precision=PRECISIONS[prec]), history=())
    try:
        ref = [m.transform2d(x[q], kz[q], ky[q]) for q in range(n)]
        for _ in range(4):
            for f, a in zip(NAMES, x):
                m.set_field(f, a)
            src = [m.layer_ptr(f) for f in NAMES[:n]]
            _lib.check(m.L.qss_transform2d_batched(
                m.h, n, (ctypes.c_int * n)(*kz), (ctypes.c_int * n)(*ky),
                ctypes.cast((ctypes.c_void_p * n)(*src), _lib._dpp),
                ctypes.cast((ctypes.c_void_p * n)(*[src[q] for q in to]), _lib._dpp), 1.0),
                "qss_transform2d_batched")
            for q in range(n):
                got = m.get_field(NAMES[to[q]])
                # one form or the other of the same transform
                assert max_rel(got, ref[q]) < (1e-13 if prec == "fp64" else 3e-6), q
    finally:
        m.close()


def test_output_half_on_another_input():
    from tertia_amd import _lib
    from tertia_amd.mesh import Mesh
    ny, nz = 64, 64
    m = Mesh(small(ny=ny, nz=nz, nslices=5), history=("Ex",))   # five planes in a row
    try:
        x = np.random.default_rng(5).standard_normal((5, nz, ny))
        for s in range(5):
            m.set_history("Ex", s, x[s])
        half = ny * nz * 8 // 2
        base = m.history_ptr("Ex")
        src = (base, base + 4 * half)               # planes 0 and 2
        dst = (base + 3 * half, base + 7 * half)    # from 1.5 (half of it on plane 2) and 3.5
        kinds = (ctypes.c_int * 2)(0, 1)
        _lib.check(m.L.qss_transform2d_batched(
            m.h, 2, kinds, kinds, ctypes.cast((ctypes.c_void_p * 2)(*src), _lib._dpp),
            ctypes.cast((ctypes.c_void_p * 2)(*dst), _lib._dpp), 1.0), "qss_transform2d_batched")
        flat = np.concatenate([m.history("Ex", s).reshape(-1) for s in range(5)])
        for q, (plane, at) in enumerate(((0, 3), (2, 7))):
            got = flat[at * ny * nz // 2:][:ny * nz].reshape(nz, ny)
            assert max_rel(got, m.transform2d(x[plane], q, q)) < 1e-13, q
    finally:
        m.close()
