"""GPU: tuning a mixed-precision context changes its speed, not its results.

Another order of the sums (another depth of slab, split over waves, or particle
split) moves the last bits of the float products, so contexts tuned one after the
other have to use one order whatever the timings said.  Bitwise, at grids where the
fastest shapes of two orders lie within a per cent of each other (the tuner's picks
changed from context to context there) and at one whose sides are not multiples of
32."""
import numpy as np
import pytest

from tertia_amd.params import PRECISIONS, small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["mixed32", "bf16x3", "bf16x6"])
@pytest.mark.parametrize("ny,nz", [(128, 128), (256, 256), (48, 64), (208, 112)])
def test_tuned_contexts_agree(prec, ny, nz):
    import ctypes
    from tertia_amd import _lib
    from tertia_amd.mesh import Mesh
    p = small(ny=ny, nz=nz, nslices=4, precision=PRECISIONS[prec])
    rng = np.random.default_rng(ny + nz)
    names = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "Jx", "Jy")
    planes = [rng.standard_normal((nz, ny)) for _ in names]
    first = None
    for i in range(8):
        m = Mesh(p, history=("Ex", "Psi"))
        try:
            m.autotune(1 + i % 3)
            got = {"split": m.particle_split}
            for n in (1, 2, 3, 6, 8):
                for f, x in zip(names, planes):
                    m.set_field(f, x)
                kinds = (ctypes.c_int * n)(*[q % 2 for q in range(n)])
                src = (ctypes.c_void_p * n)(*[m.layer_ptr(f) for f in names[:n]])
                dst = (ctypes.c_void_p * n)(*[m.layer_ptr(f, "P") for f in names[:n]])
                _lib.check(m.L.qss_transform2d_batched(
                    m.h, n, kinds, kinds, ctypes.cast(src, _lib._dpp),
                    ctypes.cast(dst, _lib._dpp), 1.0), "qss_transform2d_batched")
                for f in names[:n]:
                    got[n, f] = m.get_field(f, "P")
            m.MoveAllSplitLayers()
            for f in ("Ex", "Psi"):
                got[f] = np.stack([m.history(f, s) for s in range(p.nslices)])
        finally:
            m.close()
        if first is None:
            first = got
        for k in got:
            assert np.array_equal(first[k], got[k]), (i, k)
