"""GPU: the line-transform kernels (line.hip) at the edges of their shapes: lengths
compiled in (two and three passes), loose chains with and without a radix above 8,
the dense table (odd lengths, prime factors above 13) on either axis, partial
strips of columns, and planes small enough for one work-group.

Transforms against the oracle at the transform tests' bound (1e-13 of the largest
result); sweeps, which run the fused Guess and Iterate rows, against the oracle at
the small sweeps' bound (rel-L2 1e-10)."""
import numpy as np
import pytest

from tests.helpers import max_rel
from tertia_amd.params import QSS_SHAPE_NGP_REF, small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,ny", [(32, 40), (64, 48), (80, 96), (192, 160), (512, 320), (200, 312),
                                   (242, 208), (484, 250), (512, 512)])
def test_line_transform_vs_oracle(oracle_mod, nz, ny):
    from tertia_amd.mesh import Mesh
    m = Mesh(small(ny=ny, nz=nz, nslices=1), history=())
    try:
        x = np.random.default_rng(ny + 1000 * nz).standard_normal((nz, ny))
        for kz in (0, 1):
            for ky in (0, 1):
                ref = oracle_mod.transform2d(x, kz, ky, use_fft=False, nthreads=4)
                assert max_rel(m.transform2d(x, kz, ky, 0.25), 0.25 * ref) < 1e-13, (kz, ky)
    finally:
        m.close()


@pytest.mark.parametrize("ny,nz,kw", [
    (32, 32, {}), (48, 80, {}), (192, 64, {"n_iter": 0}), (320, 160, {}),   # compiled lengths
    (36, 100, {}), (52, 66, {"n_iter": 1}),                                # loose chains
    (33, 48, {}), (48, 35, {}), (121, 97, {"shape": QSS_SHAPE_NGP_REF}), (34, 74, {}),   # dense
    (128, 256, {}), (17, 19, {})])
def test_sweep_on_line_grids_vs_oracle(oracle_mod, ny, nz, kw):
    from tertia_amd.mesh import Mesh
    p = small(ny=ny, nz=nz, nslices=12, **kw)
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
            print(ny, nz, f, "%.1e" % e, flush=True)
            assert e <= 1e-10, (f, e)
    finally:
        m.close()
        o.close()


@pytest.mark.parametrize("nz,ny", [(32, 32), (64, 48), (40, 128), (312, 200), (512, 512),
                                   (8, 4), (66, 36), (26, 286),                  # lines
                                   (194, 256), (17, 19), (31, 64)])              # dense
def test_noalloc_lines_vs_oracle(oracle_mod, nz, ny):
    """The context-free transform on both sides of its rule (lengths compiled in, loose
    chains, down to the shortest; a side without a chain makes both dense), out of place and in place; its tables
    are built on the device."""
    import ctypes
    from tertia_amd.mesh import Mesh
    m = Mesh(small(ny=ny, nz=nz, nslices=2), history=())
    try:
        x = np.random.default_rng(nz + 1000 * ny).standard_normal((nz, ny))
        s = ctypes.c_void_p(m.stream)
        for kz in (0, 1):
            for ky in (0, 1):
                ref = 0.25 * oracle_mod.transform2d(x, kz, ky, use_fft=False, nthreads=4)
                m.set_field("Rho", x)
                for dst in ("Jx", "Rho"):
                    assert m.L.qss_transform2d_noalloc(ny, nz, kz, ky, m.layer_ptr("Rho"),
                                                       m.layer_ptr(dst), 0.25, s) == 0
                got = m.get_field("Jx")
                assert max_rel(got, ref) < 1e-13, (kz, ky)
                assert np.array_equal(m.get_field("Rho"), got)
    finally:
        m.close()


@pytest.mark.parametrize("nz,ny", [(35, 64), (64, 35), (97, 200), (313, 256), (192, 313), (19, 32)])
def test_one_line_pass_vs_oracle(oracle_mod, nz, ny):
    """One side with a chain, the other dense: a line pass and a GEMM pass, of one plane,
    of a batch and of the context-free call."""
    import ctypes
    from tertia_amd.mesh import Mesh
    m = Mesh(small(ny=ny, nz=nz, nslices=1), history=())
    try:
        x = np.random.default_rng(ny + 1000 * nz).standard_normal((nz, ny))
        for kz in (0, 1):
            for ky in (0, 1):
                ref = 0.25 * oracle_mod.transform2d(x, kz, ky, use_fft=False, nthreads=4)
                assert max_rel(m.transform2d(x, kz, ky, 0.25), ref) < 1e-13, (kz, ky)
                m.set_field("Rho", x)
                assert m.L.qss_transform2d_noalloc(ny, nz, kz, ky, m.layer_ptr("Rho"),
                                                   m.layer_ptr("Jx"), 0.25,
                                                   ctypes.c_void_p(m.stream)) == 0
                assert max_rel(m.get_field("Jx"), ref) < 1e-13, (kz, ky)
    finally:
        m.close()


@pytest.mark.parametrize("ny,nz,kw", [(151, 96, {}), (64, 313, {"n_iter": 1}), (313, 35, {})])
def test_sweep_with_one_line_pass_vs_oracle(oracle_mod, ny, nz, kw):
    """Sides beyond the dense rows' limit: the layer step's transforms by passes, the
    push field and the residual in the column pass or in the GEMM."""
    from tertia_amd.mesh import Mesh
    p = small(ny=ny, nz=nz, nslices=8, **kw)
    m, o = Mesh(p, history=("Ex", "Psi")), oracle_mod.Oracle(p, history=("Ex", "Psi"))
    try:
        rg, ro = m.MoveAllSplitLayers(), o.sweep()
        for f in ("Ex", "Psi"):
            a = np.stack([m.history(f, s) for s in range(p.nslices)])
            b = np.stack([o.history(f, s) for s in range(p.nslices)])
            assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b), f
    finally:
        m.close()
