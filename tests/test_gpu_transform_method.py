"""GPU: the transform method can be left and taken up again.  A context starts with line
transforms where it has them; a GEMM method replaces them, and setting what
transform_in_use returned before (or lines) gives the first results' bits back, in
transforms and in sweeps, eager and replayed."""
import numpy as np
import pytest

from tertia_amd.params import PRECISIONS, small

pytestmark = pytest.mark.gpu

DENSE, FACTORED, LINES = 0, 1, 2


def results(m, p, x):
    out = [m.transform2d(x, kz, ky) for kz in (0, 1) for ky in (0, 1)]
    out.append(m.MoveAllSplitLayers())
    out += [m.history("Ex", s) for s in range(p.nslices)]
    return out


# compiled lengths, small planes, loose chains, a line pass beside a GEMM pass, dense
# lines in layer steps only
@pytest.mark.parametrize("ny,nz", [(256, 256), (64, 48), (200, 312), (121, 256), (33, 35)])
@pytest.mark.parametrize("graph", [False, True])
def test_lines_come_back(ny, nz, graph):
    from tertia_amd.mesh import Mesh
    p = small(ny=ny, nz=nz, nslices=7)
    x = np.random.default_rng(ny).standard_normal((nz, ny))
    m = Mesh(p, history=("Ex",))
    try:
        m.enable_graph(graph)
        assert m.transform_in_use == LINES
        form = m.transform_method
        first = results(m, p, x)
        for method in [DENSE] + ([FACTORED] if form == FACTORED else []):
            kept = m.transform_in_use
            m.transform_method = method
            assert m.transform_in_use == method and m.transform_method == method
            other = results(m, p, x)
            assert not all(np.array_equal(a, b) for a, b in zip(first, other))
            m.transform_method = kept
            assert m.transform_in_use == LINES and m.transform_method == form
            for i, (a, b) in enumerate(zip(first, results(m, p, x))):
                assert np.array_equal(a, b), i
        m.set_gemm_variant(1)   # a forced tile shape takes the lines out of use, too
        assert m.transform_in_use == form
        m.set_gemm_variant(-1)
        assert m.transform_in_use == LINES
    finally:
        m.close()


@pytest.mark.parametrize("kw", [dict(ny=32, nz=32, precision=PRECISIONS["mixed32"]),
                                dict(ny=313, nz=35)])
def test_lines_refused_where_there_are_none(kw):
    from tertia_amd._lib import QssError
    from tertia_amd.mesh import Mesh
    m = Mesh(small(nslices=1, **kw), history=())
    try:
        assert m.transform_in_use == m.transform_method == DENSE
        with pytest.raises(QssError):
            m.transform_method = LINES
        m.transform_method = m.transform_in_use
        with pytest.raises(QssError):
            m.transform_method = 3
    finally:
        m.close()
