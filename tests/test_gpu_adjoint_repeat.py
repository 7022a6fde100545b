"""GPU: the reverse sweep gives the same gradient bits when it is run again, at every
form of its transposed gather: lists of the small and the large sorting network (1, 5
and 8 particles per cell) and sorted chunks (9, 16, 25).  Events reach a list by
atomics, in an order that differs from run to run; their sum must not."""
import numpy as np
import pytest

from tests.test_gpu_adjoint import WIN_SMALL, adjoint_grad, small_bins

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ppc_y,ppc_z,split", [(1, 1, 1), (1, 5, 1), (2, 4, 2), (3, 3, 1), (4, 4, 4),
                                               (5, 5, 2)])
def test_gradient_bits_repeat(ppc_y, ppc_z, split):
    from tertia_amd.mesh import Mesh
    p = small_bins(ppc_y=ppc_y, ppc_z=ppc_z)
    m = Mesh(p, history=("Ex",))
    try:
        m.particle_split = split
        runs = [adjoint_grad(m, p, 56, every, WIN_SMALL) for every in (8, 8, 8, 0, 0)]
    finally:
        m.close()
    assert np.abs(runs[0][1]).max() > 0
    for loss, g, ex in runs[1:3]:
        assert loss == runs[0][0] and np.array_equal(ex, runs[0][2])
        assert np.array_equal(g, runs[0][1])
    assert np.array_equal(runs[3][1], runs[4][1])
