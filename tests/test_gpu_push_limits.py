"""GPU: momenta whose square leaves the range of a double.  The Lorentz factor is then
infinite and its reciprocal 0, as in the reference's division: the particle is at
rest, deposits its density and no current, and the pass goes on without an error.
Momenta just inside the range move like any other."""
import numpy as np
import pytest

from tests.helpers import max_rel, smooth_field
from tertia_amd.params import small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("big", [1e150, 1.3e154, 1.4e154, 1e200, 1e300])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_square_overflows(oracle_mod, big, axis):
    from tertia_amd.mesh import Mesh
    ny = nz = 32
    rng = np.random.default_rng(axis)
    p = small(ny=ny, nz=nz, nslices=2, ppc_y=1, ppc_z=2)
    n = ny * nz
    mom = rng.uniform(-0.1, 0.1, size=(3, n))
    # along x backwards: forwards 1 - Vx rounds to 0 for any momentum past 1e8
    mom[axis, ::5] = -big
    cell = np.arange(n)
    parts = ((cell % ny).astype(np.int32), (cell // ny).astype(np.int32),
             rng.uniform(0.2, 0.8, n), rng.uniform(0.2, 0.8, n), *mom,
             np.arange(n, dtype=np.int64))
    fields = {f: smooth_field(rng, nz, ny, 0.1) for f in ("Ex", "Ey", "Ez", "Bx", "By", "Bz")}
    m, o = Mesh(p, history=()), oracle_mod.Oracle(p, history=())
    try:
        for f, F in fields.items():
            for lay, which in (("C", 0), ("P", 1)):
                o.set_field(f, F, which=which)
                m.set_field(f, F, layer=lay)
        o.set_particles(*parts)
        m.set_particles(*parts)
        for full in (0, 1):
            o.push_deposit(full)
            m.MoveParticlesLayerSplit(0, 0, full)
            for f in ("Jx", "Jy", "Jz", "Rho"):
                assert np.isfinite(o.get_field(f)).all()
                assert max_rel(m.get_field(f), o.get_field(f)) <= 1e-13, f
    finally:
        m.close()
