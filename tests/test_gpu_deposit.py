"""GPU: the tiled push's deposit at the edges of its branches: cells with one event,
with as many as the small and the large sorting network take (4 and 8) and one more
(the second network; the sort of a crowded round), rows of cells in the first half
of the window's cells only, in the second only and in both, CIC and NGP, and hot
particles that take several rounds.

Currents and density against the oracle at the push tests' bound (1e-13 of the
largest value: the same contributions, associated differently), and the same bits
when the pass is run again (the order in which events reach a cell's list differs
from run to run, their sum must not)."""
import numpy as np
import pytest

from tests.helpers import max_rel, smooth_field
from tertia_amd.params import QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF, small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF])
@pytest.mark.parametrize("rows", [(0, 6), (10, 16), (0, 16)])
@pytest.mark.parametrize("per_cell,hot", [(1, 0), (4, 0), (5, 0), (8, 0), (9, 0), (70, 0), (3, 8)])
def test_deposit_cell_counts(oracle_mod, shape, rows, per_cell, hot):
    from tertia_amd.mesh import Mesh
    ny = nz = 48
    rng = np.random.default_rng(per_cell + 100 * rows[0] + 1000 * rows[1])
    p = small(ny=ny, nz=nz, nslices=2, hx=0.4 if hot else 0.05, shape=shape, ppc_y=2, ppc_z=4)
    # whole cells of per_cell particles in the given rows of every tile, as many as fit
    cells = [j + ny * k for k in range(nz) for j in range(ny) if rows[0] <= k % 16 < rows[1]]
    cells = np.sort(rng.permutation(cells)[: ny * nz * 8 // per_cell])
    cell = np.repeat(cells, per_cell)
    n = len(cell)
    mom = rng.uniform(-0.1, 0.1, size=(3, n))
    if hot:
        # past one cell in a slice: several sub-steps
        mom[0, ::hot] = 3.0
        mom[1, ::hot] = rng.uniform(-4, 4, size=len(mom[1, ::hot]))
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
        runs = []
        for _ in range(2):
            m.set_particles(*parts)
            got = []
            for full in (0, 1):
                m.MoveParticlesLayerSplit(0, 0, full)
                got += [m.get_field(f) for f in ("Jx", "Jy", "Jz", "Rho")]
            runs.append(got)
        ref = []
        for full in (0, 1):
            o.push_deposit(full)
            ref += [o.get_field(f) for f in ("Jx", "Jy", "Jz", "Rho")]
        for g, r in zip(runs[0], ref):
            assert max_rel(g, r) <= 1e-13
        for a, b in zip(*runs):
            assert np.array_equal(a, b)
    finally:
        m.close()


@pytest.mark.parametrize("ny,nz,nsplit", [
    (16, 16, 1), (32, 16, 2), (16, 48, 4),   # one, two and three tiles on an axis
    (256, 256, 4), (272, 256, 2),            # one full round of the scan, and one tile row more
    (368, 368, 1)])                          # two rounds of two tiles a thread
def test_reorder_scan_edges(oracle_mod, ny, nz, nsplit):
    """The tile scan that rides on the combine's launch: every particle keeps its id,
    cell, position and momentum through two reorders (bars of the push tests), and
    the second full step, which reads the storage the first one wrote, deposits what
    the oracle does."""
    from tertia_amd.mesh import Mesh
    rng = np.random.default_rng(ny + nz + nsplit)
    p = small(ny=ny, nz=nz, nslices=2, hx=0.4, ppc_y=1, ppc_z=1)
    n = ny * nz
    cell = np.sort(rng.integers(0, n, size=n))
    parts = ((cell % ny).astype(np.int32), (cell // ny).astype(np.int32),
             rng.uniform(0, 1, n), rng.uniform(0, 1, n), *rng.uniform(-0.8, 0.8, size=(3, n)),
             np.arange(n, dtype=np.int64))
    m, o = Mesh(p, history=()), oracle_mod.Oracle(p, history=())
    try:
        m.particle_split = nsplit
        o.set_particles(*parts)
        m.set_particles(*parts)
        for _ in range(2):
            o.push_deposit(1)
            m.MoveParticlesLayerSplit(0, 0, 1)
            for f in ("Jx", "Jy", "Jz", "Rho"):
                assert max_rel(m.get_field(f), o.get_field(f)) <= 1e-13
        po, pg = o.particles(), m.particles()
        oo, og = np.argsort(po["id"]), np.argsort(pg["id"])
        for k in ("id", "cj", "ck"):
            assert np.array_equal(po[k][oo], pg[k][og]), k
        for k in ("fy", "fz", "px", "py", "pz"):
            bar = 1e-14 * (max(ny, nz) if k in ("fy", "fz") else max(1.0, np.abs(po[k]).max()))
            assert np.abs(po[k][oo] - pg[k][og]).max() <= bar, k
    finally:
        m.close()


@pytest.mark.parametrize("shape", [QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF])
@pytest.mark.parametrize("per_cell,hot", [(1, 0), (4, 0), (8, 0), (9, 0), (30, 0), (3, 6)])
def test_global_deposit_cell_counts(oracle_mod, shape, per_cell, hot):
    """The same on a grid that is not made of tiles: lists of up to 8 events are ordered
    in registers, longer ones selected from, sub-steps of one particle by their
    number; the full step also stores the particles in that order."""
    from tertia_amd.mesh import Mesh
    ny, nz = 37, 50
    rng = np.random.default_rng(7 * per_cell + hot)
    p = small(ny=ny, nz=nz, nslices=2, hx=0.4 if hot else 0.05, shape=shape, ppc_y=2, ppc_z=4)
    cells = np.sort(rng.permutation(ny * nz)[: ny * nz * 8 // per_cell])
    cell = np.repeat(cells, per_cell)
    n = len(cell)
    mom = rng.uniform(-0.1, 0.1, size=(3, n))
    if hot:
        mom[0, ::hot] = 3.0
        mom[1, ::hot] = rng.uniform(-4, 4, size=len(mom[1, ::hot]))
    parts = ((cell % ny).astype(np.int32), (cell // ny).astype(np.int32),
             rng.uniform(0.2, 0.8, n), rng.uniform(0.2, 0.8, n), *mom,
             np.arange(n, dtype=np.int64))
    m, o = Mesh(p, history=()), oracle_mod.Oracle(p, history=())
    try:
        o.set_particles(*parts)
        runs = []
        for _ in range(2):
            m.set_particles(*parts)
            got = []
            for full in (0, 1, 0):
                m.MoveParticlesLayerSplit(0, 0, full)
                got += [m.get_field(f) for f in ("Jx", "Jy", "Jz", "Rho")]
            runs.append(got + [m.particles()["id"]])
        ref = []
        for full in (0, 1, 0):
            o.push_deposit(full)
            ref += [o.get_field(f) for f in ("Jx", "Jy", "Jz", "Rho")]
        for g, r in zip(runs[0], ref):
            assert max_rel(g, r) <= 1e-13
        for a, b in zip(*runs):
            assert np.array_equal(a, b)
    finally:
        m.close()


@pytest.mark.parametrize("shape", [QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF])
@pytest.mark.parametrize("per_cell", [1, 4, 5, 8, 9])
def test_float_deposit_cell_counts(oracle_mod, shape, per_cell):
    """The float form's ordered lists at the same edges.  No fields: a current is the
    sum of some per_cell terms of a few float products each, so 1e-6 of the largest
    (ten float roundings are 6e-7); and the same bits twice."""
    from tertia_amd.mesh import Mesh
    from tertia_amd.params import PRECISIONS
    ny = nz = 48
    rng = np.random.default_rng(per_cell)
    kw = dict(ny=ny, nz=nz, nslices=2, hx=0.05, shape=shape, ppc_y=2, ppc_z=4)
    cells = np.sort(rng.permutation(ny * nz)[: ny * nz * 8 // per_cell])
    cell = np.repeat(cells, per_cell)
    n = len(cell)
    parts = ((cell % ny).astype(np.int32), (cell // ny).astype(np.int32),
             rng.uniform(0.2, 0.8, n), rng.uniform(0.2, 0.8, n),
             *rng.uniform(-0.1, 0.1, size=(3, n)), np.arange(n, dtype=np.int64))
    m = Mesh(small(precision=PRECISIONS["mixed32"], **kw), history=())
    o = oracle_mod.Oracle(small(**kw), history=())
    try:
        o.set_particles(*parts)
        runs = []
        for _ in range(2):
            m.set_particles(*parts)
            m.MoveParticlesLayerSplit(0, 0, 1)
            runs.append([m.get_field(f) for f in ("Jx", "Jy", "Jz", "Rho")])
        o.push_deposit(1)
        for f, a, b in zip(("Jx", "Jy", "Jz", "Rho"), *runs):
            assert np.array_equal(a, b)
            assert max_rel(a, o.get_field(f)) <= 1e-6, f
    finally:
        m.close()
