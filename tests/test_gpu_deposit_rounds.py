"""GPU: lists and sort give a node the same sums.  A round with more than 8 events in some
cell is sorted, the next one too while that lasts; either way a node's sums are those of
its cells' events in the order of their indices, so what lies elsewhere in the tile
must not change a bit of them, in the double and in the float form.

Second, rounds that change between the two forms within one tile, with hot particles
that take several sub-steps: the same bits when run again, and the double form against
the oracle (1e-13; a float's 1 - Vx of a hot particle has no such bound)."""
import numpy as np
import pytest

from tests.helpers import max_rel
from tertia_amd.params import PRECISIONS, QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF, small

pytestmark = pytest.mark.gpu

J = ("Jx", "Jy", "Jz", "Rho")


def particles(rng, cell, ny, mom):
    n = len(cell)
    return ((cell % ny).astype(np.int32), (cell // ny).astype(np.int32),
            rng.uniform(0.2, 0.8, n), rng.uniform(0.2, 0.8, n), *mom,
            np.arange(n, dtype=np.int64))


@pytest.mark.parametrize("prec", ["fp64", "mixed32"])
@pytest.mark.parametrize("shape", [QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF])
@pytest.mark.parametrize("per_cell", [1, 3, 8])
def test_a_crowd_elsewhere_changes_no_bit(prec, shape, per_cell):
    from tertia_amd.mesh import Mesh
    ny = nz = 48
    p = small(ny=ny, nz=nz, nslices=2, hx=0.05, shape=shape, ppc_y=2, ppc_z=4,
              precision=PRECISIONS[prec])
    out = []
    for crowd in (False, True):
        rng = np.random.default_rng(per_cell)
        cell = []
        for tk in range(0, nz, 16):
            for tj in range(0, ny, 16):   # one chunk of a tile: 192 near its low rows, 40 far above
                near = [tj + j + ny * (tk + k) for k in range(2, 10) for j in range(3, 13)]
                near = rng.permutation(near)[:72 // per_cell]
                far = [tj + 8 + ny * (tk + 14)] * 40 if crowd else \
                      [tj + 3 + j + ny * (tk + 14) for j in range(10)] * 4
                cell += sorted(np.repeat(near, per_cell)) + sorted(far)
        cell = np.array(cell)
        m = Mesh(p, history=())
        try:
            m.set_particles(*particles(rng, cell, ny, rng.uniform(-0.1, 0.1, (3, len(cell)))))
            got = []
            for full in (0, 1):
                m.MoveParticlesLayerSplit(0, 0, full)
                got += [m.get_field(f) for f in J]
            out.append(np.stack(got))
        finally:
            m.close()
    near = [k for k in range(nz) if 1 <= k % 16 <= 11]
    assert np.abs(out[0][:, near]).max() > 0
    assert np.array_equal(out[0][:, near], out[1][:, near])
    assert not np.array_equal(out[0], out[1])


@pytest.mark.parametrize("prec", ["fp64", "mixed32"])
@pytest.mark.parametrize("shape", [QSS_SHAPE_CIC, QSS_SHAPE_NGP_REF])
@pytest.mark.parametrize("counts,hot", [((12, 2), 0), ((2, 40, 3), 0), ((256,), 0), ((9, 8, 1), 7),
                                        ((4, 4), 3)])
def test_rounds_of_both_kinds(oracle_mod, prec, shape, counts, hot):
    from tertia_amd.mesh import Mesh
    ny = nz = 32
    rng = np.random.default_rng(sum(counts) + hot)
    kw = dict(ny=ny, nz=nz, nslices=2, hx=0.4 if hot else 0.05, shape=shape, ppc_y=2, ppc_z=4)
    cell, k = [], 0
    order = rng.permutation(ny * nz)
    while len(cell) < 6000 and k < ny * nz:   # runs of cells with each count in turn
        cell += [order[k]] * counts[k // 60 % len(counts)]
        k += 1
    cell = np.sort(np.array(cell)) if hot == 0 else np.array(cell)
    mom = rng.uniform(-0.1, 0.1, size=(3, len(cell)))
    if hot:
        mom[0, ::hot] = 3.0
        mom[1, ::hot] = rng.uniform(-4, 4, size=len(mom[1, ::hot]))
    parts = particles(rng, cell, ny, mom)
    m = Mesh(small(precision=PRECISIONS[prec], **kw), history=())
    o = oracle_mod.Oracle(small(**kw), history=())
    try:
        o.set_particles(*parts)
        for full in (0, 1):
            o.push_deposit(full)
        runs = []
        for split in (1, 1, 2):
            m.particle_split = split
            m.set_particles(*parts)
            for full in (0, 1):
                m.MoveParticlesLayerSplit(0, 0, full)
            runs.append([m.get_field(f) for f in J])
        for f, a, b, c in zip(J, *runs):
            assert np.array_equal(a, b), f
            if prec == "fp64":
                for g in (a, c):
                    assert max_rel(g, o.get_field(f)) <= 1e-13, f
    finally:
        m.close()
        o.close()
