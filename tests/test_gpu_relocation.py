"""Per-cell particle tables after relocation equal the sequential edits of the oracle
(swap-with-last removal, append) where the kernel's paths change: cells that gain more
particles than the scan serves (the movers are then sorted), tables longer than the workgroup's
list, cells emptied and filled, one element, and particles that stay."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,ppc,target", [
    ((5, 3), 7, 0.0),          # scan only
    ((5, 3), 40, 0.15),        # one cell gains about 80: sorted movers, list above 96
    ((3, 2, 4), 30, 0.0),
    ((3, 2, 4), 110, 0.05),    # every table is longer than the list
    ((1, 1), 9, 0.0),
    ((2, 3, 2), 47, 0.9),      # nearly all particles end in one cell
])
def test_tables_after_moves_match_sequential_edits(res, ppc, target):
    from oracle import oracle as O
    import underworld2_amd as uw
    d = len(res)
    lo, hi = (0.0,) * d, (1.0,) * d
    rng = np.random.default_rng(11)
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0", res, lo, hi)
    sw = uw.swarm.Swarm(mesh)
    P = ppc * int(np.prod(res))
    x = rng.random((P, d))
    sw.add_particles_with_coordinates(x)
    m = O.Mesh(res, lo, hi)
    own0 = sw.owningCell.data[:, 0].copy()
    ptr, pid = sw.cell_tables()
    assert np.array_equal(pid, np.argsort(own0, kind="stable"))  # appended in index order
    T = O.CellTables(m, ptr, pid, cap=P)
    for step in range(3):
        move = rng.random(P) < 0.35
        x = sw.particleCoordinates.data.copy()
        x[move] = rng.random((int(move.sum()), d))
        pull = rng.random(P) < target
        x[pull] = rng.random((int(pull.sum()), d)) / np.array(res)  # the first cell
        sw.particleCoordinates.data[:] = x
        sw.update_particle_owners()
        assert T.update(x) == 0
        ptr, pid = sw.cell_tables()
        eptr, epid = T.csr()
        assert np.array_equal(ptr, eptr) and np.array_equal(pid, epid), step
        assert np.array_equal(sw.owningCell.data[:, 0], T.owner)
