"""Discrete-Voronoi weights and centroids equal the sequential oracle's bit for bit where the
round-at-a-time kernel changes path: the lines between its 32- and 64-bit masks and the sequential
kernel (32, 33, 64, 65, 129 particles), several particles in one grid cell, one particle, layouts
with exact ties, particles on walls and corners, and clusters whose cells are disconnected."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(d, res, x):
    import underworld2_amd as uw
    from oracle import oracle as O
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0", res, (0.0,) * d, (1.0,) * d)
    sw = uw.swarm.Swarm(mesh)
    sw.add_particles_with_coordinates(x)
    ptr, pid = sw.cell_tables()
    coords = sw.particleCoordinates.data.copy()
    xi0 = O.coincident_map(O.Mesh(res, (0.0,) * d, (1.0,) * d), ptr, pid, coords)
    xo, wo = O.dvc_all(d, ptr, xi0)
    for _ in range(2):  # a second pass on the same workspace
        xg, wg = sw.integration_points(dvc=True)
        assert np.array_equal(wg, wo)
        assert np.array_equal(xg, xo)
    return np.diff(ptr)


def _in_cells(res, counts, rng, place):
    d = len(res)
    out = []
    for e, n in enumerate(counts):
        idx = np.array([e % res[0], (e // res[0]) % res[1]] + ([e // (res[0] * res[1])] if d == 3 else []))
        out.append((idx + place(n, d, rng)) / np.array(res))
    return np.concatenate(out)


UNIFORM = lambda n, d, rng: rng.random((n, d))
CLUSTER = lambda n, d, rng: np.clip(rng.random(d) + 0.06 * rng.standard_normal((n, d)), 0.0, 1.0)
COPLANAR = lambda n, d, rng: np.concatenate([rng.random((n, d - 1)), np.full((n, 1), 0.37)], 1)


@pytest.mark.parametrize("d,place", [(2, UNIFORM), (3, UNIFORM), (2, CLUSTER), (3, CLUSTER), (3, COPLANAR)])
def test_counts_around_every_line(d, place):
    counts = [1, 2, 7, 31, 32, 33, 47, 63, 64, 65, 100, 128, 129, 20, 25, 30, 5, 16]
    res = (6, 3) if d == 2 else (3, 3, 2)
    got = _check(d, res, _in_cells(res, counts, np.random.default_rng(6), place))
    if place is not CLUSTER:
        assert sorted(got) == sorted(counts)


@pytest.mark.parametrize("d,k", [(2, 3), (2, 4), (3, 2), (3, 3)])
def test_symmetric_layouts_with_ties(d, k):
    res = (4, 3) if d == 2 else (3, 2, 2)
    g = (np.arange(k) + 0.5) / k
    lat = np.stack(np.meshgrid(*([g] * d), indexing="ij"), -1).reshape(-1, d)
    _check(d, res, _in_cells(res, [1] * int(np.prod(res)), np.random.default_rng(1), lambda n, dd, r: lat))


@pytest.mark.parametrize("d", [2, 3])
def test_faces_corners_and_many_elements(d):
    rng = np.random.default_rng(8)
    res = (37, 23) if d == 2 else (11, 9, 7)
    x = rng.random((int(np.prod(res)) * 24, d))
    x[:200] = np.round(x[:200])                      # corners of the box
    x[200:400, 0] = np.round(x[200:400, 0] * res[0]) / res[0]  # element faces
    _check(d, res, x)


@pytest.mark.parametrize("d", [2, 3])
def test_many_elements_left_to_the_sequential_kernel(d):
    """Several workgroups' worth of elements with ties, with 65-130 particles (on either side of the
    128 that kernel holds) and with none of both, in every order."""
    res = (29, 23) if d == 2 else (9, 8, 7)
    E = int(np.prod(res))
    rng = np.random.default_rng(9)
    g = (np.arange(2) + 0.5) / 2
    lat = np.stack(np.meshgrid(*([g] * d), indexing="ij"), -1).reshape(-1, d)
    kind = rng.integers(0, 4, E)
    sizes = np.choose(kind, [2 ** d, rng.integers(65, 131, E), rng.integers(33, 65, E), rng.integers(1, 33, E)])
    it = iter(kind)
    _check(d, res, _in_cells(res, sizes, rng, lambda n, dd, r: lat if next(it) == 0 else r.random((n, dd))))
