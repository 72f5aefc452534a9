"""K applies of small grids against the streaming element kernels (selected with an explicit
chunk, themselves checked against the oracle in test_gpu_parity3d.py).

3D: the kernel that evaluates a chunk's element levels side by side shares the element arithmetic
and the order of the node sums, so every value is equal; grids at the tile edges (7 columns), the
level counts 2, 3 and 4 of its dispatch and one element.
2D: the assembled stencil sums the same terms in another order: per row 36 products and sums of
rounding u each, so |dy| <= 40 u sum|K||x| (u = 2^-53, 2^-24), row by row; FP32 entries add u.
Irregular Dirichlet masks reach every form of the row-sum block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(res, hi, seed, mask=None):
    import underworld2_amd as uw
    from underworld2_amd import _lib as L
    d = len(res)
    rng = np.random.default_rng(seed)
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0", res, (0.0,) * d, hi)
    v, p = uw.mesh.MeshVariable(mesh, d), uw.mesh.MeshVariable(mesh.subMesh, 1)
    sets = mesh.specialSets
    if mask is None:
        walls = tuple(sets[f"Min{a}_VertexSet"] + sets[f"Max{a}_VertexSet"] for a in "IJK"[:d])
    else:
        walls = tuple(uw.mesh.IndexSet(np.flatnonzero(rng.random(mesh.nodesGlobal) < mask), mesh.nodesGlobal)
                      for _ in range(d))
    st = uw.systems.Stokes(v, p, fn_viscosity=1.0, fn_bodyforce=(0.0,) * d,
                           conditions=[uw.conditions.DirichletCondition(v, walls)])
    eta = np.exp(2.0 * rng.standard_normal((mesh.elementsGlobal, 3 ** d)))
    L.check(L.lib().uwg_stokes_assemble_fields(st._h, L.dptr(eta), None))
    return mesh, v, p, st, rng.standard_normal(mesh.nodesGlobal * d)


def _apply(st, which, x):
    from underworld2_amd import _lib as L
    y = np.zeros_like(x)
    L.check(L.lib().uwg_stokes_apply(st._h, which, 0, L.dptr(x), L.dptr(y)))
    return y


@pytest.mark.parametrize("res", [(1, 1, 1), (6, 7, 2), (7, 6, 13), (8, 15, 3), (22, 13, 9), (26, 28, 30), (36, 41, 40)])
def test_3d_levels_side_by_side_equal_streaming(res):
    from underworld2_amd import _lib as L
    *keep, st, x = _system(res, (1.0, 0.9, 1.3), 3)
    got = [_apply(st, w, x) for w in (0, 4, 5, 6, 7)]
    try:
        L.lib().uwg_set_apply_chunk(2, 0)
        ref = [_apply(st, w, x) for w in (0, 4, 5, 6, 7)]
    finally:
        L.lib().uwg_set_apply_chunk(-1, 0)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("res,mask", [((1, 1), None), ((3, 2), 0.3), ((31, 29), 0.1), ((64, 5), None), ((130, 61), 0.02)])
def test_2d_stencil_against_element_kernel(res, mask):
    from underworld2_amd import _lib as L
    *keep, st, x = _system(res, (1.0, 1.3), 4, mask)
    got = [_apply(st, w, x) for w in (0, 4, 6, 7)]
    try:
        L.lib().uwg_set_apply_chunk(0, 1)
        ref = [_apply(st, w, x) for w in (0, 4, 6, 7)]
        # sum |K| |x| row by row: of the nodes three apart in either direction a row meets one
        rows = np.abs(x)
        for c in range(18):
            e = np.zeros((res[1] + 1, res[0] + 1, 2))
            e[(c // 2) // 3::3, (c // 2) % 3::3, c % 2] = 1.0
            rows = rows + np.abs(_apply(st, 0, e.ravel() * x))
    finally:
        L.lib().uwg_set_apply_chunk(0, -1)
    for a, b, u in zip(got, ref, (2.0 ** -53, 2.0 ** -24, 2.0 ** -53, 2.0 ** -24)):
        assert (np.abs(a - b) <= 40 * u * rows).all()


@pytest.mark.parametrize("res", [(31, 29), (64, 5)])
def test_2d_chunk_of_32_rows_is_a_chunk(res):
    """Every chunk size selects the element kernel, whose sums do not depend on it, 32 as well; a
    negative one restores the automatic choice, here the stencil, whose sums are ordered otherwise."""
    from underworld2_amd import _lib as L
    *keep, st, x = _system(res, (1.0, 1.3), 5)
    auto = _apply(st, 0, x)
    try:
        got = []
        for kz in (31, 32, 33):
            L.lib().uwg_set_apply_chunk(0, kz)
            got.append(_apply(st, 0, x))
    finally:
        L.lib().uwg_set_apply_chunk(0, -1)
    assert np.array_equal(got[1], got[0]) and np.array_equal(got[1], got[2])
    assert not np.array_equal(got[1], auto) and np.array_equal(_apply(st, 0, x), auto)


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("where", ["inside", "first column", "last column", "dirichlet"])
def test_2d_a_value_that_is_not_finite_stays_with_its_elements(where, value):
    """As in the element kernel: the nodes around it and no others, and none beside its own row where
    the value stands on a Dirichlet dof, whose column is zero."""
    from underworld2_amd import _lib as L
    res = (9, 6)
    mesh, *keep, st, x = _system(res, (1.0, 1.3), 6)
    nx = res[0] + 1
    # free dofs: component 1 on the side walls, both inside; component 0 is fixed on the side walls
    at = {"inside": 2 * (4 + 3 * nx), "first column": 2 * (3 * nx) + 1, "last column": 2 * (nx - 1 + 2 * nx) + 1,
          "dirichlet": 2 * (nx - 1 + 3 * nx)}[where]
    x[at] = value
    got = [_apply(st, w, x) for w in (0, 4, 6, 7)]
    try:
        L.lib().uwg_set_apply_chunk(0, 1)
        ref = [_apply(st, w, x) for w in (0, 4, 6, 7)]
    finally:
        L.lib().uwg_set_apply_chunk(0, -1)
    assert all(0 < (~np.isfinite(b)).sum() <= 18 for b in ref)
    for a, b, u in zip(got, ref, (2.0 ** -53, 2.0 ** -24, 2.0 ** -53, 2.0 ** -24)):
        f = np.isfinite(b)
        assert np.array_equal(np.isfinite(a), f)
        # 36 products and sums of rounding u on either side of entries up to the largest row
        assert np.abs(a[f] - b[f]).max() <= 40 * 18 * u * np.abs(b[f]).max()
