"""Sum-factorised Q2 apply with element results summed per vertex, and G^T with a lane per vertex:
grids of one element, odd and even sizes, remainders of the eight elements a workgroup takes, and
layers of element results kept in a ring."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stokes(res):
    import underworld2_amd as uw
    dim = len(res)
    mesh = uw.mesh.FeMesh_Cartesian("Q2/dPc1", res, (0.0,) * dim, (1.0, 0.8, 0.7)[:dim])
    vel, p = uw.mesh.MeshVariable(mesh, dim), uw.mesh.MeshVariable(mesh.subMesh, 1)
    x = uw.function.input()
    walls = [mesh.specialSets[f"Min{n}_VertexSet"] + mesh.specialSets[f"Max{n}_VertexSet"] for n in "IJK"[:dim]]
    st = uw.systems.Stokes(vel, p, fn_viscosity=1.0 + 3.0 * x[0] * x[1], fn_bodyforce=(0.0,) * (dim - 1) + (-1.0,),
                           conditions=[uw.conditions.DirichletCondition(vel, tuple(walls))])
    st._prepare_values()
    return st, vel.data.size, int(np.prod(res)) * (dim + 1)


def _apply(st, which, x, n_out):
    import underworld2_amd._lib as L
    y = np.zeros(n_out)
    L.check(L.lib().uwg_stokes_apply(st._h, which, 0, L.dptr(np.ascontiguousarray(x, np.float64)), L.dptr(y)),
            "apply")
    return y


def _kernel(kind):
    import underworld2_amd._lib as L
    L.check(L.lib().uwg_set_q2_apply_kernel(kind), "kernel")


# (30, 36, 100): 32 MiB hold 47 layers' results in double and 95 in single precision
RES = [(1, 1, 1), (2, 1, 3), (3, 3, 3), (5, 4, 3), (9, 2, 7), (30, 36, 100)]


@pytest.mark.parametrize("res", RES)
def test_apply_matches_the_dense_kernel(res):
    """Both kernels sum the same products: three passes of sums of 3 or 5 terms to a point and three
    back, then a vertex's up to 8 elements, or sums of 27 and 125 terms, 30 roundings deep either way
    where a tree or random signs halve a sum's: 30 eps of the largest row."""
    st, n, _ = _stokes(res)
    x = np.random.default_rng(3).standard_normal(n)
    try:
        _kernel(0)
        ref = _apply(st, 0, x, n)
    finally:
        _kernel(2)
    scale = np.abs(ref).max()
    assert np.abs(_apply(st, 0, x, n) - ref).max() < 30 * np.finfo(np.float64).eps * scale
    assert np.abs(_apply(st, 4, x, n) - ref).max() < 30 * np.finfo(np.float32).eps * scale


@pytest.mark.parametrize("res", [r for r in RES if min(r) > 1])
def test_cycle_with_fused_row_operations(res):
    """One V-cycle with the residual and the smoother step in the vertex kernel against the
    separate passes of the dense kernel.  The five applies perturb their rows by at most 30 eps of
    the largest each, which the smoother takes back to the iterate as D^-1 / theta does the rows
    themselves: 5 x 30 eps of the largest value."""
    st, n, _ = _stokes(res)
    x = np.random.default_rng(4).standard_normal(n)
    try:
        _kernel(0)
        ref = _apply(st, 3, x, n)
    finally:
        _kernel(2)
    got = _apply(st, 3, x, n)
    assert np.abs(got - ref).max() < 150 * np.finfo(np.float64).eps * np.abs(ref).max()


@pytest.mark.parametrize("res", [(1, 1), (5, 3), (33, 17), (1, 1, 1), (2, 1, 3), (5, 4, 3), (9, 2, 7)])
def test_divergence_matches_the_gradient(res):
    """G^T u against the adjoint of G: (G p, u) = (p, G^T u) row by row, p the unit vectors of the
    first and the last element and a random vector.  Sums of 81 products, 16 eps each way."""
    st, n, m = _stokes(res)
    rng = np.random.default_rng(5)
    u = rng.standard_normal(n)
    q = _apply(st, 2, u, m)
    scale = np.abs(q).max()
    for i in {*range(min(m, 8)), *range(max(0, m - 8), m)}:
        p = np.zeros(m)
        p[i] = 1.0
        assert abs(_apply(st, 1, p, n) @ u - q[i]) < 81 * 16 * np.finfo(np.float64).eps * scale
    p = rng.standard_normal(m)
    assert abs(_apply(st, 1, p, n) @ u - q @ p) < 16 * np.sqrt(n) * np.finfo(np.float64).eps * np.abs(q) @ np.abs(p)


@pytest.mark.parametrize("res", [(1, 1), (3, 3), (1, 1, 1), (3, 1, 1), (5, 3, 1)])
def test_schur_blocks_of_ragged_element_counts(res):
    """approxS blocks against the oracle's where the elements leave workgroups partly empty (four
    per workgroup in 3D, eight in 2D): sums of 81 terms of one sign pattern, 1e-12 of the largest."""
    from oracle import q2_oracle as Q
    import underworld2_amd._lib as L
    dim = len(res)
    st, _, _ = _stokes(res)
    om = Q.Q2Mesh(res, (0.0,) * dim, (1.0, 0.8, 0.7)[:dim])
    Ke, _ = Q.gauss_assembly(om, lambda X: 1.0 + 3.0 * X[:, 0] * X[:, 1],
                             lambda X: np.stack([0 * X[:, 0]] * (dim - 1) + [-1.0 + 0 * X[:, 0]], -1))
    S = np.zeros((om.E, om.npe, om.npe))
    L.check(L.lib().uwg_stokes_get_assembly(st._h, 0, None, None, L.dptr(S)), "assembly")
    want = Q.element_approxS(Ke, Q.element_G(om))
    assert np.abs(S - want).max() < 1e-12 * np.abs(want).max()
