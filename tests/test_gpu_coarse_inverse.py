"""Gauss-Jordan inverse of the coarsest operator, eight pivots a launch: matrices of 8 to 360 unknowns
with and without a remainder of the eight pivots and of the 16 x 64 tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# an odd direction keeps the hierarchy at one level, whose cycle is the product with the inverse
@pytest.mark.parametrize("res", [(1, 1), (2, 1), (4, 1), (2, 1, 1), (4, 2, 1), (5, 4, 3)])
def test_operator_times_inverse(res):
    """K V(b) = b to eps times the condition number of the scaled operator (viscosities 1 to 10,
    at most 6 elements across: below 1e4), times 16 for n products of random rounding."""
    import underworld2_amd as uw
    import underworld2_amd._lib as L
    dim = len(res)
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0", res, (0.0,) * dim, (1.0,) * dim)
    vel, p = uw.mesh.MeshVariable(mesh, dim), uw.mesh.MeshVariable(mesh.subMesh, 1)
    x = uw.function.input()
    walls = tuple(mesh.specialSets[f"Min{n}_VertexSet"] + mesh.specialSets[f"Max{n}_VertexSet"] for n in "IJK"[:dim])
    st = uw.systems.Stokes(vel, p, fn_viscosity=1.0 + 9.0 * x[0], fn_bodyforce=(0.0,) * dim,
                           conditions=[uw.conditions.DirichletCondition(vel, walls)])
    st._prepare_values()
    n = vel.data.size
    b = np.random.default_rng(2).standard_normal(n)
    got = b
    for which in (3, 0):
        y = np.zeros(n)
        L.check(L.lib().uwg_stokes_apply(st._h, which, 0, L.dptr(np.ascontiguousarray(got)), L.dptr(y)), "apply")
        got = y
    assert np.abs(got - b).max() < 16e4 * np.finfo(np.float64).eps * np.abs(b).max()
