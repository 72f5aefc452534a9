"""Solves through the passes joined in the Krylov step: Gram-Schmidt with the norm in the update (up to
2^20 unknowns) and separate from it, dot products over 1 to 40 vectors (groups of eight, a second
batch after 32), G added into the operator's result.  The preconditioner's joined passes are held
against a host restatement in test_gpu_cycle_parts.py; here a wrong one shows in the iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stokes(res):
    import underworld2_amd as uw
    dim = len(res)
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0", res, (0.0,) * dim, (1.0,) * dim)
    vel, p = uw.mesh.MeshVariable(mesh, dim), uw.mesh.MeshVariable(mesh.subMesh, 1)
    x = uw.function.input()
    fn = uw.function
    walls = tuple(mesh.specialSets[f"Min{n}_VertexSet"] + mesh.specialSets[f"Max{n}_VertexSet"] for n in "IJK"[:dim])
    st = uw.systems.Stokes(vel, p, fn_viscosity=fn.branching.conditional([(x[0] > 0.5, 30.0), (True, 1.0)]),
                           fn_bodyforce=(0.0,) * (dim - 1) + (fn.math.cos(3.0 * x[0]),),
                           conditions=[uw.conditions.DirichletCondition(vel, walls)])
    return uw, st, vel, p


# 4305 (odd) and 214 unknowns; 48^3: 463,539, two per thread; 64^3: 1,086,019, above 2^20; and the
# iterations that separate passes took
@pytest.mark.parametrize("res,restart,its", [((6, 10, 14), 3, (66, 65)), ((6, 10, 14), 9, (35, 35)),
                                             ((6, 10, 14), 40, (28, 29)), ((10, 6), 17, (13, 15)),
                                             ((48, 48, 48), 40, (25, 26)), ((64, 64, 64), 40, (24, 26))])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_residual_of_the_unjoined_operators(res, restart, its, precision):
    """The residual that uwg_stokes_residuals forms with separate K, G, G^T and vector passes is the
    one the joined passes converged to: the outer tolerance 1e-7 relative to the right-hand side
    (the pressure part is zero), and 10 % for the rounding that the Arnoldi estimate does not see.
    The iterations are those of separate passes; one more or less leaves room for a last step whose
    residual lies on the tolerance."""
    uw, st, vel, p = _stokes(res)
    s = uw.systems.Solver(st)
    s.set_method("block")
    s.set_precision(precision)
    s.set_restart(restart)
    s.set_outer_rtol(1e-7)
    s.solve()
    r = s.get_stats()
    assert r.converged
    assert np.hypot(r.res_momentum, r.res_continuity) < 1.1e-7 * r.norm_f
    assert abs(r.outer_its - its[precision == "mixed"]) <= 1
