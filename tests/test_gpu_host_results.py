"""Results the device writes to host memory: short interpolation lists against long ones, from several
threads on one field, and a solve's Gram-Schmidt columns, polled for or waited for."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _interp(f, x):
    import underworld2_amd._lib as L
    import ctypes
    x = np.ascontiguousarray(x)
    v, ok = np.zeros((len(x), f.nodeDofCount)), np.zeros(len(x), np.int32)
    L.check(L.lib().uwg_field_interpolate(f._h, len(x), L.dptr(x), L.dptr(v),
                                          ok.ctypes.data_as(ctypes.POINTER(ctypes.c_int))), "interpolate")
    return v, ok


def _field(order, dim, nc):
    import underworld2_amd as uw
    res = (7, 5, 6)[:dim]
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0" if order == 1 else "Q2/dPc1", res, (0.0,) * dim, (1.0,) * dim)
    f = uw.mesh.MeshVariable(mesh, nc)
    f.data[:] = np.random.default_rng(1).standard_normal(f.data.shape)
    return f


# 64 KB hold 65536 // (8 (dim + nc) + 4) points: 2340 scalars in 2D, 1260 vectors in 3D
@pytest.mark.parametrize("order,dim,nc", [(1, 2, 1), (1, 3, 3), (2, 2, 2), (2, 3, 3)])
def test_short_lists_match_long_ones(order, dim, nc):
    """The same kernel on both sides: identical values and flags, points outside included."""
    f = _field(order, dim, nc)
    cap = 65536 // (8 * (dim + nc) + 4)
    x = np.random.default_rng(2).uniform(-0.02, 1.02, (cap + 1, dim))
    v, ok = _interp(f, x)
    assert 0 < ok.sum() < len(x)
    for n in (1, 2, 63, cap - 1, cap):
        vs, oks = _interp(f, x[:n])
        assert np.array_equal(vs, v[:n]) and np.array_equal(oks, ok[:n])


def test_threads_share_a_field():
    f = _field(1, 3, 3)
    xs = [np.random.default_rng(k).uniform(0, 1, (40 + k, 3)) for k in range(4)]
    ref = [_interp(f, x)[0] for x in xs]
    bad = []

    def work(k):
        for _ in range(25):
            if not np.array_equal(_interp(f, xs[k])[0], ref[k]):
                bad.append(k)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_a_call_that_reports_an_earlier_error_gives_its_buffer_back_idle():
    """A failed allocation leaves an error that the next launch reports, with its kernel under way; the
    call waits for it before the buffer serves another call."""
    import ctypes
    import underworld2_amd._lib as L
    f = _field(1, 3, 3)
    xs = [np.random.default_rng(k).uniform(0, 1, (1000, 3)) for k in range(2)]
    ref = [_interp(f, x)[0] for x in xs]
    for _ in range(20):
        p = ctypes.c_void_p()
        assert L.lib().hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0
        with pytest.raises(Exception):
            _interp(f, xs[0])
        assert np.array_equal(_interp(f, xs[1])[0], ref[1])
    assert np.array_equal(_interp(f, xs[0])[0], ref[0])


@pytest.mark.parametrize("res,method", [((10, 6), "block"), ((10, 6), "schur"), ((64, 64, 64), "block")])
def test_repeated_solves_see_the_same_columns(res, method):
    """The host reads every Gram-Schmidt column from memory the device writes: on the small grid within
    the 100 us that it polls, at 64^3, where an iteration takes milliseconds, after a wait.  A
    column read early or late would change the iteration; the sums' order is fixed, so solves of one
    system in turn with solves of another agree bit for bit."""
    import underworld2_amd as uw
    dim, fn, x = len(res), uw.function, uw.function.input()

    def solver(eta):
        mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0", res, (0.0,) * dim, (1.0,) * dim)
        vel, p = uw.mesh.MeshVariable(mesh, dim), uw.mesh.MeshVariable(mesh.subMesh, 1)
        walls = tuple(mesh.specialSets[f"Min{n}_VertexSet"] + mesh.specialSets[f"Max{n}_VertexSet"] for n in "IJK"[:dim])
        st = uw.systems.Stokes(vel, p, fn_viscosity=fn.branching.conditional([(x[0] > 0.5, eta), (True, 1.0)]),
                               fn_bodyforce=(0.0,) * (dim - 1) + (fn.math.cos(3.0 * x[0]),),
                               conditions=[uw.conditions.DirichletCondition(vel, walls)])
        s = uw.systems.Solver(st)
        s.set_method(method)
        s.set_outer_rtol(1e-6)
        return s, vel, p
    systems = [solver(30.0), solver(3.0)]
    seen = []
    for _ in range(3):
        for s, vel, p in systems:
            s.solve()
            q = s.get_stats()
            seen.append((q.outer_its, q.pressure_its, q.velocity_total_its, vel.data.copy(), p.data.copy()))
    for k in (2, 3, 4, 5):
        assert seen[k][:3] == seen[k % 2][:3]
        assert np.array_equal(seen[k][3], seen[k % 2][3]) and np.array_equal(seen[k][4], seen[k % 2][4])
