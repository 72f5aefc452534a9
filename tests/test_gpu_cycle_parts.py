"""The multigrid cycle and the block preconditioner against a host restatement that takes every part
by itself: the smoother's steps (first, from a guess, with the recurrence), the restriction, the
coarsest solve, the prolongation (a thread per dof, and per vertex on large grids), and the pressure
row z = -S^-1 (r - G^T u).  The restatement applies the level operators through the plain apply, which
other tests hold against the oracle, and does the rest in double precision on the host."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS, EPS32 = np.finfo(np.float64).eps, np.finfo(np.float32).eps


def _lib():
    from underworld2_amd import _lib as L
    return L


def _system(res, lid=False, order=1):
    import underworld2_amd as uw
    d = len(res)
    mesh = uw.mesh.FeMesh_Cartesian("Q1/dQ0" if order == 1 else "Q2/dPc1", res, (0.0,) * d, (1.0, 0.9, 1.2)[:d])
    vel, p = uw.mesh.MeshVariable(mesh, d), uw.mesh.MeshVariable(mesh.subMesh, 1)
    sets, fn, x = mesh.specialSets, uw.function, uw.function.input()
    walls = [sets[f"Min{a}_VertexSet"] + sets[f"Max{a}_VertexSet"] for a in "IJK"[:d]]
    if lid:  # the top's x velocity grows along x: the lifted continuity row is the same in all its elements
        walls[0] = walls[0] + sets[f"Max{'IJK'[d - 1]}_VertexSet"]
        top = sets[f"Max{'IJK'[d - 1]}_VertexSet"].data
        vel.data[top, 0] = mesh.data[top, 0]
    st = uw.systems.Stokes(vel, p, fn_viscosity=1.0 + 30.0 * x[0] * x[d - 1],
                           fn_bodyforce=(0.0,) * (d - 1) + (fn.math.cos(3.0 * x[0]),),
                           conditions=[uw.conditions.DirichletCondition(vel, tuple(walls))])
    vel._push()
    st._prepare_values()
    return uw, st, vel, p


class Cycle:
    """V(2,2) Chebyshev cycle; `kind`: the level apply (0 FP64, 4 as the FP32 cycle has it)."""

    def __init__(self, st, kind, first=0):
        L = _lib()
        self.L, self.st, self.kind = L, st, kind
        n = ctypes.c_int()
        L.check(L.lib().uwg_stokes_levels(st._h, ctypes.byref(n), None))
        r = np.zeros((n.value, 3), np.int32)
        L.check(L.lib().uwg_stokes_levels(st._h, ctypes.byref(n), r.ctypes.data_as(ctypes.POINTER(ctypes.c_int))))
        self.dim = 2 if r[0, 2] <= 1 and st._velocityField.nodeDofCount == 2 else 3
        self.nn = [tuple(v + 1 for v in q[:self.dim]) for q in r]
        self.free, self.dinv, self.lmax = {}, {}, {}
        for l in range(first, n.value):
            N = int(np.prod(self.nn[l]))
            m = np.zeros(N, np.uint8)
            L.check(L.lib().uwg_stokes_level_mask(st._h, l, m.ctypes.data_as(ctypes.POINTER(ctypes.c_ubyte))))
            self.free[l] = np.stack([(m >> d) & 1 == 0 for d in range(self.dim)], 1).ravel()
            if l == n.value - 1:
                self.last = l
                self.K = np.stack([self.apply(l, e, 0) for e in np.eye(N * self.dim)], 1)
                continue
            self.dinv[l] = 1.0 / self._diagonal(l)
            i = np.arange(N * self.dim, dtype=np.uint64)  # the library's start vector
            h = (i * 2654435761) & 0xffffffff
            h ^= h >> 15
            h = (h * 2246822519) & 0xffffffff
            h ^= h >> 13
            x = (h & 0xffff) / 65536.0 + 0.25
            for _ in range(12):
                y = self.dinv[l] * self.apply(l, x, 0)
                self.lmax[l] = np.linalg.norm(y)
                x = y / self.lmax[l]

    def apply(self, l, x, kind=None):
        y = np.zeros(x.size)
        self.L.check(self.L.lib().uwg_stokes_apply(self.st._h, self.kind if kind is None else kind, l,
                                                   self.L.dptr(np.ascontiguousarray(x)), self.L.dptr(y)))
        return y

    def _grid(self, l, v):  # [z][y][x][component]
        return v.reshape(self.nn[l][::-1] + (self.dim,))

    def _diagonal(self, l):
        d = np.zeros(int(np.prod(self.nn[l])) * self.dim)
        for c in range(3 ** self.dim * self.dim):  # unit vectors three nodes apart do not meet
            e = np.zeros(d.size)
            node = c // self.dim
            s = tuple(slice(node // 3 ** k % 3, None, 3) for k in range(self.dim))
            self._grid(l, e)[s + (c % self.dim,)] = 1.0
            d += e * self.apply(l, e, 0)
        return d

    def restrict(self, l, r):  # from level l
        v = self._grid(l, np.where(self.free[l], r, 0.0))
        for ax in range(self.dim):
            v = np.moveaxis(v, ax, 0)
            c = v[::2].copy()
            c[1:] += 0.5 * v[1::2]
            c[:-1] += 0.5 * v[1::2]
            v = np.moveaxis(c, 0, ax)
        return np.where(self.free[l + 1], v.ravel(), 0.0)

    def prolong(self, l, xc):  # to level l
        v = self._grid(l + 1, xc)
        for ax in range(self.dim):
            v = np.moveaxis(v, ax, 0)
            f = np.zeros((2 * v.shape[0] - 1,) + v.shape[1:])
            f[::2] = v
            f[1::2] = 0.5 * (v[1:] + v[:-1])
            v = np.moveaxis(f, 0, ax)
        return np.where(self.free[l], v.ravel(), 0.0)

    def smooth(self, l, b, x=None, degree=2):
        lo, hi = 0.12 * self.lmax[l], 1.1 * self.lmax[l]
        theta, delta = 0.5 * (hi + lo), 0.5 * (hi - lo)
        rho = delta / theta
        for k in range(degree):
            r = b if x is None else b - self.apply(l, x)
            if k == 0:
                d = self.dinv[l] * r / theta
            else:
                new = 1.0 / (2.0 * theta / delta - rho)
                d = new * rho * d + 2.0 * new / delta * (self.dinv[l] * r)
                rho = new
            x = d if x is None else x + d
        return x

    def run(self, l, b, seen=None):
        if seen is not None:
            seen[l] = b
        if l == self.last:
            return np.linalg.solve(self.K, b)
        x = self.smooth(l, b)
        x = x + self.prolong(l, self.run(l + 1, self.restrict(l, b - self.apply(l, x)), seen))
        return self.smooth(l, b, x)


@pytest.fixture(params=["auto", "chunk"])
def chunk(request):
    L = _lib()
    if request.param == "chunk":
        L.lib().uwg_set_apply_chunk(2, 4)
    yield request.param
    L.lib().uwg_set_apply_chunk(-1, -1)


# two to four levels, even and odd coarse sizes; the last two have 200,000 (3D) and 500,000 (2D)
# vertices between them and the sizes of a thread per dof
CYCLES = [(24, 24), (40, 24), (64, 96), (12, 10, 8), (16, 12, 8), (32, 24, 40), (64, 64, 48), (1024, 512)]


@pytest.mark.parametrize("res", CYCLES)
def test_double_precision_cycle(res, chunk):
    """A smoothing step adds D^-1 (b - K x) / theta, rounded by a few eps of |D^-1| |K| |x|, at most 2 x,
    to an iterate whose former errors it does not enlarge; a level has six such sums and two
    transfers: 100 eps of the largest value per level."""
    uw, st, vel, p = _system(res)
    c = Cycle(st, 0)
    assert c.last >= 1
    b = np.random.default_rng(1).standard_normal(vel.data.size)
    want = c.run(0, b)
    got = c.apply(0, b, 3)
    err = np.abs(got - want).max() / np.abs(want).max()
    print(f"{res}: {c.last + 1} levels, {err:.1e}", flush=True)
    assert err < 100 * EPS * (c.last + 1)


@pytest.mark.parametrize("res", [(16, 12, 8), (32, 24, 40)])
def test_3d_cycle_bits_do_not_depend_on_the_kernels(res):
    """Side by side or streaming, the element kernels round alike."""
    L = _lib()
    uw, st, vel, p = _system(res)
    b, out = np.random.default_rng(2).standard_normal(vel.data.size), []
    for kz in (-1, 2):
        L.lib().uwg_set_apply_chunk(kz, 0)
        y = np.zeros(b.size)
        L.check(L.lib().uwg_stokes_apply(st._h, 3, 0, L.dptr(b), L.dptr(y)))
        out.append(y)
    L.lib().uwg_set_apply_chunk(-1, 0)
    assert np.array_equal(*out)


@pytest.mark.parametrize("res", [(24, 24), (64, 96), (16, 12, 8), (32, 24, 40)])
def test_single_precision_cycle(res, chunk):
    """A mixed solve records what its first cycle, on the right-hand side over its norm, restricts to
    every level and what it leaves there.  Rounding: of the right-hand side b, the smoothed iterate
    being about D^-1 b, a few eps per level; of the residual that is left, eps of the rows' terms |K| |x|,
    at most twice their diagonal's."""
    L = _lib()
    uw, st, vel, p = _system(res)
    s = uw.systems.Solver(st)
    s.set_method("block")
    s.set_precision("mixed")
    s.options.scr.ksp_max_it = 1

    def record(level, kind, n):
        L.check(L.lib().uwg_stokes_capture(st._h, level, kind, 1, 1))
        with pytest.warns(UserWarning):
            s.solve()
        v, k = np.zeros(n, np.float32), ctypes.c_int()
        L.check(L.lib().uwg_stokes_get_captured(st._h, v.ctypes.data_as(ctypes.POINTER(ctypes.c_float)),
                                                ctypes.byref(k)))
        assert k.value == 1
        L.check(L.lib().uwg_stokes_capture(st._h, level, 0, 0, 1))
        return v.astype(np.float64)
    c = Cycle(st, 4)
    f = np.zeros(vel.data.size)
    L.check(L.lib().uwg_stokes_get_rhs(st._h, L.dptr(f)))
    f = np.where(c.free[0], f, 0.0)
    f = (f / np.linalg.norm(f)).astype(np.float32).astype(np.float64)
    seen = {}
    c.run(0, f, seen)
    for l in range(1, c.last + 1):
        b = record(l, 0, c.free[l].size)
        assert np.linalg.norm(b - seen[l]) < 50 * l * EPS32 * np.linalg.norm(seen[l]), l
    for l in range(1, c.last):
        b = record(l, 0, c.free[l].size)
        x = c.run(l, b)
        assert np.linalg.norm(record(l, 1, b.size) - (b - c.apply(l, x))) < 4 * EPS32 * np.linalg.norm(x / c.dinv[l]), l


def test_single_precision_prolongation_per_vertex():
    """128^3 elements: level 1 has 274,625 vertices, and its cycle's residual is recorded."""
    L = _lib()
    uw, st, vel, p = _system((128, 128, 128))
    s = uw.systems.Solver(st)
    s.set_method("block")
    s.set_precision("mixed")
    s.options.scr.ksp_max_it = 1
    out = []
    for kind in (0, 1):
        L.check(L.lib().uwg_stokes_capture(st._h, 1, kind, 1, 1))
        with pytest.warns(UserWarning):
            s.solve()
        v, k = np.zeros(65 ** 3 * 3, np.float32), ctypes.c_int()
        L.check(L.lib().uwg_stokes_get_captured(st._h, v.ctypes.data_as(ctypes.POINTER(ctypes.c_float)),
                                                ctypes.byref(k)))
        out.append(v.astype(np.float64))
    L.check(L.lib().uwg_stokes_capture(st._h, 1, 0, 0, 1))
    c = Cycle(st, 4, first=1)
    x = c.run(1, out[0])
    assert np.linalg.norm(out[1] - (out[0] - c.apply(1, x))) < 4 * EPS32 * np.linalg.norm(x / c.dinv[1])


PLAIN = [(res, prec, False) for res in ((12, 8), (12, 10, 8)) for prec in ("fp64", "mixed", "mixed-refine")]


@pytest.mark.parametrize("res,precision,learned", PLAIN + [((12, 10, 8), prec, True) for prec in ("fp64", "mixed")])
@pytest.mark.parametrize("lid", [False, True])
def test_pressure_row_after_one_iteration(res, lid, precision, learned):
    """One iteration of the coupled solve gives a multiple a of the preconditioned first vector, so that
    with u the free velocities S p - G^T u = -a r for the first vector's pressure part r: zero, or with
    the moving lid zero except for one value in its elements.  A learned stencil without output is
    the identity, its entries D^-1 rounded to 8 bits.  p and u are rounded once each, a in both; FP32
    vectors round to EPS32."""
    L = _lib()
    d = len(res)
    uw, st, vel, p = _system(res, lid)
    s = uw.systems.Solver(st)
    s.set_method("block")
    s.set_precision(precision)
    s.options.scr.ksp_max_it = 1
    if learned:
        from underworld2_amd import learned as M
        net = M.StencilNet(8, 1, seed=1)
        q = net.get_params()
        q[-27 * 9:] = 0.0
        net.set_params(q)
        L.check(L.lib().uwg_stokes_load_schur_nn(st._h, 8, 1, q.size, q.ctypes.data_as(ctypes.POINTER(ctypes.c_float))))
        s._learned = True
    with pytest.warns(UserWarning):
        s.solve()
    E, N = int(np.prod(res)), vel.data.shape[0]
    W, fe, S = np.zeros((3 ** d, E)), np.zeros((E, 2 ** d * d)), np.zeros(E)
    L.check(L.lib().uwg_stokes_get_assembly(st._h, 0, L.dptr(W), L.dptr(fe), L.dptr(S)))
    div = np.zeros(E)
    L.check(L.lib().uwg_stokes_apply(st._h, 2, 0, L.dptr(np.ascontiguousarray(vel.data)), L.dptr(div)))
    got = S * p.data[:, 0] - div
    eps = 200 * (EPS32 if precision == "mixed-refine" else EPS) + (2.0 ** -8 if learned else 0.0)
    tol = eps * max(np.abs(div).max(), np.abs(S * p.data[:, 0]).max())
    top = np.arange(E) >= E - E // res[-1]
    assert np.abs(p.data).max() > 0 and np.abs(got[~top]).max() <= tol
    if lid:
        assert np.ptp(got[top]) <= tol and (got[top] < -2 * tol).all()
    else:
        assert np.abs(got[top]).max() <= tol


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_q2_pressure_row_after_one_iteration(precision):
    """The same with the blocks of dPc1 pressures: S p = G^T u block by block."""
    L = _lib()
    res = (6, 4, 5)
    uw, st, vel, p = _system(res, order=2)
    s = uw.systems.Solver(st)
    s.set_method("block")
    s.set_precision(precision)
    s.options.scr.ksp_max_it = 1
    with pytest.warns(UserWarning):
        s.solve()
    E = int(np.prod(res))
    S, q = np.zeros((E, 4, 4)), np.zeros(E * 4)
    L.check(L.lib().uwg_stokes_get_assembly(st._h, 0, None, None, L.dptr(S)))
    L.check(L.lib().uwg_stokes_apply(st._h, 2, 0, L.dptr(np.ascontiguousarray(vel.data)), L.dptr(q)))
    sp = np.einsum("erc,ec->er", S, p.data.reshape(E, 4)).ravel()
    assert np.abs(q).max() > 0 and np.abs(sp - q).max() < 1e3 * EPS * np.abs(q).max()
