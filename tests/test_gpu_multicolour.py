"""The multicolour solve's arithmetic does not depend on how the matrix is stored: a
row's block products are added in ascending mesh column, the diagonal block in its
place, and sums over the vectors run in the order of the device rows.

* Product and sweeps bit for bit against numpy loops in that order, on random blocks
  and on a flow's own Jacobian, with two colours and more, in the three ways a slice is
  worked on (one wave, four, eight).
* Norms bit for bit against the row-major path's.
* Solutions of a flow's own system after the iterations the solver takes, against
  the same recurrence in 80-bit floats: the device is no further from it than twice
  what plain numpy sweeps and products of the same precision are (they round the same
  operations; the factor is for the different order of the dot products' sums).  At low
  Mach number a block's rows differ by orders of magnitude, and a form that reuses the
  right-hand side of the 5x5 solves for the product (A z = y + ...) is 3 (plate) to 22
  times (SA bump) further off with the same residual.
"""
import numpy as np
import pytest

import cfdg
import cfdg.cases as cases
from helpers import perturbed_state
from test_gpu_sliced import FORMS, _solver

pytestmark = pytest.mark.gpu


def _times(B, x):
    """Block products, summed over the block's columns in order."""
    t = B[..., 0] * x[..., None, 0]
    for j in range(1, 5):
        t = t + B[..., j] * x[..., None, j]
    return t


def _lu(D):
    """LU of 5x5 blocks with the largest pivot (bsr_helpers.hpp:278-321)."""
    a, n = D.copy(), np.arange(len(D))
    piv = np.empty((len(D), 5), int)
    for k in range(5):
        p = piv[:, k] = k + np.argmax(np.abs(a[:, k:, k]), axis=1)
        row = a[n, p].copy()
        a[n, p] = a[:, k]
        a[:, k] = row
        inv = a.dtype.type(1) / a[:, k, k]
        for r in range(k + 1, 5):
            a[:, r, k] = a[:, r, k] * inv
            a[:, r, k + 1:] = a[:, r, k + 1:] - a[:, r, k, None] * a[:, k, k + 1:]
    return a, piv


def _lu_solve(lu, piv, s):
    s, n = s.copy(), np.arange(len(s))
    for k in range(5):
        t = s[:, k].copy()
        s[:, k] = s[n, piv[:, k]]
        s[n, piv[:, k]] = np.where(piv[:, k] == k, s[:, k], t)
    for a in range(1, 5):
        for b in range(a):
            s[:, a] = s[:, a] - lu[:, a, b] * s[:, b]
    for a in range(4, -1, -1):
        for b in range(a + 1, 5):
            s[:, a] = s[:, a] - lu[:, a, b] * s[:, b]
        s[:, a] = s[:, a] / lu[:, a, a]
    return s


class Host:
    """Product and multicolour sweeps in numpy at one precision.  The factors are formed
    in float64, or in the precision itself when that is wider."""

    def __init__(self, rp, cols, dg, B, colour, dtype):
        self.rp, self.cols, self.dg, self.colour = rp, cols, dg, colour
        self.B = B.astype(dtype)
        self.lu, self.piv = _lu(B[dg].astype(np.promote_types(dtype, np.float64)))
        self.lu = self.lu.astype(dtype)
        self.most = int(np.max(np.diff(rp)))

    def _entries(self, rows, k):
        """Rows that have a k-th entry, and that entry."""
        e = self.rp[rows] + k
        has = e < self.rp[rows + 1]
        return has, e[has]

    def product(self, x):
        x = x.reshape(-1, 5)
        y, rows = np.zeros_like(x), np.arange(len(self.dg))
        for k in range(self.most):
            has, e = self._entries(rows, k)
            y[has] = y[has] + _times(self.B[e], x[self.cols[e]])
        return y.ravel()

    def sweep(self, r):
        r = r.reshape(-1, 5)
        z, n = np.zeros_like(r), int(self.colour.max()) + 1
        for step, c in enumerate(list(range(n)) + list(range(n - 2, -1, -1))):
            rows = np.nonzero(self.colour == c)[0]
            acc = r[rows].copy()
            for k in range(self.most):
                has, e = self._entries(rows, k)
                use = self.colour[self.cols[e]] < c if step < n else self.dg[rows[has]] != e
                at = np.nonzero(has)[0][use]
                acc[at] = acc[at] - _times(self.B[e[use]], z[self.cols[e[use]]])
            z[rows] = _lu_solve(self.lu[rows], self.piv[rows], acc)
        return z.ravel()

    def bicgstab(self, b, iterations):
        dot = np.promote_types(b.dtype, np.float64).type
        inner = lambda u, v: (u.astype(dot) * v.astype(dot)).sum()  # noqa: E731
        one = b.dtype.type
        x, r, r0 = np.zeros_like(b), b.copy(), b.copy()
        p, v = np.zeros_like(b), np.zeros_like(b)
        rho = inner(r0, r)
        alpha = omega = dot(1)
        for it in range(iterations):
            if it == 0:
                p = r.copy()
            else:
                rho_new = inner(r0, r)
                beta = (rho_new / rho) * (alpha / omega)
                p = one(beta) * p + one(-beta * omega) * v + r
                rho = rho_new
            ph = self.sweep(p)
            v = self.product(ph)
            alpha = rho / inner(r0, v)
            s = r + one(-alpha) * v
            sh = self.sweep(s)
            t = self.product(sh)
            omega = inner(t, s) / inner(t, t)
            x = x + one(alpha) * ph + one(omega) * sh
            r = s + one(-omega) * t
        return x


def _host(s, B, dtype):
    rp, cols, dg = s.bsr_pattern()
    return Host(rp, cols, dg, B, s.sgs_row_groups(cfdg.SGS_MULTICOLOUR)[0], dtype)


FLOWS = {
    "ramp": lambda n: cases.ramp(ni=n, nj=n - 3, nk=5),
    "plate": lambda n: cases.plate(ni=n, nj=n - 5, nk=9, limiter="UNLIMITED", cfl=50.0),
    "plate_sa": lambda n: cases.plate_sa(ni=n, nj=n - 5, nk=9, cfl=50.0),
    "bump_sa": lambda n: cases.bump_sa(ni=n, nj=n - 3, nk=n - 4),
}


def _flow(kind, n, form="fp64"):
    case = FLOWS[kind](n)
    s = cfdg.Solver(cfdg.Mesh.generate(**case.mesh), case.numerics, case.bcs)
    if form != "fp64":
        s.set_precision(FORMS[form])
    if kind.endswith("_sa"):
        s.set_turbulence(cases.turbulence(case, update=cfdg.TURB_FROZEN))
    s.set_state(perturbed_state(s, case, amp=0.002))
    s.eval_residual()
    s.compute_dt()
    s.assemble_jacobian()
    return s


def _check_bits(s, form):
    B = s.bsr_values()
    r = np.random.default_rng(3).standard_normal(5 * s.n_cells)
    h = _host(s, B, np.float64)
    assert np.array_equal(s.spmv(r), h.product(r))
    if FORMS[form].krylov == cfdg.PREC_FP32:
        h, r = _host(s, B, np.float32), r.astype(np.float32)
    assert np.array_equal(s.sgs_apply(cfdg.SGS_MULTICOLOUR, r), h.sweep(r).astype(np.float64))


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("kind, size", [("hex", (1, 1, 1)), ("hex", (13, 11, 3)), ("tet", (2, 1, 3)), ("tet", (11, 13, 9)),
                                        ("tet", (21, 19, 17)), ("hex", (41, 40, 31)), ("hex", (64, 64, 49))])
def test_random_blocks_bitwise(kind, size, form):
    _check_bits(_solver(kind, size, form)[1], form)


def _hub_solver(size, form):
    """Two cells with some thirty faces more, to cells all over the mesh: more blocks than
    a kernel holds at a time, and faces that are not in the order of their cells."""
    ni, nj, nk = size
    case = cases.ramp(ni=ni, nj=nj, nk=nk, gradient="GREEN_GAUSS_CELL")
    m = cfdg.Mesh.generate(**case.mesh)
    a, at, n = m.arrays(), m.n_inner_faces, m.n_cells
    couples = {tuple(sorted(c)) for c in zip(a["face_owner"][:at], a["face_neigh"][:at])}
    new = []
    for hub in (0, n // 2):
        for k in range(30):
            c = k * 7919 % n
            if c != hub and tuple(sorted((hub, c))) not in couples:
                couples.add(tuple(sorted((hub, c))))
                new.append((hub, c))
    own = np.array([h for h, _ in new])
    corners = a["face_nodes"][:a["face_nodes_off"][1]]
    extra = dict(face_owner=own, face_neigh=[c for _, c in new], face_patch=-1, face_type=a["face_type"][0],
                 face_cx=a["cell_cx"][own] + 1e-3, face_cy=a["cell_cy"][own], face_cz=a["cell_cz"][own],
                 face_nx=1.0, face_ny=0.0, face_nz=0.0, face_area=1e-3)
    for k, v in extra.items():
        a[k] = np.insert(a[k], at, np.broadcast_to(v, len(new)))
    o = a["face_nodes_off"]
    a["face_nodes"] = np.insert(a["face_nodes"], o[at], np.tile(corners, len(new)))
    step = len(corners) * np.arange(1, len(new) + 1)
    a["face_nodes_off"] = np.concatenate([o[:at + 1], o[at] + step, o[at + 1:] + step[-1]])
    s = cfdg.Solver(cfdg.Mesh.from_arrays(a, m.n_patches), case.numerics, case.bcs)
    s.set_precision(FORMS[form])
    rng = np.random.default_rng(11)
    rp, cols, dg = s.bsr_pattern()
    v = 0.1 * rng.standard_normal((len(cols), 5, 5)) / 5.0
    v[dg] += np.eye(5) * (1.5 + rng.random((n, 1, 1)))
    s.set_bsr_values(v)
    return s


@pytest.mark.parametrize("form", ["fp64", "bf16"])
@pytest.mark.parametrize("size", [(7, 6, 5), (41, 40, 31), (64, 64, 49)])
def test_many_faces_bitwise(size, form):
    s = _hub_solver(size, form)
    assert np.max(np.diff(s.bsr_pattern()[0])) > 30
    _check_bits(s, form)
    h = _host(s, s.bsr_values(), np.float64)
    b = np.random.default_rng(5).standard_normal(5 * s.n_cells)
    x, res = s.linear_solve(cases.default_linparams(rel_tol=1e-6), b=b)
    assert res.status == cfdg.CONVERGED
    assert np.linalg.norm(b - h.product(x)) <= 1.05e-6 * np.linalg.norm(b)
    if form == "fp64":  # the products inside the iteration, not only their end
        y, r3 = s.linear_solve(cases.default_linparams(rel_tol=1e-30, abs_tol=0.0, max_iter=3), b=b)
        ref = h.bicgstab(b, 3)
        assert r3.iterations == 3 and np.max(np.abs(y - ref)) <= 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("form", ["fp64", "bf16"])
@pytest.mark.parametrize("kind", sorted(FLOWS))
def test_flow_jacobian_bitwise(kind, form):
    _check_bits(_flow(kind, 17, form), form)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("kind, n", [("plate", 6), ("plate", 41), ("bump_sa", 13)])
def test_norms_are_the_row_major_ones(kind, n, form):
    """Sums of the sliced vectors in the order of the device rows: the residual's norm
    with a guess against the solve without preconditioner, which works row by row, and
    an implicit step's norms against those of the residual."""
    s = _flow(kind, n, form)
    b, x0 = np.random.default_rng(7).standard_normal((2, 5 * s.n_cells))
    lp = cases.default_linparams(max_iter=0)
    none = cases.default_linparams(max_iter=0)
    none.preconditioner = cfdg.PRECOND_NONE
    for guess in (x0, None):
        assert (s.linear_solve(lp, b=b, x0=guess)[1].initial_residual
                == s.linear_solve(none, b=b, x0=guess)[1].initial_residual)
    l2 = s.residual_norms()
    R = s.residual()[0]
    # without a right-hand side given: -R, its sums formed with it
    assert s.linear_solve(lp)[1].initial_residual == s.linear_solve(lp, b=-R.T.ravel())[1].initial_residual
    assert np.array_equal(np.array(s.implicit_step(cases.default_linparams()).l2), l2)


@pytest.mark.parametrize("form", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("kind, n", [("plate", 33), ("plate_sa", 33), ("bump_sa", 13)])
def test_update_is_as_exact_as_the_plain_form(kind, n, form):
    s = _flow(kind, n, form)
    if form != "fp64":  # one inner solve, so that its iterations are those of the recurrence
        s.set_precision(cfdg.Precision.make(FORMS[form].block_storage, cfdg.PREC_FP32, max_outer=1))
        s.assemble_jacobian()
    dtype = np.float64 if form == "fp64" else np.float32
    B = s.bsr_values()
    b = -s.residual()[0].T.ravel()
    x, res = s.linear_solve(cases.default_linparams(), b=b)
    assert 1 <= res.iterations <= 30
    exact = _host(s, B, np.longdouble).bicgstab(b.astype(dtype).astype(np.longdouble), res.iterations)
    plain = _host(s, B, dtype).bicgstab(b.astype(dtype), res.iterations)
    assert np.finfo(np.longdouble).eps < 1e-18
    err = lambda y: np.linalg.norm((y - exact).reshape(-1, 5), axis=0)  # noqa: E731
    norm = np.linalg.norm(exact.reshape(-1, 5), axis=0)
    print(kind, form, res.iterations, "device", err(x) / norm, "plain", err(plain.astype(np.longdouble)) / norm)
    assert (err(x) <= 2.0 * err(plain.astype(np.longdouble)) + np.finfo(dtype).eps * norm).all()
