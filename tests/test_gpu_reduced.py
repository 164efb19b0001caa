"""BiCGSTAB with the multicolour sweeps against a plain float64 numpy BiCGSTAB with
the full sweeps and products, iterate by iterate: from a zero and from a given guess,
with two colours (hexahedra) and more (tetrahedra), ragged slices, and on either side
of the slice count at which a launch changes its form.  One cell, and a system whose
s vanishes when alpha rounds to 1, must end at the solution.

Tolerance: the iterates of the dominant matrix (condition number below 10) differ
by the rounding of a few hundred operations per row and iteration, and the
recurrence's scalars amplify it by less than the condition number per iteration:
1e-12 of the largest entry after three iterations.
"""
import numpy as np
import pytest

import cfdg
import cfdg.cases as cases
from test_gpu_sliced import FORMS, _sgs, _solver, _spmv

pytestmark = pytest.mark.gpu


def _bicgstab(A, M, b, x, iterations):
    r = b - A(x)
    r0, p, v = r.copy(), np.zeros_like(r), np.zeros_like(r)
    rho = alpha = omega = 1.0
    rho = r0 @ r
    for it in range(iterations):
        if it == 0:
            p = r.copy()
        else:
            rho_new = r0 @ r
            p = r + (rho_new / rho) * (alpha / omega) * (p - omega * v)
            rho = rho_new
        ph = M(p)
        v = A(ph)
        alpha = rho / (r0 @ v)
        s = r - alpha * v
        sh = M(s)
        t = A(sh)
        omega = (t @ s) / (t @ t)
        x = x + alpha * ph + omega * sh
        r = s - omega * t
    return x, np.linalg.norm(r)


@pytest.mark.parametrize("guess", [False, True])
@pytest.mark.parametrize("kind, size", [("hex", (3, 2, 1)), ("hex", (13, 11, 3)), ("tet", (2, 1, 3)), ("tet", (7, 6, 5)),
                                        ("tet", (11, 13, 9)), ("hex", (41, 40, 31)), ("hex", (64, 64, 49))])
def test_iterates_match_numpy(kind, size, guess):
    mesh, s, rp, cols, dg, v = _solver(kind, size, "fp64")
    colour = s.sgs_row_groups(cfdg.SGS_MULTICOLOUR)[0]
    rng = np.random.default_rng(17)
    b = rng.standard_normal(5 * mesh.n_cells)
    x0 = rng.standard_normal(5 * mesh.n_cells) if guess else np.zeros(5 * mesh.n_cells)
    A = lambda x: _spmv(rp, cols, v, x)  # noqa: E731
    M = lambda r: _sgs(rp, cols, dg, v, colour, r)  # noqa: E731
    for n in (1, 3) if mesh.n_cells < 20000 else (2,):
        lp = cases.default_linparams(rel_tol=1e-30, abs_tol=0.0, max_iter=n)
        x, res = s.linear_solve(lp, b=b, x0=x0 if guess else None)
        ref, rnorm = _bicgstab(A, M, b, x0, n)
        assert res.iterations == n
        assert np.max(np.abs(x - ref)) <= 1e-12 * np.max(np.abs(ref))
        assert abs(res.final_residual - rnorm) <= 1e-10 * np.linalg.norm(b)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("kind, size", [("hex", (13, 11, 3)), ("tet", (7, 6, 5)), ("tet", (41, 23, 19)), ("hex", (41, 40, 31)),
                                        ("hex", (64, 64, 49))])
def test_forms_reach_the_tolerance(kind, size, form):
    """More iterations than a batch, past the 32nd (true residual norm); the
    recurrence's residual stands for the true one up to rounding."""
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
    B = s.bsr_values()
    b = np.random.default_rng(5).standard_normal(5 * mesh.n_cells)
    # the FP32 Krylov forms gain a factor 10 in each of at most 8 passes
    for rel, most in ((1e-3, 100), (1e-10, 100), (0.0, 40)) if FORMS[form].krylov == cfdg.PREC_FP64 else ((1e-3, 100), (1e-6, 100)):
        lp = cases.default_linparams(rel_tol=rel, abs_tol=0.0, max_iter=most)
        x, res = s.linear_solve(lp, b=b)
        true = np.linalg.norm(b - _spmv(rp, cols, B, x)) / np.linalg.norm(b)
        if rel > 0.0:
            assert res.status == cfdg.CONVERGED and true <= 1.05 * rel
        else:
            assert true <= 1e-13  # rounding of b - A x at |A| |x| of a few |b|


def test_one_colour_and_exact_first_step():
    mesh, s, rp, cols, dg, v = _solver("hex", (1, 1, 1), "fp64")
    b = np.arange(1.0, 6.0)
    x, res = s.linear_solve(cases.default_linparams(rel_tol=1e-12), b=b)
    assert res.status == cfdg.CONVERGED
    assert np.allclose(x, np.linalg.solve(v[0], b), rtol=1e-12, atol=0.0)
    # no off-diagonal blocks: M = A, s = r - v vanishes when alpha rounds to 1
    for size in ((3, 2, 1), (4, 4, 4), (13, 11, 3)):
        mesh, s, rp, cols, dg, v = _solver("hex", size, "fp64")
        w = np.zeros_like(v)
        w[dg] = v[dg]
        s.set_bsr_values(w)
        for seed in range(4):
            b = np.random.default_rng(seed).standard_normal(5 * mesh.n_cells)
            x, res = s.linear_solve(cases.default_linparams(rel_tol=1e-10), b=b)
            ref = np.linalg.solve(w[dg], b.reshape(-1, 5, 1)).ravel()
            assert res.status == cfdg.CONVERGED
            assert np.max(np.abs(x - ref)) <= 1e-12 * np.max(np.abs(ref))
