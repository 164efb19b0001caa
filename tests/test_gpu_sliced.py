"""The multicolour kernels on the sliced block layout (one wave per slice of
64 rows of a colour, four up to 1,536 slices, or eight up to 384) at the sizes where the
layout can go wrong: one cell, less than a slice, ragged colours, several
colours with lower and upper blocks (tetrahedra), and just above the slice
count at which a launch changes its form.  Random diagonally dominant blocks;
the reference is a float64 numpy sweep over the colours.

Tolerances: a row of the product or of a sweep is at most 7 block products and
one 5x5 solve, about 50 rounded operations; two sweeps of a dominant matrix
do not amplify: 100 eps of the arithmetic, 1e-13 of the largest entry in FP64
(eps 1.1e-16, a factor 10 for the solve) and 1e-5 in FP32 (eps 6e-8).
"""
import numpy as np
import pytest

import cfdg
import cfdg.cases as cases

pytestmark = pytest.mark.gpu

FORMS = {
    "fp64": cfdg.Precision.make(),
    "fp32": cfdg.Precision.make(cfdg.PREC_FP32, cfdg.PREC_FP32),
    "bf16": cfdg.Precision.make(cfdg.PREC_BF16, cfdg.PREC_FP32),
    "fp64 blocks, fp32 krylov": cfdg.Precision.make(cfdg.PREC_FP64, cfdg.PREC_FP32),
}


def _case(kind, size):
    ni, nj, nk = size
    return (cases.ramp if kind == "hex" else cases.bump)(ni=ni, nj=nj, nk=nk, gradient="GREEN_GAUSS_CELL")


def _solver(kind, size, form):
    case = _case(kind, size)
    mesh = cfdg.Mesh.generate(**case.mesh)
    s = cfdg.Solver(mesh, case.numerics, case.bcs)
    s.set_precision(FORMS[form])
    rng = np.random.default_rng(11)
    rp, cols, dg = s.bsr_pattern()
    v = 0.2 * rng.standard_normal((len(cols), 5, 5)) / 5.0
    v[dg] = np.eye(5) * (1.5 + rng.random((mesh.n_cells, 1, 1))) + 0.3 * rng.standard_normal((mesh.n_cells, 5, 5)) / 5.0
    s.set_bsr_values(v)
    return mesh, s, rp, cols, dg, v


def _off_rows(rp, dg):
    rows = np.repeat(np.arange(len(dg)), np.diff(rp))
    off = np.ones(len(rows), bool)
    off[dg] = False
    return rows, off


def _spmv(rp, cols, B, x):
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    y = np.zeros((len(rp) - 1, 5))
    np.add.at(y, rows, np.einsum("kij,kj->ki", B, x.reshape(-1, 5)[cols]))
    return y.ravel()


def _sgs(rp, cols, dg, B, colour, r):
    rows, off = _off_rows(rp, dg)
    z = np.zeros((len(dg), 5))
    r = r.reshape(-1, 5)
    for c in list(range(colour.max() + 1)) + list(range(colour.max() - 1, -1, -1)):
        k = np.nonzero(off & (colour[rows] == c))[0]
        acc = r.copy()
        np.add.at(acc, rows[k], -np.einsum("kij,kj->ki", B[k], z[cols[k]]))
        i = colour == c
        z[i] = np.linalg.solve(B[dg[i]], acc[i][:, :, None])[:, :, 0]
    return z.ravel()


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("kind, size", [("hex", (1, 1, 1)), ("hex", (3, 2, 1)), ("hex", (13, 11, 3)), ("tet", (2, 1, 3)),
                                        ("tet", (7, 6, 5)), ("hex", (41, 40, 31)), ("hex", (64, 64, 49))])
def test_product_and_sweeps_match_numpy(kind, size, form):
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
    B = s.bsr_values()
    if form.startswith("fp64"):
        assert np.array_equal(B, v)
    r = np.random.default_rng(3).standard_normal(5 * mesh.n_cells)
    y = _spmv(rp, cols, B, r)
    assert np.max(np.abs(s.spmv(r) - y)) <= 1e-13 * np.max(np.abs(y))
    colour = s.sgs_row_groups(cfdg.SGS_MULTICOLOUR)[0]
    z = _sgs(rp, cols, dg, B, colour, r)
    tol = 1e-13 if form == "fp64" else 1e-5
    assert np.max(np.abs(s.sgs_apply(cfdg.SGS_MULTICOLOUR, r) - z)) <= tol * np.max(np.abs(z))


@pytest.mark.parametrize("form", ["fp64", "bf16"])
@pytest.mark.parametrize("kind, size", [("hex", (13, 11, 3)), ("tet", (7, 6, 5))])
def test_orders_share_a_context(kind, size, form):
    """The sequential sweep runs on a row-major copy of the blocks, the
    multicolour one on the sliced layout; a context that alternates between
    them gives the same bits as fresh contexts, and both solve the system to
    the tolerance asked for."""
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
    b = np.random.default_rng(5).standard_normal(5 * mesh.n_cells)
    B = s.bsr_values()
    lps = [cases.default_linparams(rel_tol=1e-8, max_iter=100, order=o)
           for o in (cfdg.SGS_SEQUENTIAL, cfdg.SGS_MULTICOLOUR)]
    none = cases.default_linparams(rel_tol=1e-8, max_iter=100)
    none.preconditioner = cfdg.PRECOND_NONE
    fresh = [_solver(kind, size, form)[1].linear_solve(lp, b=b)[0] for lp in lps + [none]]
    for k in (0, 1, 2, 0, 1, 1, 2, 0):
        x, res = s.linear_solve((lps + [none])[k], b=b)
        assert res.status == cfdg.CONVERGED
        assert np.array_equal(x, fresh[k])
        # the recurrence's residual stands for the true one up to rounding
        assert np.linalg.norm(b - _spmv(rp, cols, B, x)) <= 1.05e-8 * np.linalg.norm(b)
    s.set_bsr_values(2.0 * v)  # the copy follows the blocks
    for lp, x0 in zip(lps, fresh):
        assert np.allclose(s.linear_solve(lp, b=2.0 * b)[0], x0, rtol=0.0, atol=1e-6 * np.max(np.abs(x0)))


@pytest.mark.parametrize("form", sorted(FORMS))
def test_blocks_are_zero_until_set(form):
    """In a new context and after a change of the storage, also where the memory held
    another system's blocks before."""
    for size in ((41, 40, 31), (41, 40, 31), (13, 11, 3)):
        mesh, s, rp, cols, dg, v = _solver("hex", size, form)
        assert s.bsr_values().any()
        s.close()
        case = _case("hex", size)
        s = cfdg.Solver(mesh, case.numerics, case.bcs)
        assert not s.bsr_values().any()
        s.set_bsr_values(v)
        s.set_precision(cfdg.Precision.make(cfdg.PREC_BF16, cfdg.PREC_FP32))
        assert not s.bsr_values().any()
        s.set_precision(FORMS[form])
        if FORMS[form].block_storage != cfdg.PREC_BF16:
            assert not s.bsr_values().any()
        s.close()
