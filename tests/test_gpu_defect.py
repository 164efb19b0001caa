"""The defect correction of the FP32 forms never leaves a larger residual than it was
given: an inner solve that its iteration limit ends with a grown residual is added
with the multiple that has the smallest one.  Blocks far from dominant, few
iterations, both SGS orders; the returned residual is that of the returned x
(1e-6 of the operator's size: x and b - A x in FP64 over FP32 or BF16 blocks).
"""
import numpy as np
import pytest

import cfdg
import cfdg.cases as cases
from test_gpu_multicolour import Host
from test_gpu_sliced import FORMS, _solver, _spmv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [cfdg.SGS_MULTICOLOUR, cfdg.SGS_SEQUENTIAL])
@pytest.mark.parametrize("form", ["fp32", "bf16"])
@pytest.mark.parametrize("kind, size", [("hex", (13, 11, 3)), ("tet", (7, 6, 5))])
def test_residual_does_not_grow(kind, size, form, order):
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
    kept = 0
    for seed in range(6):
        rng = np.random.default_rng(seed)
        w = rng.standard_normal(v.shape)
        w[dg] += 2.0 * np.eye(5)
        s.set_bsr_values(w)
        B = s.bsr_values()
        b = rng.standard_normal(5 * mesh.n_cells)
        for most in (1, 2, 5, 20):
            x, res = s.linear_solve(cases.default_linparams(rel_tol=1e-3, max_iter=most, order=order), b=b)
            if res.status == cfdg.DIVERGED:
                continue
            kept += 1
            assert res.final_residual <= res.initial_residual * (1.0 + 1e-12)
            true = np.linalg.norm(b - _spmv(rp, cols, B, x))
            size_ax = np.linalg.norm(_spmv(rp, cols, np.abs(B), np.abs(x)))
            assert abs(true - res.final_residual) <= 1e-6 * (np.linalg.norm(b) + size_ax)
    assert kept >= 20  # of 24


@pytest.mark.parametrize("form", ["fp32", "bf16"])
@pytest.mark.parametrize("kind, size", [("hex", (13, 11, 3)), ("tet", (7, 6, 5))])
def test_grown_correction_is_shortened(kind, size, form):
    """One pass of few iterations: where numpy's float32 correction doubles the residual, the
    solve returns the multiple of its own with the smallest one: b - A x orthogonal to
    A x.  1e-9: x = e - (1 - theta) e carries eps |e|, 1e-10 |x| with theta above 1e-6."""
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
    s.set_precision(cfdg.Precision.make(FORMS[form].block_storage, cfdg.PREC_FP32, max_outer=1))
    colour = s.sgs_row_groups(cfdg.SGS_MULTICOLOUR)[0]
    grown = 0
    for seed in range(6):
        rng = np.random.default_rng(seed)
        w = rng.standard_normal(v.shape)
        w[dg] += 2.0 * np.eye(5)
        s.set_bsr_values(w)
        B = s.bsr_values()
        b = rng.standard_normal(5 * mesh.n_cells)
        for most in (1, 2, 3):
            e = Host(rp, cols, dg, B, colour, np.float32).bicgstab(b.astype(np.float32), most).astype(np.float64)
            ae = _spmv(rp, cols, B, e)
            x, res = s.linear_solve(cases.default_linparams(rel_tol=1e-3, max_iter=most), b=b)
            if res.iterations != most or np.linalg.norm(b - ae) <= 2.0 * np.linalg.norm(b):
                continue
            grown += 1
            assert res.final_residual <= res.initial_residual
            ax = _spmv(rp, cols, B, x)
            assert np.linalg.norm(ax) > 1e-6 * np.linalg.norm(b)  # not just dropped
            assert abs((b - ax) @ ax) <= 1e-9 * np.linalg.norm(b - ax) * np.linalg.norm(ax)
    assert grown >= 6
