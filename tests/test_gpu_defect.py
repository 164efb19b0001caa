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
from test_gpu_sliced import FORMS, _solver, _spmv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [cfdg.SGS_MULTICOLOUR, cfdg.SGS_SEQUENTIAL])
@pytest.mark.parametrize("form", ["fp32", "bf16"])
@pytest.mark.parametrize("kind, size", [("hex", (13, 11, 3)), ("tet", (7, 6, 5))])
def test_residual_does_not_grow(kind, size, form, order):
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
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
            assert res.final_residual <= res.initial_residual * (1.0 + 1e-12)
            true = np.linalg.norm(b - _spmv(rp, cols, B, x))
            size_ax = np.linalg.norm(_spmv(rp, cols, np.abs(B), np.abs(x)))
            assert abs(true - res.final_residual) <= 1e-6 * (np.linalg.norm(b) + size_ax)
