"""The sequential SGS order on either side of the row count up to which both
sweeps run in one launch with z in LDS (4,096 rows in FP64, 8,192 with FP32
vectors), at one row, less than a wave's twelve rows, levels that are not a
multiple of twelve, and rows with more blocks than are requested ahead
(tetrahedra), against a float64 numpy sweep in mesh order.

Tolerances: test_gpu_sliced.py.
"""
import numpy as np
import pytest

import cfdg
import cfdg.cases as cases
from test_gpu_sliced import FORMS, _solver, _spmv

pytestmark = pytest.mark.gpu


def _sequential(rp, cols, dg, B, r):
    n = len(dg)
    inv = np.linalg.inv(B[dg])
    z, r = np.zeros((n, 5)), r.reshape(-1, 5)
    for i in list(range(n)) + list(range(n - 1, -1, -1)):
        k = np.arange(rp[i], rp[i + 1])
        k = k[k != dg[i]]
        z[i] = inv[i] @ (r[i] - np.einsum("kij,kj->i", B[k], z[cols[k]]))
    return z.ravel()


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("kind, size", [("hex", (1, 1, 1)), ("hex", (3, 2, 1)), ("hex", (13, 11, 3)), ("tet", (7, 6, 5)),
                                        ("hex", (16, 16, 16)), ("hex", (17, 241, 1)), ("hex", (32, 16, 16)),
                                        ("tet", (11, 25, 5))])
def test_sweeps_match_numpy(kind, size, form):
    mesh, s, rp, cols, dg, v = _solver(kind, size, form)
    B = s.bsr_values()
    tol = 1e-13 if form == "fp64" else 1e-5
    for seed in (3, 4):  # nothing of the first call is left
        r = np.random.default_rng(seed).standard_normal(5 * mesh.n_cells)
        z = _sequential(rp, cols, dg, B, r)
        assert np.max(np.abs(s.sgs_apply(cfdg.SGS_SEQUENTIAL, r) - z)) <= tol * np.max(np.abs(z))
    b = np.random.default_rng(5).standard_normal(5 * mesh.n_cells)
    x, res = s.linear_solve(cases.default_linparams(rel_tol=1e-6, order=cfdg.SGS_SEQUENTIAL), b=b)
    if mesh.n_cells > 1:  # one block: s vanishes or not with the rounding of alpha
        assert res.status == cfdg.CONVERGED
        assert np.linalg.norm(b - _spmv(rp, cols, B, x)) <= 1.05e-6 * np.linalg.norm(b)
