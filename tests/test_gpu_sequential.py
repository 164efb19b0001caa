"""The sequential SGS order on either side of the row count up to which both
sweeps run in one launch with z in LDS (4,096 rows in FP64, 8,192 with FP32
vectors), at one row, less than a wave's twelve rows, levels that are not a
multiple of twelve, and rows with more blocks than are requested ahead
(tetrahedra), against a float64 numpy sweep in mesh order.

Tolerances: test_gpu_sliced.py.
"""
from concurrent.futures import ThreadPoolExecutor

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


@pytest.mark.parametrize("form", ["fp64", "bf16"])
def test_threads_with_systems_of_different_size(form):
    """The kernel's LDS limit is one for the process: a small system's call between
    another thread's large ones changes nothing."""
    sizes = [(16, 16, 16), (48, 8, 6), (13, 11, 12)] if form == "fp64" else [(32, 16, 16), (48, 8, 12), (13, 23, 12)]
    solvers = [_solver("hex", n, form)[1] for n in sizes]
    r = [np.random.default_rng(k).standard_normal(5 * s.n_cells) for k, s in enumerate(solvers)]
    alone = [s.sgs_apply(cfdg.SGS_SEQUENTIAL, x) for s, x in zip(solvers, r)]

    def work(k):
        return all(np.array_equal(solvers[k].sgs_apply(cfdg.SGS_SEQUENTIAL, r[k]), alone[k]) for _ in range(20))

    with ThreadPoolExecutor(len(sizes)) as pool:
        assert all(pool.map(work, range(len(sizes))))
