"""set_state / get_state: the state is permuted on the device from and to a
staging buffer, and arrays of 2 MiB and more move through the pinned slots of
several threads in pieces of 1 MiB.  A round trip must give the same bits back,
at one cell, below and just above the line between the two copies, with a last
piece that is not full, with more pieces than slots, and with rows of a caller's
array that are longer than the cell count (whose tail is neither read nor
written).
"""
import ctypes as C

import numpy as np
import pytest

import cfdg
import cfdg.cases as cases

pytestmark = pytest.mark.gpu


# 5 planes of 8 bytes: 52,429 cells are 2 MiB; the last size is 20 pieces
@pytest.mark.parametrize("size", [(1, 1, 1), (13, 11, 3), (52, 48, 21), (107, 49, 10), (97, 73, 74)])
def test_state_round_trip(size):
    ni, nj, nk = size
    case = cases.ramp(ni=ni, nj=nj, nk=nk, gradient="GREEN_GAUSS_CELL")
    s = cfdg.Solver(cfdg.Mesh.generate(**case.mesh), case.numerics, case.bcs)
    n = s.n_cells
    rng = np.random.default_rng(n)
    for _ in range(2):  # the slots are used again
        U = rng.standard_normal((5, n))
        s.set_state(U)
        assert np.array_equal(s.get_state(), U)
    lib = cfdg.lib
    W = np.full((5, n + 7), np.nan)
    W[:, :n] = rng.standard_normal((5, n))
    assert lib.cfdg_set_state(s._h, W.ctypes.data_as(C.c_void_p), W.shape[1]) == 0
    V = np.full((5, n + 9), 3.0)
    assert lib.cfdg_get_state(s._h, V.ctypes.data_as(C.c_void_p), V.shape[1]) == 0
    assert np.array_equal(V[:, :n], W[:, :n]) and (V[:, n:] == 3.0).all()
    assert lib.cfdg_set_state(s._h, W.ctypes.data_as(C.c_void_p), n - 1) != 0
    assert np.array_equal(s.get_state(), W[:, :n])
