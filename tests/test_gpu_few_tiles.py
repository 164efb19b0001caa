"""The residual's forms for few tiles (at most 256, one per CU: two lanes per cell in
the gradient kernel, one face per lane in the flux kernel) and for more, on either
side of the line, with ragged tiles, every limiter and eddy viscosity: gradients,
limiters and residual against the oracle at the tolerances of test_gpu_parity.py.
"""
import numpy as np
import pytest

import cfdg
import cfdg.cases as cases
from helpers import assert_close_scaled
from test_gpu_parity import _pair, _rel_check

pytestmark = pytest.mark.gpu

SMALL = [((1, 1, 1), l) for l in ("VENKAT", "UNLIMITED")]
SMALL += [(n, l) for n in ((7, 5, 3), (33, 9, 5)) for l in ("VENKAT", "BARTH", "VAN_ALBADA", "UNLIMITED")]


@pytest.mark.parametrize("eddy", [False, True])
@pytest.mark.parametrize("size, limiter", SMALL + [((40, 40, 39), "VENKAT"), ((44, 40, 40), "VENKAT")])
def test_residual_matches_oracle(size, limiter, eddy):
    ni, nj, nk = size
    mesh, gpu, ora = _pair(cases.plate(ni=ni, nj=nj, nk=nk, limiter=limiter))
    tiles = gpu.gradient_form()[2]
    assert tiles <= 256 if size != (44, 40, 40) else tiles > 256
    if eddy:
        mut = 1e-4 * np.random.default_rng(1).random(gpu.n_total)
        for s in (gpu, ora):
            s.set_eddy_viscosity(mut)
    for s in (gpu, ora):
        s.eval_residual()
    (gg, pg), (go, po) = gpu.gradients(), ora.gradients()
    assert_close_scaled(gg, go, np.abs(go).max(axis=1, keepdims=True), 1e-12, "gradients")
    # a limiter is a ratio of differences of the gradients above
    assert np.max(np.abs(pg - po)) <= 1e-10
    Rg, lg = gpu.residual()
    Ro, lo = ora.residual()
    assert_close_scaled(Rg, Ro, ora.flux_scale(), 1e-12, "residual")
    _rel_check(lg, lo, 1e-12, "spectral radius")


def _stencil_equal(mesh, a, b):
    """Cells whose primitives, and those of all cells that share a node, agree in every bit."""
    off, nodes = mesh.array("cell_nodes_off"), mesh.array("cell_nodes")
    bad = (a[:, :mesh.n_cells] != b[:, :mesh.n_cells]).any(axis=0)
    cell = np.repeat(np.arange(mesh.n_cells), np.diff(off))
    touched = np.zeros(nodes.max() + 1, bool)
    touched[nodes[bad[cell]]] = True
    return ~np.bincount(cell[touched[nodes]], minlength=mesh.n_cells).astype(bool)


@pytest.mark.parametrize("kind, size, few", [("ramp", (2, 1, 1), True), ("ramp", (33, 9, 5), True), ("ramp", (97, 31, 9), True),
                                             ("ramp", (128, 128, 5), False), ("plate_sa", (33, 9, 5), True)])
def test_gradients_are_the_sequential_sums(kind, size, few):
    """Each gradient is one sum over the stencil in order, whatever the number of lanes
    that share a cell, so it equals the oracle's in every bit (and with it a cell's
    gradient does not depend on the number of tiles) -- where the primitives do, which
    are formed with another division order in places."""
    ni, nj, nk = size
    mesh, gpu, ora = _pair(getattr(cases, kind)(ni=ni, nj=nj, nk=nk))
    form, tiles = gpu.gradient_form()[:2]
    assert form == cfdg.GRAD_LDS and (tiles <= 256) == few
    if kind.endswith("_sa"):
        for s in (gpu, ora):
            s.set_turbulence(cases.turbulence(cases.plate_sa(ni=ni, nj=nj, nk=nk)))
    for s in (gpu, ora):
        s.eval_residual()
    same = _stencil_equal(mesh, gpu.primitives(), ora.primitives())
    assert same.mean() > 0.1
    n = mesh.n_cells
    gg, go = gpu.gradients()[0][:, :n], ora.gradients()[0][:, :n]
    assert np.array_equal(gg[:, same], go[:, same])
