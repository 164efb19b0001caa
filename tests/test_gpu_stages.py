"""Stage times (cfdg_stage_times), taken from the device clock at the stage
boundaries: positive for the stages that ran, zero for those that did not, and
together no longer than the host's clock around the call."""
import time

import numpy as np
import pytest

import cfdg
import cfdg.cases as cases
from helpers import perturbed_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [cfdg.SGS_MULTICOLOUR, cfdg.SGS_SEQUENTIAL])
@pytest.mark.parametrize("recon", [cfdg.FIRST_ORDER, cfdg.MUSCL])
def test_stage_times(order, recon):
    case = cases.ramp(ni=24, nj=16, nk=8)
    case.numerics.reconstruction = recon
    s = cfdg.Solver(cfdg.Mesh.generate(**case.mesh), case.numerics, case.bcs)
    assert not np.any(s.stage_times())
    s.set_state(perturbed_state(s, case))
    s.eval_residual()
    s.eval_residual()
    t0 = time.perf_counter()
    s.eval_residual()
    wall = 1e3 * (time.perf_counter() - t0)
    t = np.asarray(s.stage_times())
    assert t[0] > 0.0 and t[3] > 0.0 and not t[4:].any()
    assert (t[1:3] > 0.0).all() if recon == cfdg.MUSCL else not t[1:3].any()
    assert t.sum() <= wall
    lp = cases.default_linparams(order=order)
    s.implicit_step(lp)
    t0 = time.perf_counter()
    s.implicit_step(lp)
    wall = 1e3 * (time.perf_counter() - t0)
    t = np.asarray(s.stage_times())
    assert t[4] > 0.0 and t[5] > 0.0 and t.sum() <= wall


@pytest.mark.parametrize("recon", [cfdg.FIRST_ORDER, cfdg.MUSCL])
def test_timing_the_flux_kernel_leaves_the_stage_times(recon):
    case = cases.ramp(ni=24, nj=16, nk=8)
    case.numerics.reconstruction = recon
    s = cfdg.Solver(cfdg.Mesh.generate(**case.mesh), case.numerics, case.bcs)
    s.set_state(perturbed_state(s, case))
    s.implicit_step(cases.default_linparams())
    s.eval_residual()
    before = np.asarray(s.stage_times()).copy()
    assert s.time_flux_kernel(3) > 0.0
    assert np.array_equal(s.stage_times(), before)


def test_stage_times_of_a_mesh_without_boundary():
    """No ghost cells, so no kernel for their gradients: the stages around it keep
    their times."""
    case = cases.ramp(ni=24, nj=16, nk=8)
    m = cfdg.Mesh.generate(**case.mesh)
    a, n = m.arrays(), m.n_inner_faces
    a["face_nodes"] = a["face_nodes"][:a["face_nodes_off"][n]]
    a["face_nodes_off"] = a["face_nodes_off"][:n + 1]
    for k in a:
        if k.startswith("face_") and not k.startswith("face_nodes"):
            a[k] = a[k][:n]
    s = cfdg.Solver(cfdg.Mesh.from_arrays(a, 0), case.numerics, [])
    s.set_state(perturbed_state(s, case))
    s.eval_residual()
    t0 = time.perf_counter()
    s.eval_residual()
    wall = 1e3 * (time.perf_counter() - t0)
    t = np.asarray(s.stage_times())
    assert (t[:2] > 0.0).all() and t[3] > 0.0 and t.sum() <= wall
