"""Captured steps and what is done to the solvers between them: graphs hold the
solvers' buffers and launch shapes, so a change drops every kept one."""

import numpy as np
import pytest

from conftest import mesh_path

pytestmark = pytest.mark.gpu


def _pair(pressure="pcg"):
    """A stepper that captures its steps and one that does not."""
    from nsfem_amd import fem
    ctx = fem.ChorinContext(fem.TriangleMesh.load_gmsh(mesh_path("c3")), fem.DfgConditions(1e-3, 1.0))
    pair = []
    for captured in (1, 0):
        cfg = fem.ChorinConfig(fem.SolverConfig("pcg", 2000, 1e-13, 1), fem.SolverConfig(pressure, 8000, 1e-13, 1), stepGraph=captured)
        pair.append(fem.Chorin(ctx, cfg))
        pair[-1].set_time_step(1e-3)
    return pair


def _step(cap, reg, same=True):
    sc, sr = cap.step(), reg.step()
    (uc, pc), (ur, pr) = cap.download(), reg.download()
    if same:  # the same kernels in the same order
        assert np.array_equal(uc, ur) and np.array_equal(pc, pr)
    else:  # other launch shapes: both within the solves' 1e-13 of the same step
        assert np.max(np.abs(uc - ur)) <= 1e-10 * np.max(np.abs(ur))
        assert np.max(np.abs(pc - pr)) <= 1e-10 * np.max(np.abs(pr))
    return sc, sr


def test_autotuning_after_captured_steps_drops_their_graphs():
    """Autotuning reallocates the solvers' partial sums and block tables."""
    cap, reg = _pair()
    for _ in range(3):
        _step(cap, reg)
    builds = cap.step_graph_info()["builds"]
    cap.autotune(2)
    for _ in range(3):
        sc, _ = _step(cap, reg, same=False)
        assert sc["capturedStep"] == 1
    assert cap.step_graph_info()["builds"] > builds


def test_an_option_that_one_solver_rejects_still_drops_the_graphs():
    """"both" reaches the velocity solver before the pressure solver rejects
    it."""
    from nsfem_amd._lib import NsfemInvalidArgument
    cap, reg = _pair("amg_pcg")
    for _ in range(3):
        _step(cap, reg)
    builds = cap.step_graph_info()["builds"]
    for ch in (cap, reg):
        with pytest.raises(NsfemInvalidArgument):
            ch.set_solver_option("preconditioner", 1, "both")
    for _ in range(3):
        sc, _ = _step(cap, reg)
        assert sc["capturedStep"] == 1
    assert cap.step_graph_info()["builds"] > builds
