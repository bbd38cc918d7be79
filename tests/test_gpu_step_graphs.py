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


# relative changes of the velocity between steps: each lowers the pressure's first
# residual against its last solution, so the iteration counts of the levels lie
# further apart than one graph's budgets cover
LEVELS = (1.0, 1e-2, 1e-4, 1e-6, 1e-8, 0.0)


class _Levels:
    """The pair on a channel of 9,000 nodes, stepped at a chosen level of pressure iterations."""

    def __init__(self):
        from nsfem_amd import fem, mesher
        m = mesher.channel_mesh(9000, seed=7)
        cond = fem.DfgConditions(viscosity=2.4e-3, peakVelocity=1.5, channelHeight=1.0)
        ctx = fem.ChorinContext(mesher.to_triangle_mesh(m), cond)
        self.tau = float(m["h"]) ** 2 / (700 * 2.4e-3)
        self.pair = []
        for captured in (1, 0):
            cfg = fem.ChorinConfig(fem.SolverConfig("pcg", 500, 1e-10, 1), fem.SolverConfig("pcg", 6000, 1e-10, 1), stepGraph=captured)
            self.pair.append(fem.Chorin(ctx, cfg))
        self.set_time_step(self.tau)
        y = ctx.velocity_mesh()[0][:, 1]
        self.u = np.concatenate([1.5 * 4 * y * (1 - y), np.zeros_like(y)]) + 0.02 * np.random.default_rng(3).standard_normal(2 * y.size)
        self.step(1.0)

    def set_time_step(self, tau):
        for ch in self.pair:
            ch.set_time_step(tau)

    def step(self, level):
        """Three steps, each from a velocity that differs by the level from the one before."""
        for k in range(3):
            for ch in self.pair:
                ch.upload_velocity(self.u * (1 + level * ((k + 1) % 2)))
            sc, sr = _step(*self.pair)
            assert (sc["itersTent"], sc["itersPressure"], sc["itersFinal"]) == (sr["itersTent"], sr["itersPressure"], sr["itersFinal"])
        for ch in self.pair:
            ch.upload_velocity(self.u)
        _step(*self.pair)
        return self.info()

    def info(self):
        i = self.pair[0].step_graph_info()
        return i["builds"], tuple(i["budgets"])


def test_kept_graphs_are_taken_again():
    s = _Levels()
    for level in (LEVELS[0], LEVELS[3]) * 2:
        s.step(level)
    builds, high = s.step(LEVELS[0])
    for _ in range(3):
        now, low = s.step(LEVELS[3])
        assert now == builds and low[1] < high[1]
        assert s.step(LEVELS[0]) == (builds, high)


def test_kept_graphs_end_with_their_time_step_and_options():
    """tau is an argument of the captured kernels; an option changes the launches."""
    s = _Levels()
    for level in (LEVELS[0], LEVELS[3]) * 2:
        s.step(level)
    for tau in (s.tau / 2, s.tau):
        before = s.info()[0]
        s.set_time_step(tau)
        for level in (LEVELS[0], LEVELS[3]) * 2:
            s.step(level)
        assert s.info()[0] >= before + 2  # one for each level at the least
    for kind in (1, 0):
        before = s.info()[0]
        for ch in s.pair:
            ch.set_solver_option("preconditioner", kind, "both")
        for level in (LEVELS[0], LEVELS[3]):
            s.step(level)
        assert s.info()[0] > before


def test_more_budgets_than_graphs_are_kept():
    """The oldest of four goes: coming back to it builds it anew."""
    s = _Levels()
    for level in LEVELS:
        s.step(level)
    first, budgets = s.info()[0], set()
    for level in LEVELS:
        budgets.add(s.step(level)[1])
    assert first > 4 and len(budgets) > 4 and s.info()[0] > first
