"""The solve's forms at the block counts where they change, and the divisions of its
preconditioner outside the fast form's range, against the FP32 oracle.

A workgroup of the solve keeps at most 64 blocks in one set of quads per wave, at most 256 in
four, streams up to 512 from memory and walks larger counts block by block; a set holds four
blocks, so counts that are not multiples of four leave its last one part full. Every form gives
the same bits: the fields, the State and the particles equal the oracle's.
"""
import numpy as np
import pytest

import oracle
from natray_amd import Sim, abi, scenes
from tests import helpers

pytestmark = pytest.mark.gpu


def solve_and_compare(s, groups, steps=2):
    s.scene.solve_groups = groups
    sim, orc = Sim.from_scene(s), oracle.Oracle.from_scene(s, "f32")
    for step in range(steps):
        for ph in range(abi.N_PHASES):
            sim.phase(ph)
            orc.phase(ph)
            if ph != abi.PHASE_SOLVE:
                continue
            a, b = sim.state(), orc.state()
            # A solve that stops at its start leaves no alpha and beta of its own.
            for k in ("n_blocks", "solve_iters", "unconverged", "rz", "b_norm", "r_norm") + (("alpha", "beta") if b.solve_iters else ()):
                x, y = getattr(a, k), getattr(b, k)
                assert x == y or (x != x and y != y), (groups, step, k, x, y)
            np.testing.assert_array_equal(sim.grid()["cf"], orc.grid()["cf"], err_msg=f"groups {groups} step {step}")
    np.testing.assert_array_equal(sim.particles(), orc.particles())
    n = sim.n_blocks()
    sim.close()
    orc.close()
    return n


# 32k particles in ~176 blocks, 262k in ~950 (four to a chunk).
@pytest.mark.parametrize("n,side,precision,groups,per_group", [
    (32768, 64, abi.CG_FP32, 1, (65, 256)),
    (32768, 64, abi.CG_FP32, 2, (65, 256)),
    (32768, 64, abi.CG_FP32, 3, (1, 64)),
    (32768, 64, abi.CG_FP32, 59, (1, 64)),
    (32768, 64, abi.CG_MIXED, 1, (65, 256)),
    (32768, 64, abi.CG_MIXED, 5, (1, 64)),
    (262144, 128, abi.CG_FP32, 1, (513, 4096)),
    (262144, 128, abi.CG_FP32, 3, (257, 512)),
    (262144, 128, abi.CG_FP32, 4, (65, 256)),
    (262144, 128, abi.CG_FP32, 15, (1, 80)),
    (262144, 128, abi.CG_FP32, 200, (1, 64)),
    (262144, 128, abi.CG_MIXED, 3, (257, 512)),
    (262144, 128, abi.CG_MIXED, 4, (65, 256)),
])
def test_forms(n, side, precision, groups, per_group):
    s = scenes.balloon_impact(side=side, n=n, seed=groups + 1, iters=400, capacity=4096, precision=precision, refresh_every=4)
    blocks = solve_and_compare(s, groups)
    assert per_group[0] <= -(-blocks // groups) <= per_group[1]


def test_ragged_blocks_and_few():
    """A few particles in a few blocks, spread so that faces are missing on every side."""
    rng = np.random.default_rng(3)
    for count in (1, 9, 120):
        P = helpers.records(rng.uniform(0.2, 0.8, (count, 3)), vel=rng.uniform(-2, 2, (count, 3)))
        for precond in (abi.PRECOND_BLOCK_SGS, abi.PRECOND_JACOBI):
            solve_and_compare(helpers.box_scene(P, side=32, precond=precond, gravity=9.81), 7)


@pytest.mark.parametrize("precision", [abi.CG_FP32, abi.CG_MIXED])
@pytest.mark.parametrize("what", ["divisor", "dividend", "zero"])
def test_divisions_outside_the_fast_range(what, precision):
    """A diagonal above 2^30 (cells of 1 m at steps of 20 ns), residuals below 2^-70, and a
    residual of zero."""
    side, per = 16, 8
    cells = np.stack(np.meshgrid(*[np.arange(5, 11)] * 3, indexing="ij"), -1).reshape(-1, 3)
    u = scenes.uniform01(5, cells.shape[0] * per * 3).reshape(-1, per, 3)
    pos = ((cells[:, None] + u) / side).reshape(-1, 3)
    speed = {"divisor": 3.0, "dividend": 1e-28, "zero": 0.0}[what]
    vel = speed * (scenes.uniform01(6, pos.size).reshape(-1, 3) - 0.5)
    s = helpers.box_scene(helpers.records(pos, vel=vel), side=side, precision=precision, gravity=0.0 if what != "divisor" else 9.81)
    if what == "divisor":
        s.params.origin[3] = 1.0
        s.particles[:, :3] *= side
        s.params.fluid[3] = 0.5
        s.scene.fixed_dt = 2e-8
    solve_and_compare(s, 3)


@pytest.mark.parametrize("iters", [1, 2, 3])
@pytest.mark.parametrize("groups", [1, 3])
def test_few_iterations(iters, groups):
    """Solves that end at their first iterations: the last two directions, one of them the solve's
    own start after a single iteration, are among the fields compared."""
    s = scenes.balloon_impact(side=64, n=32768, seed=2, iters=iters, capacity=4096)
    solve_and_compare(s, groups)


@pytest.mark.parametrize("refresh", [0, 3])
@pytest.mark.parametrize("n,side,groups,per_group", [
    (32768, 64, 1, (65, 256)),
    (32768, 64, 3, (1, 64)),
    (32768, 64, 59, (1, 64)),
    (262144, 128, 8, (65, 256)),
    (262144, 128, 16, (60, 64)),
    (262144, 128, 200, (1, 64)),
])
def test_pipelined_forms(n, side, groups, per_group, refresh):
    """The pipelined solve holds at most 64 blocks a workgroup on the chip and walks larger counts
    from memory; with replacements of the residual and without."""
    s = scenes.balloon_impact(side=side, n=n, seed=groups + 1, iters=400, capacity=4096, precision=abi.CG_PIPELINED,
                              refresh_every=refresh)
    blocks = solve_and_compare(s, groups)
    assert per_group[0] <= -(-blocks // groups) <= per_group[1]


def test_pipelined_ragged_blocks_and_few():
    rng = np.random.default_rng(3)
    for count in (1, 9, 120):
        P = helpers.records(rng.uniform(0.2, 0.8, (count, 3)), vel=rng.uniform(-2, 2, (count, 3)))
        for precond in (abi.PRECOND_BLOCK_SGS, abi.PRECOND_JACOBI):
            for iters in (1, 40):
                solve_and_compare(helpers.box_scene(P, side=32, precond=precond, gravity=9.81, precision=abi.CG_PIPELINED,
                                                    iters=iters), 7)
