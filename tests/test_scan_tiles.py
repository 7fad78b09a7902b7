"""Binning in domains of one scan tile (1,024 block slots), of exactly one, of one more, and of more
tiles than a workgroup has threads: the blocks, their particles and the counts against the FP32
oracle, with water in the first and last slots that can hold any.
"""
import numpy as np
import pytest

import oracle
from natray_amd import Sim, abi
from tests import helpers
from tests.test_gpu_parity import compare_grid, compare_sorted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(16, 16, 16), (32, 32, 64), (32, 36, 64), (272, 268, 264)])
@pytest.mark.parametrize("capacity", [512, 40])
def test_tiles(dims, capacity):
    rng = np.random.default_rng(7)
    h = np.float32(1.0 / 16)
    lo, hi = np.full(3, 5.0), np.asarray(dims) - 7.0
    cells = np.concatenate([lo + rng.integers(0, 2, (40, 3)), hi + rng.integers(0, 2, (40, 3)), rng.uniform(lo, hi, (20, 3)) // 1])
    pos = ((cells + rng.random(cells.shape)) * h).astype(np.float32)
    s = helpers.box_scene(helpers.records(pos, vel=rng.uniform(-1, 1, pos.shape)), side=16, capacity=capacity, iters=40)
    s.params.dims[:3] = list(dims)
    s.params.bdims[:3] = [n // 4 for n in dims]
    sim, orc = Sim.from_scene(s), oracle.Oracle.from_scene(s, "f32")
    for step in range(2):
        for ph in range(abi.N_PHASES):
            orc.phase(ph)
            if orc.state().overflow:
                with pytest.raises(abi.NatrayError, match="capacity"):
                    sim.phase(ph)
                return
            sim.phase(ph)
            if ph == abi.PHASE_BIN:
                assert sim.state().n_blocks == orc.state().n_blocks
                g = sim.grid()
                compare_grid(f"{dims} step {step}", g, orc.grid(), cf_fields=())
                compare_sorted(f"{dims} step {step}", sim, orc, g)
        assert sim.state().max_speed == orc.state().max_speed
    np.testing.assert_array_equal(sim.particles(), orc.particles())
    sim.close()
    orc.close()
