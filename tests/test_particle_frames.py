"""Particles' places in cells, bit for bit: P2G, G2P and the block marks form (p - origin) / h by a
division whose divisor is known in advance. Particles on the cells' and blocks' faces and one float
beside them, for cell sizes that are no power of two, against the FP32 oracle.
"""
import numpy as np
import pytest

import oracle
from natray_amd import Sim, abi
from tests import helpers
from tests.test_gpu_parity import compare_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,origin", [
    (1.0 / 16, (0.0, 0.0, 0.0)),
    (0.0123, (-0.37, 0.11, 5.0)),
    (0.1, (1e-3, -1.0, 0.3)),
    (float(np.nextafter(np.float32(2.0), np.float32(0.0))), (-7.0, 0.0, 3.0)),
    (3.1e-4, (0.0, -1e-3, 0.02)),
])
def test_faces(h, origin):
    rng = np.random.default_rng(11)
    h, o = np.float32(h), np.asarray(origin, np.float32)
    cells = rng.integers(5, 11, (600, 3)).astype(np.float32)
    frac = rng.choice(np.float32([0.0, 0.5, 0.25, 0.77]), (600, 3))
    pos = o + (cells + frac) * h
    side = rng.integers(-1, 2, (600, 3))
    pos = np.where(side < 0, np.nextafter(pos, np.float32(-np.inf)), np.where(side > 0, np.nextafter(pos, np.float32(np.inf)), pos))
    P = helpers.records(pos, vel=rng.uniform(-1, 1, (600, 3)) * h, C=rng.uniform(-1, 1, (600, 9)))
    s = helpers.box_scene(P, side=16, iters=60, gravity=9.81 * float(h))
    s.params.origin[:3] = [float(v) for v in o]
    s.params.origin[3] = float(h)
    s.params.fluid[3] = 0.5 * float(h)
    sim, orc = Sim.from_scene(s), oracle.Oracle.from_scene(s, "f32")
    for step in range(2):
        for ph in range(abi.N_PHASES):
            sim.phase(ph)
            orc.phase(ph)
            if ph in (abi.PHASE_P2G, abi.PHASE_G2P):
                compare_grid(f"h {h} step {step} phase {ph}", sim.grid(), orc.grid(), acc=ph == abi.PHASE_P2G)
    assert sim.n_blocks() > 0
    np.testing.assert_array_equal(sim.particles(), orc.particles())
    sim.close()
    orc.close()
