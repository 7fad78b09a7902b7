"""A batch's default launch shape is one that the autotuner times: tuning can only replace it by a
faster one."""
import pytest

from natray_amd import Sim, abi
from natray_amd.batch import Batch
from tests.test_batch import small_set

pytestmark = pytest.mark.gpu


def test_the_tuner_times_the_default_shape():
    sims = [Sim.from_scene(s) for s in small_set(abi.CG_FP32)[:2]]
    b = Batch(sims)
    default = b.shape()
    tuned = b.tune(1, iters=400)
    assert f"blocks{default['blocks_per_cu']}_waves{default['waves_per_cu']}" in tuned["ms_per_step"]
    assert default["cells_per_cu"] == tuned["best"]["cells_per_cu"]
    assert len(tuned["ms_per_step"]) == 9
    b.close()
    for s in sims:
        s.close()
