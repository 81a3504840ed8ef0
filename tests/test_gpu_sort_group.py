"""The fused sampling and sort whose gather is shared by the work-group
(m >= 256) against the oracle, bit for bit: work-groups of two waves and of
four, three planes (fewer than waves) to twelve, the robot arm at m = 1024,
candidates of the exchange from every plane."""
import numpy as np
import pytest

import esthera_amd as ea
from test_gpu_filter import run_pair

pytestmark = pytest.mark.gpu

CASES = [(ea.MODEL_ROBOTARM5, 1024, 3, 8), (ea.MODEL_ROBOTARM5, 256, 5, 2), (ea.MODEL_DH6, 512, 3, 1),
         (ea.MODEL_DH6, 256, 4, 9), (ea.MODEL_UNICYCLE, 256, 3, 4), (ea.MODEL_RANDOMWALK3, 1024, 2, 17)]


@pytest.mark.parametrize("model,m,G,t", CASES)
def test_shared_gather_equals_oracle(model, m, G, t, engine):
    desc = ea.filter_desc(model, m=m, G=G, t=t, topology=ea.TOPO_RING, resampler=ea.RESAMPLE_SYSTEMATIC,
                          weights=ea.WEIGHTS_LOG, seed=61)
    f = ea.Filter(engine, desc, None if model == ea.MODEL_ROBOTARM5 else
                  {ea.MODEL_DH6: lambda: ea.dh6_scenario(7, 2)[0],
                   ea.MODEL_UNICYCLE: lambda: ea.unicycle_scenario(7, 4, 20.0, 2)[0],
                   ea.MODEL_RANDOMWALK3: lambda: ea.randomwalk3_scenario(7, 2)[0]}[model]())
    assert f.set_fusion(True), "the fused launch is expected here"
    f.close()
    run_pair(engine, desc, 6)
