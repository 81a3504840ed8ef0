"""Resampling by four waves per sub-filter (few sub-filters of many planes)
and, beyond, by one, at both sides of the line on a device of 256 compute
units: particles, weights and estimates of whole filters against the oracle."""
import pytest

import esthera_amd as ea
from test_gpu_filter import run_pair

pytestmark = pytest.mark.gpu

CASES = [(ea.MODEL_ROBOTARM5, 1024, 2, 9, ea.TOPO_RING, ea.RESAMPLE_MULTINOMIAL, ea.WEIGHTS_LINEAR, 0, 4),
         (ea.MODEL_ROBOTARM5, 1024, 4, 2, ea.TOPO_ALL2ALL, ea.RESAMPLE_SYSTEMATIC, ea.WEIGHTS_LOG, 1, 4),
         (ea.MODEL_DH6, 1024, 3, 1, ea.TOPO_RING, ea.RESAMPLE_SYSTEMATIC, ea.WEIGHTS_LOG, 0, 4),
         (ea.MODEL_DH6, 512, 256, 1, ea.TOPO_TORUS, ea.RESAMPLE_SYSTEMATIC, ea.WEIGHTS_LOG, 0, 2),
         (ea.MODEL_DH6, 512, 257, 1, ea.TOPO_RING, ea.RESAMPLE_MULTINOMIAL, ea.WEIGHTS_LOG, 0, 2),
         (ea.MODEL_ROBOTARM5, 1024, 769, 1, ea.TOPO_RING, ea.RESAMPLE_SYSTEMATIC, ea.WEIGHTS_LOG, 0, 1)]


@pytest.mark.parametrize("model,m,G,t,topo,res,weights,carry,steps", CASES)
@pytest.mark.parametrize("threshold", [1.0, 0.4])
def test_waves_per_sub_filter_equal_oracle(model, m, G, t, topo, res, weights, carry, steps, threshold, engine):
    if threshold < 1.0 and G > 4:
        pytest.skip("the gate is covered at the small sizes")
    desc = ea.filter_desc(model, m=m, G=G, t=t, topology=topo, resampler=res, weights=weights, carry=carry,
                          threshold=threshold, seed=23)
    run_pair(engine, desc, steps)
