"""An estimate read as soon as the step's argmax has published it, while the
resampling still runs, equals the one read after the whole stream has ended,
bit for bit: before the first step, after every step, twice without a step,
after a queue longer than the poll, through graph replay, the cross-step
launch, the argmax in a launch of its own, and a restored snapshot."""
import numpy as np
import pytest

import esthera_amd as ea
from test_gpu_filter import run_pair

pytestmark = pytest.mark.gpu

# m, G, t, topology, resampler, weights, landmarks
CASES = [(256, 16, 1, ea.TOPO_RING, ea.RESAMPLE_SYSTEMATIC, ea.WEIGHTS_LOG, 4),
         (16, 33, 1, ea.TOPO_RING, ea.RESAMPLE_ALIAS, ea.WEIGHTS_LINEAR, 2),
         (128, 9, 0, ea.TOPO_NONE, ea.RESAMPLE_ALIAS, ea.WEIGHTS_LOG, 4),
         (512, 4096, 4, ea.TOPO_TORUS, ea.RESAMPLE_SYSTEMATIC, ea.WEIGHTS_LOG, 32),
         (64, 9000, 2, ea.TOPO_ALL2ALL, ea.RESAMPLE_MULTINOMIAL, ea.WEIGHTS_LOG, 4)]


@pytest.mark.parametrize("m,G,t,topo,res,weights,L", CASES)
def test_early_estimate_is_the_final_one(m, G, t, topo, res, weights, L, engine):
    desc = ea.filter_desc(ea.MODEL_UNICYCLE, m=m, G=G, t=t, topology=topo, resampler=res, weights=weights, seed=5)
    params, ctrl, meas, _ = ea.unicycle_scenario(5, L, 20.0, 8)
    early, late, graph = (ea.Filter(engine, desc, params) for _ in range(3))
    graph.use_graph(True)
    for f in (early, late, graph):
        f.init_uniform(np.zeros(3, np.float32))

    def check(what):
        got = [bytes(early.estimate()), bytes(graph.estimate()), bytes(early.estimate())]
        late.sync()
        want = bytes(late.estimate())
        late.sync()
        assert want == bytes(late.estimate())
        assert got == [want] * 3, what

    check("before the first step")
    snap = None
    for k in range(8):
        for f in (early, late, graph):
            f.step(ctrl[k], meas[k], 0.1)
        check(f"step {k}")
        if k == 3:
            snap = late.snapshot()
    for k in range(24):
        for f in (early, late, graph):
            f.step(ctrl[k % 8], meas[k % 8], 0.1)
    check("after a queue of steps")
    for f in (early, late, graph):
        f.restore(snap)
        for k in range(4, 6):
            f.step(ctrl[k], meas[k], 0.1)
    check("restored")
    for f in (early, late, graph):
        f.close()


@pytest.mark.parametrize("G", [1, 2, 127, 129, 1023, 1025, 2049, 4100])
def test_argmax_over_many_sub_filters(G, engine):
    """The argmax's loads ahead of each other, at the edges of its batches:
    the oracle's estimate, with the tolerances of the whole-filter tests."""
    desc = ea.filter_desc(ea.MODEL_RANDOMWALK3, m=16, G=G, t=0, topology=ea.TOPO_NONE,
                          resampler=ea.RESAMPLE_SYSTEMATIC, weights=ea.WEIGHTS_LOG, threshold=0.0, seed=G)
    run_pair(engine, desc, 3)
