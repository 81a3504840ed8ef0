"""The next step's MTGP32 words in shares of the step's own launches: in the
resampling alone (few particles), split between the sampling and the
resampling, and over all three launches of an unfused step; through graph
replay, a switched-off prefetch, and a snapshot restored mid-run.  Particles
and weights equal the oracle's bit for bit after every step."""
import ctypes

import numpy as np
import pytest

import esthera_amd as ea
import oracle as O

pytestmark = pytest.mark.gpu

# m, G, landmarks, resampler: two rounds per stream, all in the resampling; 18 rounds, split
CASES = [(256, 64, 4, ea.RESAMPLE_SYSTEMATIC), (64, 100, 4, ea.RESAMPLE_ALIAS), (512, 512, 20, ea.RESAMPLE_ALIAS)]


def same(f, o, what):
    st, w = f.particles()
    ost, ow = o.read(3)
    assert np.array_equal(st.view(np.uint32), ost.view(np.uint32)), f"particles, {what}"
    assert np.array_equal(w.view(np.uint32), ow.view(np.uint32)), f"weights, {what}"


@pytest.mark.parametrize("m,G,L,res", CASES)
def test_carried_words_equal_oracle(m, G, L, res, engine):
    desc = ea.filter_desc(ea.MODEL_UNICYCLE, m=m, G=G, t=1, topology=ea.TOPO_RING, resampler=res,
                          weights=ea.WEIGHTS_LOG, seed=77)
    params, ctrl, meas, _ = ea.unicycle_scenario(77, L, 20.0, 10)
    fs = {k: ea.Filter(engine, desc, params) for k in ("plain", "two launches", "graph", "prefetch off and on")}
    fs["two launches"].set_fusion(False)
    fs["graph"].use_graph(True)
    o = O.Filter(desc, params, ctypes.sizeof(params))
    for f in list(fs.values()) + [o]:
        f.init_uniform(np.zeros(3, np.float32))
    snap = None
    for k in range(10):
        if k in (2, 5):
            fs["prefetch off and on"].set_prefetch(k == 5)
        for name, f in fs.items():
            f.step(ctrl[k], meas[k], 0.1)
        o.step(ctrl[k], meas[k], 0.1)
        for name, f in fs.items():
            same(f, o, f"{name}, step {k}")
        if k == 4:
            snap = fs["plain"].snapshot()
    r = ea.Filter(engine, desc, params)
    r.restore(snap)
    for k in range(5, 10):
        r.step(ctrl[k], meas[k], 0.1)
    same(r, o, "restored")
    for f in list(fs.values()) + [r]:
        f.close()
