"""MTGP32 words of several steps per launch on the second stream, in blocks of
three and four steps, and inline words whose steps record no event, through
graph replay, prefetch switched off and on in the middle of a block, per-stage
timing and a snapshot restored mid-block: particles and weights equal the
oracle's bit for bit."""
import ctypes

import numpy as np
import pytest

import esthera_amd as ea
import oracle as O
from test_gpu_carried_words import same

pytestmark = pytest.mark.gpu

# block steps, landmarks, sub-filters of 512
CASES = [(0, 40, 64), (3, 4, 96), (4, 4, 96)]


@pytest.mark.parametrize("block,L,G", CASES)
def test_blocks_equal_oracle(block, L, G, engine, monkeypatch):
    if block:
        monkeypatch.setenv("ESTH_RNG_BLOCK_STEPS", str(block))
    desc = ea.filter_desc(ea.MODEL_UNICYCLE, m=512, G=G, t=1, topology=ea.TOPO_RING,
                          resampler=ea.RESAMPLE_SYSTEMATIC, weights=ea.WEIGHTS_LOG, seed=19)
    params, ctrl, meas, _ = ea.unicycle_scenario(19, L, 40.0, 14)
    fs = {k: ea.Filter(engine, desc, params) for k in ("plain", "graph", "prefetch off and on", "timed in between")}
    assert fs["plain"].rng_mode() == ((False, block) if block else (True, 1))
    fs["graph"].use_graph(True)
    o = O.Filter(desc, params, ctypes.sizeof(params))
    for f in list(fs.values()) + [o]:
        f.init_uniform(np.zeros(3, np.float32))
    snap = None
    for k in range(14):
        if k in (3, 5, 8, 9):
            fs["prefetch off and on"].set_prefetch(k in (5, 9))
        if k in (4, 10):
            fs["timed in between"].set_timing(2 if k == 4 else 0)
        for f in list(fs.values()) + [o]:
            f.step(ctrl[k], meas[k], 0.1)
        if k in (3, 4, 5, 9, 10, 13):
            for name, f in fs.items():
                same(f, o, f"{name}, step {k}")
        if k == 5:
            snap = fs["plain"].snapshot()
    r = ea.Filter(engine, desc, params)
    r.restore(snap)
    for k in range(6, 14):
        r.step(ctrl[k], meas[k], 0.1)
    same(r, o, "restored")
    for f in list(fs.values()) + [r]:
        f.close()


def test_block_length_by_size(engine):
    """Four steps where two blocks stay within the cache, fewer beyond."""
    for m, G, want in ((128, 3001, 4), (512, 4096, 3)):
        desc = ea.filter_desc(ea.MODEL_RANDOMWALK3 if m == 128 else ea.MODEL_UNICYCLE, m=m, G=G, t=1,
                              topology=ea.TOPO_RING, resampler=ea.RESAMPLE_SYSTEMATIC, weights=ea.WEIGHTS_LOG, seed=3)
        p = ea.randomwalk3_scenario(3, 1)[0] if m == 128 else ea.unicycle_scenario(3, 4, 20.0, 1)[0]
        f = ea.Filter(engine, desc, p)
        assert f.rng_mode() == (False, want)
        f.close()
