"""The sort on packed keys (m >= 256) against the oracle's network, bit for
bit, over the key patterns where an order by (key, position) could differ from
the network's swaps: equal keys in groups of every size, zeros of both signs,
infinities, subnormals and NaN, mixed per sub-filter so that a launch holds
waves of both paths."""
import numpy as np
import pytest

import esthera_amd as ea
import oracle as O

pytestmark = pytest.mark.gpu

DB = ea.DeviceBuffer


def keys(kind, rng, m):
    k = rng.normal(-30.0, 8.0, m).astype(np.float32)
    if kind == 1:      # one pair of equal keys
        k[rng.integers(m)] = k[rng.integers(m)]
    elif kind == 2:    # groups of equal keys
        k = rng.integers(-9, 9, m).astype(np.float32)
    elif kind == 3:    # mostly underflowed weights
        k = np.where(rng.random(m) < 0.7, np.float32(0.0), rng.random(m, dtype=np.float32))
    elif kind == 4:    # weight 0 in the log domain, and an overflow
        k[rng.random(m) < 0.1] = -np.inf
        k[rng.random(m) < 0.01] = np.inf
    elif kind == 5:    # subnormals of both signs
        k = (rng.integers(-50, 50, m) * 1e-45).astype(np.float32)
        k[k == 0.0] = 0.0
    elif kind == 6:    # zeros of both signs
        k = np.where(rng.random(m) < 0.5, np.float32(-0.0), np.float32(0.0))
        k[rng.random(m) < 0.2] = 1.0
    elif kind == 7:    # NaN
        k[rng.random(m) < 0.02] = np.nan
    elif kind == 8:    # all equal
        k[:] = k[0]
    return k


@pytest.mark.parametrize("m", [256, 512, 1024])
@pytest.mark.parametrize("S", [3, 12])
def test_packed_sort_is_the_network(m, S, engine):
    rng = np.random.default_rng(m + S)
    G = 9 * 5 + 2          # every pattern in each wave of a work-group, and a partial work-group
    w = np.concatenate([keys(g % 9, rng, m) for g in range(G)])
    st = rng.normal(size=S * m * G).astype(np.float32)
    dw, dst, dout, dwin, dperm = DB.from_array(w), DB.from_array(st), DB(st.nbytes), DB(G * 8), DB(w.nbytes)
    ea.check(ea.lib().esth_stage_sort(dw.ptr, dst.ptr, dout.ptr, S, m, G, dwin.ptr, dperm.ptr))
    ow, oout, owin, operm = O.block_sort(w, st, S, m, G)
    for got, want in ((dperm.to_array(np.int32, w.size), operm),
                      (dw.to_array(np.uint32, w.size), ow.view(np.uint32)),
                      (dout.to_array(np.uint32, st.size), oout.view(np.uint32)),
                      (dwin.to_array(np.uint32, 2 * G), owin.view(np.uint32))):
        bad = np.nonzero(got != want)[0]
        assert bad.size == 0, f"{bad.size} differ, first in sub-filter {bad[0] // m % G}"
