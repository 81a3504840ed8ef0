"""The global top-t of the all-to-all exchange at the edges of its ranges
(candidates in registers up to 8 per thread of the work-group, read per round
beyond), with equal weights across threads and sub-filters: the exchange
equals the oracle's."""
import numpy as np
import pytest

import esthera_amd as ea
import oracle as O

pytestmark = pytest.mark.gpu

DB = ea.DeviceBuffer


@pytest.mark.parametrize("G,t", [(2, 3), (63, 1), (1024, 1), (205, 5), (2048, 4), (2731, 3)])
@pytest.mark.parametrize("values", [3, 1000])
def test_top_t_equals_oracle(G, t, values, engine):
    m, S = 16, 3
    rng = np.random.default_rng(G + values)
    w = -np.sort(-rng.integers(0, values, m * G).astype(np.float32).reshape(G, m), axis=1).ravel()
    st = rng.normal(size=S * m * G).astype(np.float32)
    dw, dst = DB.from_array(w), DB.from_array(st)
    ea.check(ea.lib().esth_stage_exchange(dst.ptr, dw.ptr, S, m, G, t, ea.TOPO_ALL2ALL, 0, 0))
    ost, ow = O.exchange(st, w, S, m, G, t, ea.TOPO_ALL2ALL)
    assert np.array_equal(dw.to_array(np.uint32, w.size), ow.view(np.uint32))
    assert np.array_equal(dst.to_array(np.uint32, st.size), ost.view(np.uint32))
