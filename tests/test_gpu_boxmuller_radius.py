"""The device's Box-Muller radius over every first uniform there is (2^23 of
them, and the values next to [1, 2)), bit for bit the oracle's."""
import numpy as np
import pytest

import esthera_amd as ea
import oracle as O

pytestmark = pytest.mark.gpu


def test_radius_of_every_uniform(engine):
    u = np.empty(2 * ((1 << 23) + 4), np.float32)
    u[0:2 << 23:2] = (np.arange(1 << 23, dtype=np.uint32) | np.uint32(0x3F800000)).view(np.float32)
    u[2 << 23::2] = [2.0, 1.5, np.nextafter(np.float32(2.0), np.float32(1.0)), 1.0]   # 2.0: ln 0
    u[1::2] = 1.25
    d = ea.DeviceBuffer.from_array(u)
    ea.check(ea.lib().esth_stage_boxmuller(d.ptr, u.size))
    got, want = d.to_array(np.uint32, u.size), O.boxmuller(u).view(np.uint32)
    bad = np.nonzero(got != want)[0]
    assert bad.size == 0, f"{bad.size} differ, first for {u[bad[0] & ~1]!r}"
