"""A fused launch that leaves LDS for the generator beside it (robot arms of a
million particles and more): the same particles, weights and estimates as with
the sampling and the sort in two launches, bit for bit."""
import numpy as np
import pytest

import esthera_amd as ea

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,G,layout", [(512, 2048, ea.LAYOUT_SOA), (512, 3072, ea.LAYOUT_SOA), (256, 4096, ea.LAYOUT_AOS),
                                        (256, 6144, ea.LAYOUT_PACKED)])
def test_room_for_the_generator_equals_two_launches(m, G, layout, engine):
    d = ea.filter_desc(ea.MODEL_ROBOTARM5, m=m, G=G, t=1, topology=ea.TOPO_RING, resampler=ea.RESAMPLE_SYSTEMATIC,
                       weights=ea.WEIGHTS_LOG, seed=11, layout=layout)
    c, z = ea.RobotArm5Control(), ea.RobotArm5Measurement()
    for i in range(5):
        c.angles[i], z.angles[i] = 0.05, 2.35
    z.x, z.y = 1.0, 2.0
    fs = [ea.Filter(engine, d), ea.Filter(engine, d)]
    assert fs[0].set_fusion(True) and not fs[1].set_fusion(False)
    for f in fs:
        f.init_uniform(np.zeros(9, np.float32))
        for _ in range(6):
            f.step(c, z, 0.0589)
    (sa, wa), (sb, wb) = fs[0].particles(), fs[1].particles()
    assert np.array_equal(sa.view(np.uint32), sb.view(np.uint32)) and np.array_equal(wa.view(np.uint32), wb.view(np.uint32))
    assert bytes(fs[0].estimate()) == bytes(fs[1].estimate())
    for f in fs:
        f.close()
