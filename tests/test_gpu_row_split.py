"""3D order 5 FP64: the row split's element groups, which meet at their own counters, against 4-wave
workgroups that split elements, from part of a tile to several tiles per workgroup."""
import numpy as np
import pytest

import dgk
from workloads import conf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", (0, 1))
@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 2, 2), (7, 5, 9), (10, 9, 8)])
def test_row_split_groups_agree_with_the_element_split(cells, order):
    """Both sum 252 products per value in FP64 in another order: per evaluation at most about 252 * 2^-53 =
    3e-14 of the terms' size, far below 1e-12 after three small steps (relative L2)."""
    print(f"cells {cells} order {order}", flush=True)
    m = dgk.gen_box(*cells, 1.0, 0.8, 0.7, 5, 0.05, 2, [1, 1, 2, 2, 1, 2], "1:Wall;2:Abs",
                    conf("Wall=Reflecting\nAbs=Absorbing\n"))
    u = np.random.default_rng(3).standard_normal((4, m.K * m.Np))
    out = []
    for shape in (0, 1):
        s = dgk.Solver(m, 340.0, 1.225, v0=(30.0, -10.0, 5.0), flux_sign=dgk.SIGN_STABLE)
        try:
            s.set_tile_shape(shape)
            s.set_launch(100, order)
            s.set_state(u)
            s.rk4(3, 1e-6)
            out.append(s.get_state())
        finally:
            s.close()
    assert np.linalg.norm(out[0] - out[1]) <= 1e-12 * np.linalg.norm(out[1])
