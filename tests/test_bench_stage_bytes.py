"""bench.py reports the bytes that the stage kernel moves, hand-counted here, for the single legs and the
batch groups."""
import inspect

import pytest

from test_bench_model import bench


def test_stage_bytes_hand_count():
    # 3D P3, 6 elements, 15 faces of which 6 on the boundary
    dof, trace, faces = 4 * 6 * 20, 2 * 9 * 10 * 4, 6 * 4
    # FP64: u in and V1 out; V1, u in and W, V2 out; V2, u in and V3 out; V3, W in and u out
    words = (2 + 4 + 3 + 3) / 4
    geometry = 6 * 9 * 8 + faces * (4 * 8 + 8)
    assert bench.stage_bytes(3, 3, 6, 15, 6, 8, False) == dof * words * 8 + trace * 8 + geometry
    # FP32 compensated: u in and A, V1 out; V1, u, A in and A, V2 out; V2, u, A in and A, V3 out; V3, u, A
    # in and u out, with a 2-byte low word in and out
    words = (3 + 5 + 5 + 4 + 1) / 4
    geometry = 6 * 9 * 4 + faces * (4 * 4 + 8)
    assert bench.stage_bytes(3, 3, 6, 15, 6, 4, True) == dof * words * 4 + trace * 4 + geometry


@pytest.mark.parametrize("leg", [bench.single_leg, bench.batch_leg])
def test_rooflines_count_them(leg):
    src = inspect.getsource(leg)
    assert "stage_bytes(" in src and "algorithmic_bytes(" not in src
