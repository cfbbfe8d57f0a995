"""GPU parity of scans of few points, whose rays are walked in segments that go
round the XCDs: cells and values against the oracle, bit for bit, into a new map
and into it again, and rays longer than the 16-bit walk takes."""
import numpy as np
import pytest

from conftest import assert_same_cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,voxel", [(1, 0.1), (2, 0.1), (63, 0.1), (64, 0.1), (65, 0.1), (129, 0.1), (513, 0.1),
                                     (4100, 0.1), (8128, 0.2), (8200, 0.2), (3, 0.001)])
def test_few_points(ctx, n, voxel):
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(n)
    d = rng.standard_normal((n, 3))
    pts = (d / np.linalg.norm(d, axis=1, keepdims=True) * rng.uniform(0.2, 40.0, (n, 1))).astype(np.float32)
    m, om = bx.ProbabilisticMap(ctx, voxel), oracle.ProbMap(voxel)
    for origin in ((0.3, -0.2, 1.1), (0.3, -0.2, 1.1), (1.3, 0.4, 1.0)):
        m.insert_point_cloud(pts, origin, 35.0)
        om.insert_point_cloud(pts, origin, 35.0)
    assert m.update_count == om.update_count
    assert_same_cells(m.cells(), om.cells(), f"{n} points")
    m.close()
    om.close()
