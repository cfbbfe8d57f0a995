"""GPU parity of one-scan calls on both sides of the size up to which winners
are listed in point order (16384 points), into an empty map and then into the
map in use, eager and allocation-free: cells and update counts against the
oracle, bit for bit."""
import numpy as np
import pytest

from conftest import assert_same_cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 257, 5000, 16_384, 16_385])
@pytest.mark.parametrize("noalloc", [False, True])
def test_scans_in_point_order(ctx, n, noalloc):
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(n)
    m, om = bx.ProbabilisticMap(ctx, 0.2), oracle.ProbMap(0.2)
    m.reserve(60_000, 4_000)
    for step in range(4):
        # several points a voxel, some beyond the range
        p = (rng.integers(-30, 30, (n, 3)) * 0.2 + 0.1 + 0.04 * rng.random((n, 3))).astype(np.float32)
        o = np.array([0.05, 0.3 * step, 0.1])
        if noalloc:
            d = ctx.to_device(p)
            m.insert_point_cloud_noalloc(d, o, 5.0)
            d.free()
        else:
            m.insert_point_cloud(p, o, 5.0)
        om.insert_point_cloud(p, o, 5.0)
        assert_same_cells(m.cells(), om.cells(), f"{n} points, scan {step}")
    m.close()
    om.close()
