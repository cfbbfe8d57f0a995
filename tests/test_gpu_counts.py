"""The ray update counts of a batch whose wavefronts and workgroups hold
endpoints of several maps: each map's count and cells equal those of the same
scan inserted alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (63, 1, 64), (5, 300, 2, 255, 17, 1), (64, 192, 1000, 3, 3, 3, 3, 900)])
def test_batches_of_small_scans(ctx, sizes):
    import bonxai_amd as bx
    rng = np.random.default_rng(sum(sizes))
    scans = [((rng.random((n, 3)) * 4 - 2).astype(np.float32), rng.random(3)) for n in sizes]
    dev = [ctx.to_device(p) for p, _ in scans]
    together, alone = ([bx.ProbabilisticMap(ctx, 0.1) for _ in sizes] for _ in range(2))
    ctx.counting(True)
    try:
        for step in range(2):  # new leaves, then old ones
            bx.insert_batch(ctx, [(m, d, o + 0.3 * step, 3.0) for m, d, (_, o) in zip(together, dev, scans)])
            for m, d, (_, o) in zip(alone, dev, scans):
                m.insert_point_cloud(d, o + 0.3 * step, 3.0)
            for a, b in zip(together, alone):
                sa, sb = a.stats(), b.stats()
                for k in ("last_rays", "last_ray_updates", "last_ray_visits", "leaf_count"):
                    assert sa[k] == sb[k], (step, k)
                assert a.digest() == b.digest()
    finally:
        ctx.counting(False)
    for m in together + alone:
        m.close()
