"""GPU parity of the walk over the winner list at the sizes where its tasks
change: batches of 64 winners (remainders, batches that hold several scans),
segments of short lists, whole rays in lockstep, rays on both sides of the
32-bit closed forms.  Bit-exact against the oracle."""
import numpy as np
import pytest

from conftest import assert_same_cells

pytestmark = pytest.mark.gpu


def _sphere(n, radius, seed):
    """n points about `radius` from the origin, one voxel each."""
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((n, 3))
    v *= radius * rng.uniform(0.7, 1.3, (n, 1)) / np.linalg.norm(v, axis=1, keepdims=True)
    return v.astype(np.float32)


def _check(c, scans, voxel, max_range, what):
    """The scans into maps of their own in one call, then the same points
    from a moved sensor into the filled maps."""
    import bonxai_amd as bx
    import oracle
    maps = [bx.ProbabilisticMap(c, voxel) for _ in scans]
    models = [oracle.ProbMap(voxel) for _ in scans]
    dev = [c.to_device(p) for p in scans]
    for o in ((0.01, 0.02, 0.03), (0.33, -0.41, 0.12)):
        bx.insert_batch(c, [(m, d, o, max_range) for m, d in zip(maps, dev)])
        for m, om, p in zip(maps, models, scans):
            om.insert_point_cloud(p, np.array(o), max_range)
            assert_same_cells(m.cells(), om.cells(), f"{what}, {len(p)} points, sensor {o}")
    for x in maps + models:
        x.close()
    for d in dev:
        d.free()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 4097])
def test_short_lists(ctx, n):
    """One scan: the rays are cut into segments, the last batch has a remainder."""
    _check(ctx, [_sphere(n, 8.0, n)], 0.1, 10.0, "short list")


def test_batches_of_several_scans(ctx):
    """Scans of a few winners each, so that a batch holds several."""
    _check(ctx, [_sphere(n, 5.0, n) for n in (3, 40, 30, 1, 200, 64, 17)], 0.1, 6.0, "several scans")


@pytest.mark.parametrize("setting", [
    {"small_ray_blocks_per_cu": 1, "ray_chunk": 64},
    {"small_ray_blocks_per_cu": 1, "ray_chunk": 1024, "ray_blocks_per_cu": 1, "leaf_blocks_per_cu": 1,
     "fresh_blocks_per_cu": 1},
    {"small_ray_blocks_per_cu": 1, "ray_block": 256, "ray_chunk": 192},
])
def test_long_lists(setting):
    """More batches than the grid cuts segments for: whole rays in lockstep,
    contiguous parts an XCD (the last one shorter), runs of batches, several
    rounds of a capped grid."""
    import bonxai_amd as bx
    c = bx.Context(0)
    for k, v in setting.items():
        c.set_tuning(k, v)
    _check(c, [_sphere(60_011, 9.0, 5)], 0.1, 10.0, str(setting))
    c.close()


@pytest.mark.parametrize("cells", [32_766, 32_767, 32_768, 40_000])
def test_long_rays(ctx, cells):
    """Rays of about 2^15 cells: closed forms in 32 and in 64 bits."""
    p = np.array([[cells, 7, -3], [-cells, cells - 5, 11], [100, -cells, cells]], np.float32) * np.float32(0.1)
    _check(ctx, [p + np.float32(0.05)], 0.1, 1e6, "long rays")


@pytest.mark.parametrize("nscans", [2, 8, 9])
def test_bucket_tiles(ctx, nscans):
    """Calls of several scans around the number of bucket tiles up to which
    the bucket scan sums the earlier tiles itself."""
    _check(ctx, [_sphere(300 + 37 * k, 4.0 + k, k) for k in range(nscans)], 0.1, 8.0, f"{nscans} scans")
