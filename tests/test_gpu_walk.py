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


@pytest.mark.parametrize("nscans", [16, 17])
def test_scans_as_arguments(ctx, nscans):
    """Descriptors passed as kernel arguments (up to 16 scans) and copied."""
    _check(ctx, [_sphere(100 + 11 * k, 3.0 + 0.2 * k, k) for k in range(nscans)], 0.1, 8.0, f"{nscans} scans")


@pytest.mark.parametrize("fresh_pass", [1, 0])
def test_passes_left_out(fresh_pass):
    """Maps the host knows to be empty, filled, or neither (an asynchronous
    insert under way), alone and together in one call, before and after a
    clear, and with rays due from addHitPoint."""
    import bonxai_amd as bx
    import oracle
    c = bx.Context(0)
    c.set_tuning("fresh_pass", fresh_pass)
    pts = [_sphere(2_000, 6.0 + k, k) for k in range(3)]
    dev = [c.to_device(p) for p in pts]
    o = np.array([0.1, 0.2, 0.3])
    m, om = bx.ProbabilisticMap(c, 0.1), oracle.ProbMap(0.1)
    for rep in range(2):
        for d, p in zip(dev, pts):  # empty, then under way, then filled
            m.insert_point_cloud(d, o, 9.0, sync=False)
            om.insert_point_cloud(p, o, 9.0)
        assert m.sync() == 0
        assert_same_cells(m.cells(), om.cells(), f"asynchronous, round {rep}")
        m.insert_point_cloud(dev[0], o, 9.0)
        om.insert_point_cloud(pts[0], o, 9.0)
        assert_same_cells(m.cells(), om.cells(), f"filled, round {rep}")
        m.clear()
        om.close()
        om = oracle.ProbMap(0.1)
        m.update_count = 1
    # one call over an empty, a filled and a cleared map
    others = [bx.ProbabilisticMap(c, 0.1) for _ in range(2)]
    models = [om, oracle.ProbMap(0.1), oracle.ProbMap(0.1)]
    others[0].insert_point_cloud(dev[1], o, 9.0)
    models[1].insert_point_cloud(pts[1], o, 9.0)
    maps = [m] + others
    bx.insert_batch(c, [(x, dev[2], o, 9.0) for x in maps])
    for x, model in zip(maps, models):
        model.insert_point_cloud(pts[2], o, 9.0)
        assert_same_cells(x.cells(), model.cells(), "one call")
    # rays due into an empty map
    e, oe = bx.ProbabilisticMap(c, 0.1), oracle.ProbMap(0.1)
    for x in ([1.0, 2.0, 0.5], [-3.0, 0.2, 1.1]):
        e.add_hit_point(x)
        oe.add_hit_point(x)
    e.insert_point_cloud(pts[0], o, 9.0)
    oe.insert_point_cloud(pts[0], o, 9.0)
    assert_same_cells(e.cells(), oe.cells(), "rays due")
    for x in maps + models + [e, oe]:
        x.close()
    c.close()


@pytest.mark.parametrize("bits", [(1, 3), (2, 1), (3, 2), (4, 2), (4, 4)])
def test_new_entries_of_other_grids(ctx, bits):
    """Leaf creation with 1, 8 and 64 words of wanted leaves a root (and roots
    of fewer than 64 leaves): same cells, and exactly the leaves the cells and
    rays need (each holds a cell that is on, every scan cell being on)."""
    import bonxai_amd as bx
    import oracle

    m = bx.ProbabilisticMap.__new__(bx.ProbabilisticMap)
    bx.VoxelGrid.__init__(m, ctx, 0.1, *bits, np.uint32, _flags=bx.MAP_PROBABILISTIC)
    om = oracle.ProbMap(0.1)
    for k in range(3):
        p = _sphere(3_000, 9.0, 60 + k)
        o = np.array([0.5 * k, -0.3 * k, 0.05])
        m.insert_point_cloud(p, o, 10.0)
        om.insert_point_cloud(p, o, 10.0)
        assert_same_cells(m.cells(), om.cells(), f"bits {bits}, scan {k}")
        leaves = np.unique(om.cells()[0] >> bits[1], axis=0)
        assert m.stats()["leaf_count"] == len(leaves)
    m.close()
    om.close()


def test_leaves_made_and_removed_between_scans(ctx):
    """Leaves that bulk calls create, and leaves that releaseUnusedMemory
    removes, between the scans of one map: the scan's bits of existing leaves
    are hints, and no leaf is made twice or missed."""
    import bonxai_amd as bx
    import oracle
    m, om = bx.ProbabilisticMap(ctx, 0.1), oracle.ProbMap(0.1)
    a, b = _sphere(2_000, 5.0, 1), _sphere(2_000, 7.0, 2)
    far = np.stack([np.arange(400) % 100 - 50, np.arange(400) // 100 * 9, np.full(400, 3)], 1).astype(np.int32)
    words = np.full(len(far), (1000 << 4) | 3, np.uint32)
    m.set_values(far, words)
    om.grid.set_values(far, words)
    for p, o in ((a, [0.1, 0.2, 0.3]), (b, [0.4, 0.2, 0.3])):
        m.insert_point_cloud(p, np.array(o), 8.0)
        om.insert_point_cloud(p, np.array(o), 8.0)
    assert_same_cells(m.cells(), om.cells(), "after bulk calls")
    c = om.cells()[0]
    gone = c[c[:, 0] > 10]
    m.set_cells_off(gone)
    om.grid.set_cells_off(gone)
    m.release_unused_memory()
    om.grid.release_unused()
    for p, o in ((b, [0.2, 0.2, 0.3]), (a, [0.1, 0.3, 0.3])):
        m.insert_point_cloud(p, np.array(o), 8.0)
        om.insert_point_cloud(p, np.array(o), 8.0)
    assert_same_cells(m.cells(), om.cells(), "after releaseUnusedMemory")
    assert m.stats()["leaf_count"] == len(np.unique(om.cells()[0] >> 3, axis=0))
    m.close()
    om.close()


def test_marks_of_many_lives(ctx):
    """A map cleared more often than the marks have values: every life's scans
    read only their own marks, though the pool keeps the bytes of earlier ones
    (scans alternate, so that leaves reuse indices with other cells marked)."""
    import bonxai_amd as bx
    import oracle
    pts = [_sphere(300, 2.0, 1), _sphere(300, 3.0, 2)]
    o = np.array([0.1, 0.0, 0.2])
    want = []
    for k in range(2):
        om = oracle.ProbMap(0.1)
        om.insert_point_cloud(pts[k], o, 2.5)
        om.insert_point_cloud(pts[1 - k], o, 2.5)
        want.append((om.cells(), om.digest()))
        om.close()
    m = bx.ProbabilisticMap(ctx, 0.1)
    dev = [ctx.to_device(p) for p in pts]
    for life in range(270):
        k = life % 2
        m.update_count = 1
        m.insert_point_cloud(dev[k], o, 2.5, sync=False)
        m.insert_point_cloud(dev[1 - k], o, 2.5, sync=False)
        assert m.digest() == want[k][1], f"life {life}"
        if life in (0, 126, 127, 128, 255):
            assert_same_cells(m.cells(), want[k][0], f"life {life}")
        m.clear()
    m.close()
