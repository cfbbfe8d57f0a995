"""GPU parity of the bulk cell calls where the leaves of a bucket are more than
those whose mask bits are gathered in LDS (256; 32 of 16^3 cells), and more than
its table holds (2048).  Cells, values and prior states are compared bit for bit."""
import numpy as np
import pytest

from conftest import assert_same_cells, sorted_cells

pytestmark = pytest.mark.gpu


def _scattered(n, leaves, lb, seed):
    """n cells (some of them twice) in that many leaves, every fourth one of a cube."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil((4 * leaves) ** (1 / 3)))
    at = np.stack(np.unravel_index(rng.permutation(side ** 3)[:leaves], (side,) * 3), 1) - side // 2
    which = np.concatenate([np.arange(leaves), rng.integers(0, leaves, n - leaves)])[rng.permutation(n)]
    return ((at[which] << lb) + rng.integers(0, 1 << lb, (n, 3))).astype(np.int32)


@pytest.mark.parametrize("n,leaves,bits,dtype", [
    (16_000, 16_000, (2, 3), np.float32),   # about 64 leaves a bucket
    (260_000, 65_000, (2, 3), np.float32),  # 127
    (260_000, 131_000, (2, 3), np.int64),   # 256, some buckets more
    (520_000, 300_000, (2, 2), np.float32),  # 586
    (60_000, 16_000, (2, 4), np.float32),   # 31, some more
    (60_000, 30_000, (2, 4), np.int32),     # 59
    (130_000, 100_000, (3, 3), None),
    (130_000, 100_000, (2, 3), np.uint8),
])
def test_scattered_calls(ctx, n, leaves, bits, dtype):
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(n)
    c = _scattered(n, leaves, bits[1], leaves)
    v = None if dtype is None else rng.integers(1, 200, n).astype(dtype)
    g, og = bx.VoxelGrid(ctx, 0.1, *bits, dtype=dtype), oracle.Grid(0.1, *bits, dtype=dtype)
    some = c[rng.permutation(n)[: n // 2]]
    w = None if v is None else v[::-1][: n // 2]
    g.set_values(c[: n // 3], None if v is None else v[: n // 3])
    og.set_values(c[: n // 3], None if v is None else v[: n // 3])
    for what, got, want in (
            ("set", g.set_values(c, v, True), og.set_values(c, v)),
            ("off", g.set_cells_off(some, True), og.set_cells_off(some)),
            ("on", g.set_cells_on(c, v, True), og.set_cells_on(c, v)),
            ("off again", g.set_cells_off(c[: n // 4], True), og.set_cells_off(c[: n // 4]))):
        assert np.array_equal(got, want), what
    g.set_values(some, w)
    og.set_values(some, w)
    if dtype is None:
        assert np.array_equal(sorted_cells(g.export()[0])[0], og.export()[0])
    else:
        assert_same_cells(g.export(), og.export(), f"{n} {leaves}")
    assert g.active_cells_count() == og.active_cells_count()
    g.close()
    og.close()


def test_more_leaves_a_bucket_than_its_table(ctx):
    """9M cells, each in a leaf of its own: 2,200 leaves a bucket."""
    import bonxai_amd as bx
    n, half = 9_000_000, 4_500_000
    side = 209
    at = np.random.default_rng(9).permutation(side ** 3)[:n]
    c = (2 * np.stack(np.unravel_index(at, (side,) * 3), 1)).astype(np.int32)
    g = bx.VoxelGrid(ctx, 0.1, 4, 1, dtype=None)
    assert not g.set_cells_on(c[:half], None, True).any()
    assert np.array_equal(g.set_values(c, None, True), np.arange(n) < half)
    assert g.active_cells_count() == n
    assert g.set_cells_off(c[half // 2:], True).all()
    assert g.active_cells_count() == half // 2
    assert np.array_equal(g.lookup(c)[1], np.arange(n) < half // 2)
    g.close()


@pytest.mark.parametrize("dtype", [np.float32, np.int64])
@pytest.mark.parametrize("shift", [1, 2])
def test_values_at_odd_addresses(ctx, dtype, shift):
    """Values in a device buffer that no word of theirs is aligned in."""
    import bonxai_amd as bx
    L = bx.lib()
    n = 5000
    c = _scattered(n, 800, 3, 8)
    v = (np.arange(1, n + 1) * 3).astype(dtype)
    raw = ctx.to_device(np.concatenate([np.zeros(shift, np.uint8), v.view(np.uint8)]))
    d = ctx.to_device(c)
    for call, host in ((L.bxg_set_values, "set_values"), (L.bxg_set_cells_on, "set_cells_on")):
        g, h = bx.VoxelGrid(ctx, 0.1, dtype=dtype), bx.VoxelGrid(ctx, 0.1, dtype=dtype)
        assert call(g._h, d.ptr, raw.ptr + shift, n, None) == bx.OK
        getattr(h, host)(c, v)
        assert_same_cells(g.export(), sorted_cells(*h.export()), host)
        g.close()
        h.close()


@pytest.mark.parametrize("n,bits,dtype", [
    (1000, (2, 3), np.float32), (1024, (2, 3), np.int64), (5000, (2, 3), np.float32), (60_000, (2, 3), np.int32),
    (300_000, (2, 2), None), (300_000, (2, 4), np.float32), (600_000, (2, 3), np.uint8), (1_100_000, (2, 3), np.float32)])
@pytest.mark.parametrize("kind", ["cell", "leaf", "half"])
def test_crowded_leaves(ctx, n, bits, dtype, kind):
    """A leaf or a cell with a large part of the inputs, whose tiles leave out
    those that no result needs."""
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(n)
    side = 1 << bits[1]
    c = np.zeros((n, 3), np.int64) if kind == "cell" else rng.integers(0, side, (n, 3))
    if kind != "leaf":
        c = np.where(rng.random((n, 1)) < 0.5, c, rng.integers(-100, 100, (n, 3)))
    c = np.ascontiguousarray(c.astype(np.int32))
    v = None if dtype is None else rng.integers(1, 200, n).astype(dtype)
    g, og = bx.VoxelGrid(ctx, 0.1, *bits, dtype=dtype), oracle.Grid(0.1, *bits, dtype=dtype)
    part, w = c[n // 5:], None if v is None else v[n // 5:]
    for what, got, want in (
            ("on", g.set_cells_on(part, w, True), og.set_cells_on(part, w)),
            ("set", g.set_values(c, v, True), og.set_values(c, v)),
            ("off", g.set_cells_off(part, True), og.set_cells_off(part))):
        assert np.array_equal(got, want), what
    back = None if v is None else np.ascontiguousarray(v[::-1])
    g.set_values(c, back)
    og.set_values(c, back)
    if dtype is None:
        assert np.array_equal(sorted_cells(g.export()[0])[0], og.export()[0])
    else:
        assert_same_cells(g.export(), og.export(), f"{kind} {n}")
    assert g.active_cells_count() == og.active_cells_count()
    g.close()
    og.close()


@pytest.mark.parametrize("n,span", [(1, 16), (4000, 16), (40_000, 32), (300_000, 48), (1_100_000, 40)])
def test_dense_leaves_of_16(ctx, n, span):
    """Leaves of 16^3 cells, of which a bucket has an eighth: created by one of
    the workgroups that share them."""
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(n)
    c = rng.integers(-span, span, (n, 3)).astype(np.int32)
    v = rng.integers(1, 1 << 30, n).astype(np.int32)
    dc, dv, was = ctx.to_device(c), ctx.to_device(v), ctx.array(n, np.uint8)
    for bits in ((1, 4), (4, 4)):
        g, og = bx.VoxelGrid(ctx, 0.1, *bits, dtype=np.int32), oracle.Grid(0.1, *bits, dtype=np.int32)
        for _ in range(2):
            assert bx.lib().bxg_set_values(g._h, dc.ptr, dv.ptr, n, was.ptr) == bx.OK
            assert g.sync() == bx.OK
            assert np.array_equal(was.numpy(), og.set_values(c, v))
            assert_same_cells(g.export(), og.export(), f"{n} {bits}")
            off = c[: n // 2]
            assert np.array_equal(g.set_cells_off(off, True), og.set_cells_off(off))
        assert np.array_equal(g.set_cells_on(c, v, True), og.set_cells_on(c, v))
        assert_same_cells(g.export(), og.export(), f"{n} {bits}")
        g.close()
        og.close()
