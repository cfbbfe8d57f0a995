"""GPU parity of the bulk cell calls (setValue, setCellOn, setCellOff in input
order) against the oracle at the sizes where their tiles and buckets change,
and where a bucket has more leaves or cells than its tables hold.  Cells,
values and prior states are compared bit for bit."""
import numpy as np
import pytest

from conftest import assert_same_cells, sorted_cells

pytestmark = pytest.mark.gpu


def _inputs(spread, n, seed):
    from bonxai_amd import scenes
    rng = np.random.default_rng(seed)
    if spread == "clusters":
        return scenes.clusters(seed=seed, n=n)
    if spread == "cube":  # few leaves, many inputs a cell
        return rng.integers(-32, 32, (n, 3)).astype(np.int32)
    if spread == "line":  # one leaf: its first row
        return np.stack([rng.integers(0, 2, n), np.zeros(n, np.int64), np.zeros(n, np.int64)], 1).astype(np.int32)
    side = int(np.ceil(n ** (1 / 3)))  # every input in a leaf of its own (two cells a side)
    at = rng.permutation(side ** 3)[:n]
    return (2 * np.stack(np.unravel_index(at, (side, side, side)), 1) - side).astype(np.int32)


@pytest.mark.parametrize("spread,n,bits,dtype", [
    ("clusters", 1, (2, 3), np.float32), ("clusters", 63, (2, 3), np.int64), ("clusters", 1023, (2, 3), np.float32),
    ("clusters", 1025, (2, 3), None), ("clusters", 16_385, (2, 3), np.uint8), ("clusters", 262_143, (2, 3), np.int64),
    ("clusters", 262_145, (2, 3), np.float32), ("clusters", 524_289, (3, 2), np.float32),
    ("clusters", 1_048_577, (2, 3), np.float32), ("clusters", 2_097_153, (2, 3), None),
    ("clusters", 4_194_305, (2, 3), np.float32),  # leaves created in a pass of their own
    ("cube", 400_000, (1, 4), np.float32),        # more cells a bucket than its table holds
    ("line", 70_000, (2, 1), np.int64),           # two cells
    ("apart", 600_000, (2, 1), np.float32),       # more leaves a bucket than its table holds
    ("apart", 30_000, (1, 1), None),              # more roots a tile than its table holds
])
def test_calls_in_order(ctx, spread, n, bits, dtype):
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(n)
    c = _inputs(spread, n, n % 1000)
    v = None if dtype is None else rng.integers(0, 200, n).astype(dtype)
    g, og = bx.VoxelGrid(ctx, 0.1, *bits, dtype=dtype), oracle.Grid(0.1, *bits, dtype=dtype)
    third = n // 3 + 1
    half, w = np.ascontiguousarray(c[::2]), None if v is None else np.ascontiguousarray(v[::2][::-1])
    off = np.concatenate([c[rng.permutation(n)[:third]], c[:1] + np.int32(100_000)])  # the last has no root
    if n > 1 << 22:
        third = n  # all of it in one call
    g.set_values(c[:third], None if v is None else v[:third])
    og.set_values(c[:third], None if v is None else v[:third])
    for what, got, want in (
            ("on", g.set_cells_on(c, v, True), og.set_cells_on(c, v)),
            ("off", g.set_cells_off(off, True), og.set_cells_off(off)),
            ("set", g.set_values(half, w, True), og.set_values(half, w))):
        assert np.array_equal(got, want), what
    if dtype is None:
        assert np.array_equal(sorted_cells(g.export()[0])[0], og.export()[0])
    else:
        assert_same_cells(g.export(), og.export(), f"{spread} {n}")
    assert g.active_cells_count() == og.active_cells_count()
    g.close()
    og.close()


def test_values_at_any_address(ctx):
    """8-byte values in a buffer that is not 8-byte aligned."""
    import bonxai_amd as bx
    c = _inputs("clusters", 5000, 4)
    v = np.arange(1, 5001, dtype=np.int64) << 20
    raw = ctx.to_device(np.concatenate([np.zeros(4, np.uint8), v.view(np.uint8)]))
    d = ctx.to_device(c)
    g, h = bx.VoxelGrid(ctx, 0.1, dtype=np.int64), bx.VoxelGrid(ctx, 0.1, dtype=np.int64)
    assert bx.lib().bxg_set_values(g._h, d.ptr, raw.ptr + 4, len(c), None) == bx.OK
    h.set_values(c, v)
    assert_same_cells(g.export(), sorted_cells(*h.export()), "unaligned values")
    g.close()
    h.close()
