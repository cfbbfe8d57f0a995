"""GPU tests of bulk cell calls that the leaf pool is too small for: such a call
sets no cell, and repeated it answers as if the failed one had not been made.
Cells, values and prior states are compared bit for bit with the oracle."""
import numpy as np
import pytest

from conftest import assert_same_cells

pytestmark = pytest.mark.gpu


def _apart(n, bits, seed, shift=0):
    """n cells, each in a leaf of its own."""
    side = int(np.ceil(n ** (1 / 3)))
    at = np.random.default_rng(seed).permutation(side ** 3)[:n]
    return ((np.stack(np.unravel_index(at, (side,) * 3), 1) << bits) + shift).astype(np.int32)


def _set(g, c, v, was=None):
    import bonxai_amd as bx
    assert bx.lib().bxg_set_values(g._h, c.ptr, v.ptr, len(c), was.ptr if was is not None else None) == bx.OK


def test_more_inputs_than_the_pool_holds(ctx):
    """A device call of more leaves than are made room for."""
    import bonxai_amd as bx
    n = 6_000_000
    c = _apart(n, 1, 1)
    v = (np.arange(n) % 251 + 1).astype(np.uint8)
    g = bx.VoxelGrid(ctx, 0.1, 4, 1, dtype=np.uint8)
    old = 1000
    g.set_values(c[:old], v[:old] + np.uint8(1))
    before = g.digest()
    dc, dv, dw = ctx.to_device(c), ctx.to_device(v), ctx.array(n, np.uint8)
    _set(g, dc, dv, dw)
    assert g.sync() == bx.ERR_OUT_OF_POOL
    assert not dw.numpy().any()
    g.clear_error()
    assert g.digest() == before
    _set(g, dc, dv, dw)
    assert g.sync() == bx.OK
    assert np.array_equal(dw.numpy(), np.arange(n) < old)
    assert g.active_cells_count() == n
    vals, found = g.lookup(c)
    assert found.all() and np.array_equal(vals, v)
    g.close()


@pytest.mark.parametrize("n,lb", [(100_000, 2), (20_000, 4)])
@pytest.mark.parametrize("second", ["device", "set", "on"])
def test_calls_enqueued_one_after_the_other(ctx, second, n, lb):
    """The second call starts before the host has learnt how many leaves the
    first one created."""
    import bonxai_amd as bx
    import oracle
    rng = np.random.default_rng(3)
    busy = bx.VoxelGrid(ctx, 0.1, dtype=np.float32)
    q = rng.integers(-200, 200, (4_000_000, 3)).astype(np.int32)
    busy.set_values(q[:100_000], np.ones(100_000, np.float32))
    dq, out = ctx.to_device(q), ctx.array(len(q), np.float32)
    g, og = bx.VoxelGrid(ctx, 0.1, 2, lb, dtype=np.int32), oracle.Grid(0.1, 2, lb, dtype=np.int32)
    a = _apart(n, lb, 4)
    b = np.concatenate([_apart(n, lb, 5, 1 << 11), a[::7], _apart(n, lb, 5, 1 << 11)[::3]])  # new, set before, twice
    va, vb = np.arange(1, n + 1, dtype=np.int32), -np.arange(1, len(b) + 1, dtype=np.int32)
    da, dva, db, dvb = (ctx.to_device(x) for x in (a, va, b, vb))
    was = ctx.array(len(b), np.uint8)
    ctx.sync()
    for _ in range(40):  # about 3 ms of work before them
        busy.lookup(dq, out)
    _set(g, da, dva)
    og.set_values(a, va)
    if second == "device":
        _set(g, db, dvb, was)
        rc = g.sync()
        if rc != bx.OK:
            assert rc == bx.ERR_OUT_OF_POOL
            assert not was.numpy().any()
            g.clear_error()
            assert_same_cells(g.export(), og.export(), "after the failed call")
            _set(g, db, dvb, was)
            assert g.sync() == bx.OK
        got, want = was.numpy(), og.set_values(b, vb)
    elif second == "set":
        got, want = g.set_values(b, vb, True), og.set_values(b, vb)
    else:
        got, want = g.set_cells_on(b, vb, True), og.set_cells_on(b, vb)
    assert np.array_equal(got, want)
    assert_same_cells(g.export(), og.export(), second)
    for m in (g, og, busy):
        m.close()


@pytest.mark.parametrize("n", [1000, 300_000])
def test_calls_on_a_map_with_an_error(ctx, n):
    """Device calls enqueued behind one that failed (a coordinate out of range)
    set no cell, and every prior state reads 0."""
    import bonxai_amd as bx
    L = bx.lib()
    c = _apart(n, 3, 6)
    v = np.arange(1, n + 1, dtype=np.float32)
    g = bx.VoxelGrid(ctx, 0.1)
    g.set_values(c[: n // 2], v[: n // 2])
    before = g.digest()
    bad = c.copy()
    bad[n // 3] = 1 << 30
    dc, dv, dbad = ctx.to_device(c), ctx.to_device(v), ctx.to_device(bad)
    was = [ctx.to_device(np.ones(n, np.uint8)) for _ in range(4)]
    rc = [L.bxg_set_values(g._h, dbad.ptr, dv.ptr, n, was[0].ptr), L.bxg_set_values(g._h, dc.ptr, dv.ptr, n, was[1].ptr),
          L.bxg_set_cells_on(g._h, dc.ptr, dv.ptr, n, was[2].ptr), L.bxg_set_cells_off(g._h, dc.ptr, n, was[3].ptr)]
    assert rc == [bx.OK] * 4
    assert g.sync() == bx.ERR_COORD_RANGE
    for w in was:
        assert not w.numpy().any()
    g.clear_error()
    assert g.digest() == before
    g.close()
