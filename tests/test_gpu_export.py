"""GPU parity of the whole-map compaction (forEachCell as lists) at the sizes
where its tiles change: mask words per leaf of every leaf size, the last
wavefront and workgroup partly filled, cell types copied by word or by byte,
a capacity below the count, an unaligned value buffer, the filters."""
import ctypes

import numpy as np
import pytest

from conftest import assert_same_cells, sorted_cells

pytestmark = pytest.mark.gpu


def _leaves(n, lb, seed):
    """Coordinates of a few cells in each of n leaves, corner cells among them."""
    rng = np.random.default_rng(seed)
    side = 1 << lb
    org = np.stack(np.unravel_index(np.arange(n), (9, 9, -(-n // 81))), 1) - 4  # any n leaves
    cells = rng.integers(0, side, (n, 6, 3))
    cells[:, 0], cells[:, 1] = 0, side - 1
    return (org[:, None, :] * side + cells).reshape(-1, 3).astype(np.int32)


@pytest.mark.parametrize("lb,n", [(1, 1), (1, 255), (1, 513), (2, 256), (2, 257), (3, 1), (3, 2), (3, 31), (3, 32),
                                  (3, 33), (3, 700), (3, 8193), (4, 3), (4, 5), (4, 90)])
@pytest.mark.parametrize("dtype", [np.float32, np.int64, np.uint8, None])
def test_shapes_and_types(ctx, lb, n, dtype):
    import bonxai_amd as bx
    import oracle
    if lb == 1 and dtype == np.uint8:
        dtype = np.uint32
    c = _leaves(n, lb, n)
    v = None if dtype is None else np.arange(1, len(c) + 1).astype(dtype)
    g, og = bx.VoxelGrid(ctx, 0.1, 2, lb, dtype=dtype), oracle.Grid(0.1, 2, lb, dtype=dtype)
    g.set_values(c, v)
    og.set_values(c, v)
    if dtype is None:
        assert np.array_equal(sorted_cells(g.export()[0])[0], og.export()[0])
    else:
        assert_same_cells(g.export(), og.export(), f"{n} leaves of {1 << lb}")
    g.close()
    og.close()


def _device_export(ctx, m, flt, cap, n, shift=0):
    """bxg_export into device buffers, the values `shift` bytes off: rc, the
    count, and the first min(cap, n) cells."""
    import bonxai_amd as bx
    xyz, buf = ctx.array((max(n, 1), 3), np.int32), ctx.array(4 * n + 8, np.uint8)
    xyz.upload(np.full((max(n, 1), 3), -7, np.int32))
    buf.upload(np.full(4 * n + 8, 0xA5, np.uint8))
    cnt = ctypes.c_uint64()
    rc = bx.lib().bxg_export(m._h, flt, xyz.ptr, buf.ptr + shift, cap, ctypes.byref(cnt))
    k = min(cap, cnt.value)
    out, raw = xyz.numpy(), buf.numpy()
    assert np.all(out[k:n] == -7) and np.all(raw[:shift] == 0xA5) and np.all(raw[shift + 4 * k:] == 0xA5)
    words = raw[shift:shift + 4 * k].copy().view(np.uint32)
    xyz.free()
    buf.free()
    return rc, cnt.value, out[:k], words


@pytest.mark.parametrize("flt", [0, 1, 2])
def test_filters_capacity_and_alignment(ctx, flt):
    import bonxai_amd as bx
    import oracle
    from bonxai_amd import scenes
    pts, o = scenes.box_scan(seed=4, n=5_000)
    m, om = bx.ProbabilisticMap(ctx, 0.1), oracle.ProbMap(0.1)
    m.insert_point_cloud(pts, o, 3.0)
    om.insert_point_cloud(pts, o, 3.0)
    ref_c, ref_w = om.cells()
    p = ref_w.view(np.int32) >> 4
    keep = np.ones(len(p), bool) if flt == 0 else (p > 0 if flt == 1 else p < 0)
    n = int(keep.sum())
    assert n > 100
    for cap, shift in ((n, 0), (n, 1), (n, 2), (n - 1, 0), (65, 3), (0, 0)):
        rc, count, xyz, words = _device_export(ctx, m, flt, cap, n, shift)
        assert rc == (bx.OK if cap >= n else bx.ERR_CAPACITY) and count == n
        got = {tuple(c): w for c, w in zip(xyz.tolist(), words.tolist())}
        want = {tuple(c): w for c, w in zip(ref_c[keep].tolist(), ref_w[keep].tolist())}
        assert len(got) == len(xyz) and got.items() <= want.items(), (flt, cap, shift)
    m.close()
    om.close()
