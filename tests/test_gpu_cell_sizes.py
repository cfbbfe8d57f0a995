"""GPU test of cells of all sizes through setValue, setCellOn, lookup and export,
with the caller's buffers at aligned and at odd addresses: bytes as put in."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 4, 1])
@pytest.mark.parametrize("size", [1, 2, 3, 5, 6, 12, 16, 20, 24, 33, 48, 64, 100, 256])
def test_values_of_a_size(ctx, size, shift):
    import bonxai_amd as bx
    L = bx.lib()
    rng = np.random.default_rng(size)
    n = 3000
    c = np.unique(rng.integers(-40, 40, (2 * n, 3)).astype(np.int32), axis=0)
    c = np.ascontiguousarray(c[rng.permutation(len(c))][:n])
    v = rng.integers(1, 256, (n, size)).astype(np.uint8)
    g = bx.VoxelGrid(ctx, 0.1, dtype=np.dtype(f"V{size}"))

    def device(a):  # at that many bytes past an aligned address
        return ctx.to_device(np.concatenate([np.zeros(shift, np.uint8), a.reshape(-1)]))

    dc, half, there = ctx.to_device(c), n // 2, np.arange(n) < n // 2
    dv, dw, out, found = device(v), device(v[::-1].copy()), device(np.full(v.size, 7, np.uint8)), ctx.array(n, np.uint8)
    assert L.bxg_set_values(g._h, dc.ptr, dv.ptr + shift, half, None) == bx.OK

    def values():
        assert L.bxg_lookup(g._h, dc.ptr, n, out.ptr + shift, found.ptr) == bx.OK
        return out.numpy()[shift:].reshape(n, size), found.numpy().astype(bool)

    got, f = values()
    assert np.array_equal(f, there)
    assert np.array_equal(got, np.where(there[:, None], v, 0))
    assert L.bxg_set_cells_on(g._h, dc.ptr, dw.ptr + shift, n, None) == bx.OK  # the cells that are off only
    want = np.where(there[:, None], v, v[::-1])
    got, f = values()
    assert f.all() and np.array_equal(got, want)
    oc, count = ctx.array((n, 3), np.int32), ctypes.c_uint64()
    assert L.bxg_export(g._h, 0, oc.ptr, out.ptr + shift, n, ctypes.byref(count)) == bx.OK and count.value == n
    e, ev = oc.numpy(), out.numpy()[shift:].reshape(n, size)
    a, b = np.lexsort(e.T), np.lexsort(c.T)
    assert np.array_equal(e[a], c[b]) and np.array_equal(ev[a], want[b])
    assert L.bxg_set_cells_off(g._h, dc.ptr, half, None) == bx.OK
    got, f = values()
    assert np.array_equal(f, ~there) and np.array_equal(got, np.where(there[:, None], 0, want))
    g.close()
