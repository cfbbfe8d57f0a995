"""GPU test of engine reads behind work that was enqueued on the map before the
engine was made and leaves no event of its own: setCellOff and clear."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", ["off", "clear"])
def test_reads_see_earlier_calls(ctx, what):
    import bonxai_amd as bx
    from bonxai_amd import scenes
    pts, origin = scenes.box_scan(seed=1, n=50_000)
    m = bx.ProbabilisticMap(ctx, 0.05)
    m.insert_point_cloud(pts, origin, 10.0)
    cells = m.export()[0]
    q = np.random.default_rng(1).integers(-200, 200, (4_000_000, 3)).astype(np.int32)
    dq, out = ctx.to_device(q), ctx.array(len(q), np.uint32)
    dc, found = ctx.to_device(np.ascontiguousarray(cells)), ctx.array(len(cells), np.uint8)
    oc = ctx.array((len(cells), 3), np.int32)
    ctx.sync()
    for _ in range(40):  # about 3 ms of work before it
        m.lookup(dq, out)
    if what == "off":
        assert bx.lib().bxg_set_cells_off(m._h, dc.ptr, len(cells), None) == bx.OK
    else:
        m.clear()
    srv = bx.Server(ctx)
    srv.wait(srv.lookup(m, dc, None, found))
    info = srv.wait(srv.export(m, oc))
    srv.close()
    assert not found.numpy().any()
    assert info["count"] == 0
    m.close()
