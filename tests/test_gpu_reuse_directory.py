"""GPU test of clear(CLEAR_MEMORY) over root directories of several sizes: a
cleared map is empty, and holds what is put into it next and nothing else."""
import numpy as np
import pytest

from conftest import assert_same_cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inner_bits,roots", [(1, 0), (2, 600), (2, 5000), (3, 70_000), (1, 1_000_000)])
def test_cleared_directory_is_empty(ctx, inner_bits, roots):
    import bonxai_amd as bx
    rng = np.random.default_rng(roots)
    n = 40_000
    far = rng.integers(-60_000, 60_000, (n, 3)).astype(np.int32)  # each in a root of its own
    far = far[np.unique(far >> (inner_bits + 1), axis=0, return_index=True)[1]]
    some = np.ascontiguousarray(far[::5])
    g = bx.VoxelGrid(ctx, 0.1, inner_bits, 1, dtype=np.int32)
    g.reserve(1000, roots)
    for _ in range(3):
        g.set_values(far, np.arange(1, len(far) + 1, dtype=np.int32))
        assert g.active_cells_count() == len(far) and g.stats()["root_count"] == len(far)
        g.clear()
        assert g.active_cells_count() == 0 and g.stats()["root_count"] == 0
        assert not g.lookup(far)[1].any()
        order = np.lexsort((some[:, 2], some[:, 1], some[:, 0]))
        v = np.arange(1, len(some) + 1, dtype=np.int32)
        g.set_values(some, v)
        assert_same_cells(g.export(), (some[order], v[order]), "after clear")
        g.clear()
    g.close()
