"""GPU tests of the per-cell reference sort at the edges of its size classes.
Bar: offsets and references equal to the oracle's grid."""
import numpy as np
import pytest

from test_gpu_parity import check_grid
from test_gpu_window import _soup

pytestmark = pytest.mark.gpu


# One cell that lists every triangle: a thread's registers (to 16), a wave's
# (to 1024), a block's runs merged within LDS (to 8192), between LDS and the
# references themselves (to 16384), and tile by tile.
@pytest.mark.parametrize("n", [2, 16, 17, 64, 65, 256, 257, 1024, 1025, 4096, 4097, 8192, 8193,
                               10_000, 16_384, 16_385, 40_000])
def test_one_cell(gpu_ctx, n):
    v = _soup(n, n)
    sc, fr, offs, refs = check_grid(gpu_ctx, v, np.zeros_like(v), 1e-6)
    assert len(offs) == 2 and len(refs) == n
    sc.close()


# All classes in one grid, long cells and short ones in the same launch, also
# after a rebuild into the same lists.
def test_all_classes_in_one_grid(gpu_ctx):
    parts = [_soup(20_000, 1, 0.02)]
    for k, n in enumerate((60, 200, 900, 3000, 6000, 9000, 40_000)):
        parts.append(_soup(n, 10 + k, 0.3) * np.float32(1e-3) +
                     np.float32(0.06 + 0.12 * k))
    v = np.concatenate(parts)
    sc, fr, offs, refs = check_grid(gpu_ctx, v, np.zeros_like(v), 4.0)
    n = np.diff(offs)
    for lo, hi in ((2, 16), (17, 64), (65, 256), (257, 1024), (1025, 4096), (4097, 8192),
                   (8193, 16_384), (16_385, 1 << 20)):
        assert ((n >= lo) & (n <= hi)).any(), (lo, hi)
    for _ in range(2):
        sc.rebuild_grid_async(4.0)
        _, offs2, refs2 = sc.download_grid()
        assert np.array_equal(offs2, offs) and np.array_equal(refs2, refs)
    sc.close()
