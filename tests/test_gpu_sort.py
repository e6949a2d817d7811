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


# More long cells than blocks for them, so blocks sort cells of different
# classes (tile by tile, between LDS and the references, within LDS) one after
# another in the same LDS; wave classes and small cells with fewer and with
# more cells than waves.
@pytest.mark.parametrize("short", [100, 3000])
def test_more_cells_than_blocks(gpu_ctx, short):
    r = np.random.default_rng(short)
    sizes = np.concatenate([[4200, 5000, 8192, 8193, 9000, 16_384, 17_000, 40_000],
                            r.integers(1025, 1500, 300), r.integers(257, 1024, 60),
                            r.integers(65, 256, 100), r.integers(17, 64, short),
                            r.integers(2, 16, 300)])
    cells = r.permutation(4096)[:len(sizes)]
    at = np.stack([cells % 16, cells // 16 % 16, cells // 256], 1).repeat(sizes, 0)
    c = (at[:, None] + 0.5 + 0.1 * (r.random((len(at), 3, 3)) - 0.5)) / 16.0
    # the corners of the box that the sixteenths divide
    c = np.concatenate([c, np.zeros((1, 3, 3)), np.ones((1, 3, 3))])
    v = c.astype(np.float32).reshape(-1, 9)
    sc, fr, offs, refs = check_grid(gpu_ctx, v, np.zeros_like(v), 4090.0 / len(v))
    assert list(fr["n"]) == [16, 16, 16]
    n = np.diff(offs)
    blocks = min(max((len(refs) * 9 // 8 + 1024) // 2048, 32), 512)   # of the launch
    waves = ((n > 16) & (n <= 1024)).sum()
    light = min((waves + ((n > 1) & (n <= 16)).sum() // 512) // 16 + 1, blocks // 2)
    assert (n > 1024).sum() > blocks - light
    assert (((n > 16) & (n <= 64)).sum() > 16 * light) == (short == 3000)
    for _ in range(2):
        sc.rebuild_grid_async(4090.0 / len(v))
        _, offs2, refs2 = sc.download_grid()
        assert np.array_equal(offs2, offs) and np.array_equal(refs2, refs)
    sc.close()
