"""Small problems on grids past 2048 columns or 128 a side: the brute-force
launches (few slices) and the column path with candidate boxes in coarser
columns, against the oracle's brute force: lists, counts, offsets and flags
bit-exact.  Light counts on both sides of what a block holds at a time (256),
a last block of fewer than four cells, sides at both ends of a box shift, the
per-cluster cap and a pool that ends early.
"""
import pytest

from test_gpu_columns import test_columns_bit_exact as check

pytestmark = pytest.mark.gpu

CASES = [  # lights, screen, grid, cap, pool, crowd
    (0, (1280, 720), (256, 144, 1), 0, 1 << 16, False),
    (1, (1280, 720), (256, 144, 1), 0, 1 << 18, False),
    (100, (1280, 720), (256, 144, 1), 0, 1 << 22, False),
    (256, (1290, 730), (79, 43, 3), 0, 1 << 22, False),
    (257, (1290, 730), (79, 43, 3), 5, 1 << 22, False),
    (400, (1290, 730), (79, 43, 2), 0, 9000, True),
    (200, (1280, 720), (64, 36, 8), 0, 1 << 22, False),
    (200, (1280, 720), (64, 36, 8), 3, 20000, True),
    (90, (1030, 260), (129, 33, 4), 0, 1 << 21, False),
    (90, (1030, 260), (256, 32, 4), 0, 1 << 21, False),
    (60, (1030, 260), (257, 33, 5), 0, 1 << 21, False),
    (20, (1200, 390), (400, 130, 4), 0, 1 << 22, False),
    (3, (2000, 40), (2000, 10, 24), 0, 1 << 21, False),
    (700, (1290, 720), (129, 1, 33), 0, 1 << 22, True),
    (5000, (400, 36), (200, 1, 4), 0, 1 << 22, False),
    (600, (400, 36), (200, 2, 8), 0, 1 << 22, False),
]


@pytest.mark.parametrize("n,size,grid,cap,pool_cap,crowd", CASES)
def test_lists_bit_exact(ctx, hlib, n, size, grid, cap, pool_cap, crowd):
    assert (grid[0] > 128 or grid[0] * grid[1] > 2048) and grid[0] * grid[1] * grid[2] * n <= 1 << 22
    check(ctx, hlib, n, size, grid, cap, pool_cap, crowd)
