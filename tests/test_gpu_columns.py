"""The clustered cull's column path on the GPU at the edges of its ranges,
against the oracle's brute force: lists, counts, offsets and flags bit-exact.

The sizes sit on both sides of what the path's launches depend on: 512 lights
(every block bounds them itself), 16384 (lights scanned at a time), 512
candidates of a column (listed at a time), 16 columns per partial sum, 128
columns a side and 2048 columns (larger grids take the mark path), one to 64
slices, whole columns or a few slices per block.
"""
import numpy as np
import pytest

import oracle_lib as O
from helio_amd import abi, synth
from helio_amd.device import LightCullPass, upload_scene

pytestmark = pytest.mark.gpu


def make(n, width, height, seed=3, crowd=False):
    """n lights around the camera: points, spots, suns, lights that hold the camera, lights behind it and
    out of reach; crowd: all of them in front of the centre of the screen."""
    sc = synth.make_scene("c2_1080p_1k", width=width, height=height, num_lights=n, seed=synth.SEED_BASE + seed)
    rng = np.random.default_rng(seed)
    li = sc.lights
    if n and not crowd:
        eye = np.array(sc.camera.position_near[:3])
        li["light_type"][rng.random(n) < 0.01] = abi.HL_LIGHT_DIRECTIONAL
        near = rng.random(n) < 0.05
        li["position_range"][near, :3] = eye + rng.normal(0, 3.0, (int(near.sum()), 3))
        big = rng.random(n) < 0.02
        li["position_range"][big, 3] = 60.0
    elif n:
        li["position_range"][:, :3] = np.array((0.0, 2.0, 0.0)) + rng.normal(0, 0.5, (n, 3))
    return sc


CASES = [  # lights, screen, grid, cap, pool, crowd
    (0, (320, 180), (16, 9, 24), 0, 1 << 16, False),
    (1, (320, 180), (16, 9, 24), 0, 1 << 16, False),
    (65, (64, 64), (1, 1, 1), 0, 1 << 16, False),
    (511, (333, 177), (5, 3, 64), 0, 1 << 20, False),
    (512, (333, 177), (16, 9, 24), 0, 1 << 20, False),
    (513, (333, 177), (16, 9, 24), 0, 1 << 20, False),
    (300, (640, 360), (40, 23, 10), 0, 1 << 20, False),   # more than 8192 cells
    (700, (333, 177), (4, 4, 24), 0, 1 << 20, True),      # batches of one column
    (1025, (333, 177), (4, 4, 3), 0, 1 << 20, True),
    (900, (640, 360), (17, 1, 48), 0, 1 << 20, False),    # one column past a partial sum
    (600, (1280, 720), (128, 16, 4), 0, 1 << 21, False),  # 2048 columns
    (600, (1290, 720), (129, 8, 4), 0, 1 << 21, False),   # a side of 129: the mark path
    (16385, (256, 144), (8, 5, 6), 0, 1 << 22, False),    # two rounds of lights
    (400, (333, 177), (16, 9, 24), 7, 1 << 20, False),
    (700, (333, 177), (16, 9, 24), 7, 3000, False),
    (700, (333, 177), (4, 4, 24), 0, 5000, True),
    (400, (333, 177), (16, 9, 24), 0, 900, False),
]


@pytest.mark.parametrize("n,size,grid,cap,pool_cap,crowd", CASES)
def test_columns_bit_exact(ctx, hlib, n, size, grid, cap, pool_cap, crowd):
    print(f"[columns] lights={n} size={size} grid={grid} cap={cap} pool={pool_cap}", flush=True)
    sc = make(n, *size, crowd=crowd)
    params = synth.cluster_params(hlib, sc, grid=grid, cap=cap)
    ds = upload_scene(ctx, sc)
    cull = LightCullPass(ctx, sc.width, sc.height, clusters=params, pool_cap=pool_cap)
    cull.prepare(ds)
    for _ in range(2):  # the second call meets the first one's scratch
        cull.cgrid.pool.fill_u32(0xFFFFFFFF)
        cull.execute(ds)
    off, cnt, pool = cull.cgrid.download()
    ooff, ocnt, opool, oflags = O.cull_clusters(sc, params, pool_cap)
    assert cull.overflow() == oflags
    assert np.array_equal(cnt, ocnt) and np.array_equal(off, ooff)
    used = min(int(ooff[-1]) + int(ocnt[-1]), pool_cap)
    assert np.array_equal(pool[:used], opool[:used])
    assert np.all(pool[used:] == 0xFFFFFFFF)  # nothing past the lists
