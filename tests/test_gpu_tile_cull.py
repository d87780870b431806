"""The tile cull's super-tile path on the GPU at the edges of its ranges,
against the oracle's brute force: lists and counts bit-exact.

The sizes sit on both sides of what its launches depend on: 512 lights (every
block bounds them itself; candidates tested at a time), 16384 (lights scanned
at a time), ragged super-tiles of 1 to 64 tiles, tiles that fill up (64
lights) early, late or never, and a screen wide enough that the candidate
boxes are coarser than the super-tiles.
"""
import numpy as np
import pytest

import oracle_lib as O
from helio_amd import abi, synth
from helio_amd.device import LightCullPass, upload_scene
from test_gpu_columns import make
from test_gpu_parity import check_tile_lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,size,crowd", [
    (1, (16, 16), False), (63, (333, 177), False), (512, (333, 177), True), (513, (333, 177), True),
    (1025, (640, 360), True), (700, (1290, 730), False), (900, (3850, 2170), False), (16385, (320, 200), False),
    (300, (2064, 2208), False), (80, (16500, 17), False), (600, (17, 4200), False),
])
def test_tiles_bit_exact(ctx, n, size, crowd):
    print(f"[tiles] lights={n} size={size} crowd={crowd}", flush=True)
    sc = make(n, *size, crowd=crowd)
    ds = upload_scene(ctx, sc)
    cull = LightCullPass(ctx, sc.width, sc.height)
    cull.prepare(ds)
    for _ in range(2):  # the second call meets the first one's scratch
        cull.tiles.lists.fill_u32(0xFFFFFFFF)
        cull.execute(ds)
    lists = cull.tiles.lists.download(np.uint32).reshape(-1, 64)
    counts = cull.tiles.counts.download(np.uint32)
    ol, oc = O.cull_tiles(sc)
    check_tile_lists(lists, counts, ol, oc)
    assert all(np.all(lists[t, c:] == 0xFFFFFFFF) for t, c in enumerate(counts))  # nothing past the lists
