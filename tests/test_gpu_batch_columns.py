"""Batched culls on both paths in one plan, against the single-view path on
the same grid: the pixels bit for bit (the same lists in the same order).

Views on the column path at the edges of its ranges (no lights, one, 64 and 65
per prepared block, 4096 and 4097 scanned at a time, one column, 2048 columns,
one and 64 slices, a per-cluster cap) beside views whose grids take the mark
path (a side of 129 columns, more than 2048 columns), with light subsets in
pool order, launched eagerly and replayed from the captured graph.
"""
import numpy as np
import pytest

from helio_amd import synth
from helio_amd.batch import BatchPlan, BatchView
from helio_amd.device import upload_scene
from test_gpu_batch import single_view
from test_gpu_columns import make

pytestmark = pytest.mark.gpu

VIEWS = [  # lights, screen, grid, cap
    (0, (64, 64), (1, 1, 1), 0), (1, (64, 64), (1, 1, 64), 0), (64, (129, 65), (3, 2, 24), 0),
    (65, (333, 177), (16, 9, 24), 0), (700, (333, 177), (129, 8, 4), 0), (513, (640, 360), (128, 16, 4), 0),
    (4096, (320, 180), (5, 3, 24), 0), (4097, (320, 180), (4, 4, 24), 0), (900, (640, 360), (64, 36, 24), 0),
    (700, (333, 177), (16, 9, 24), 7), (300, (640, 360), (64, 36, 8), 5),
]


@pytest.mark.parametrize("pick", [None, (3,), (4,), (0, 8)])
def test_mixed_plans_equal_single_view(ctx, hlib, pick):
    print(f"[batch columns] views {pick}", flush=True)
    specs = VIEWS if pick is None else [VIEWS[i] for i in pick]
    scenes = [make(n, *size, seed=20 + k, crowd=k % 3 == 2) for k, (n, size, _, _) in enumerate(specs)]
    pool = np.concatenate([sc.lights for sc in scenes] + [scenes[0].lights[:0]])
    if not len(pool):
        pool = make(1, 64, 64).lights
    first = 0
    views = []
    for sc, (n, _, grid, cap) in zip(scenes, specs):
        ids = np.arange(first, first + n, dtype=np.uint32)
        first += n
        views.append(BatchView(scene=upload_scene(ctx, sc), subset=ctx.upload(ids) if n else ctx.alloc(16),
                               num_lights=n, out=ctx.alloc(sc.width * sc.height * 16),
                               clusters=synth.cluster_params(hlib, sc, grid=grid, cap=cap)))
    pool_d = ctx.upload(pool)  # the plan reads it at every launch
    plan = BatchPlan(ctx, pool_d, len(pool), views)
    try:
        refs = []
        for v, (_, _, _, cap), i in zip(views, specs, range(len(specs))):
            refs.append(single_view(ctx, hlib, v, plan.config(i), cap=cap)["out"])
        for rep in range(3):
            for v in views:
                v.out.fill_u32(0)
            if rep == 1:
                plan.capture()
            plan.launch()
            ctx.synchronize()
            for i, v in enumerate(views):
                host = v.scene.host
                got = v.out.download(np.float32, (host.height, host.width, 4))
                lit = host.depth < 1.0
                assert np.array_equal(got[lit], refs[i][lit]), f"view {i}, launch {rep}"
    finally:
        plan.destroy()
