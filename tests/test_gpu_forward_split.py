"""Forward shading on both sides of the rule by which a view's wave tiles are
shared by the block's four waves (up to 2^16 pixels; up to 2^20 with a light
for every 1400 pixels), against the oracle within the radiance bar (1e-4
relative + 1e-6, the lights' sums being reordered by the rule), on tiles and
on clusters, with skies, ragged sizes and lists shorter than four lights; the
RGBA16F target is the RGBA32F one rounded, a debug view is the decoded texel,
and a batched plan's view is the single view bit for bit.
"""
import numpy as np
import pytest

import oracle_lib as O
from helio_amd import abi, synth
from helio_amd.batch import BatchPlan, BatchView
from helio_amd.device import DeferredLightPass, upload_scene
from test_gpu_batch import single_view
from test_gpu_columns import make
from test_gpu_parity import check_radiance, hip_clusters, hip_tiles

pytestmark = pytest.mark.gpu

SIZES = [  # lights, screen
    (3, (8, 8)), (64, (61, 43)), (5, (256, 256)), (130, (256, 256)), (130, (257, 257)),
    (700, (1400, 700)), (699, (1400, 700)), (749, (1024, 1024)), (2000, (1025, 1024)),
]


@pytest.mark.parametrize("clustered", [False, True])
@pytest.mark.parametrize("n,size", SIZES)
def test_shade_parity(ctx, hlib, n, size, clustered):
    print(f"[forward split] lights={n} size={size} clustered={clustered}", flush=True)
    sc = make(n, *size)
    if clustered:
        params = synth.cluster_params(hlib, sc, grid=(4, 4, 24))
        ds, cull, off, cnt, pool, _ = hip_clusters(ctx, sc, params, 1 << 21)
        grid = O.cluster_grid_host(params, off, cnt, pool)
    else:
        ds, cull, lists, counts = hip_tiles(ctx, sc)
        grid = O.tile_grid_host(sc, np.ascontiguousarray(lists.reshape(-1)), counts)
    ref, pairs = O.shade(sc, grid, flags=abi.HL_SHADE_CLEAR_SKY)
    outs = []
    for fmt, dt in ((abi.HL_FMT_RGBA32_FLOAT, np.float32), (abi.HL_FMT_RGBA16_FLOAT, np.float16)):
        shade = DeferredLightPass(ctx, sc.width, sc.height, out_format=fmt)
        shade.prepare(ds)
        shade.out.fill_u32(0x7FC00000)
        shade.execute(ds, cull.publish(), flags=abi.HL_SHADE_CLEAR_SKY)
        outs.append(shade.out.download(dt, (sc.height, sc.width, 4)))
    check_radiance(outs[0], ref)
    with np.errstate(over="ignore"):
        want = outs[0].astype(np.float16)
    assert np.array_equal(outs[1].view(np.uint16), want.view(np.uint16))
    assert shade.count_pairs(ds, cull.publish()) == pairs


def test_debug_view_of_a_shared_view(ctx):
    sc = make(9, 61, 43)
    print("[forward split] debug view", flush=True)
    ds, cull, lists, counts = hip_tiles(ctx, sc)
    shade = DeferredLightPass(ctx, sc.width, sc.height)
    shade.debug_mode = 1
    shade.prepare(ds)
    shade.out.fill_u32(0)
    shade.execute(ds, cull.publish())
    ref, _ = O.shade(sc, O.tile_grid_host(sc, np.ascontiguousarray(lists.reshape(-1)), counts),
                     globals_=shade.globals)
    lit = sc.depth < 1.0
    assert np.array_equal(shade.output()[lit], ref[lit])


def test_batch_equals_single(ctx, hlib):
    """Views on both sides of the rule in one plan (several views a launch) and in plans of one view."""
    print("[forward split] batch", flush=True)
    sizes = [(3, (64, 64)), (130, (256, 256)), (130, (264, 256)), (700, (1400, 700)), (699, (1400, 700))]
    scenes = [make(n, *size, seed=k) for k, (n, size) in enumerate(sizes)]
    for plan_scenes in (scenes, scenes[1:2]):
        pool = np.concatenate([sc.lights for sc in plan_scenes])
        firsts = np.cumsum([0] + [len(sc.lights) for sc in plan_scenes])
        views = []
        for sc, first in zip(plan_scenes, firsts):
            ids = np.arange(first, first + len(sc.lights), dtype=np.uint32)
            views.append(BatchView(scene=upload_scene(ctx, sc), subset=ctx.upload(ids), num_lights=len(ids),
                                   out=ctx.alloc(sc.width * sc.height * 16)))
        pool_d = ctx.upload(pool)  # the plan reads it at every launch
        plan = BatchPlan(ctx, pool_d, len(pool), views)
        try:
            for v in views:
                v.out.fill_u32(0)
            plan.launch()
            ctx.synchronize()
            for i, v in enumerate(views):
                host = v.scene.host
                got = v.out.download(np.float32, (host.height, host.width, 4))
                ref = single_view(ctx, hlib, v, plan.config(i))["out"]
                lit = host.depth < 1.0
                assert np.array_equal(got[lit], ref[lit]), f"view {i} of {len(views)}"
        finally:
            plan.destroy()
