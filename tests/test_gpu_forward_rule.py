"""Forward shading on both sides of the rule for shared wave tiles (at least 16
lights; on clusters a light per 1024 pixels up to 2^18, per 448 up to 983040;
on tile lists a light per 512 up to 2^17), against the oracle within the
radiance bar, and batched plans without a shared view (whose launch has no
class sums), with only shared ones and with both, against the single views bit
for bit.
"""
import numpy as np
import pytest

from helio_amd.batch import BatchPlan, BatchView
from helio_amd.device import upload_scene
from test_gpu_batch import single_view
from test_gpu_columns import make
from test_gpu_forward_split import test_shade_parity as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,size,clustered", [
    (15, (61, 43), True), (16, (128, 128), True), (15, (128, 128), False), (32, (128, 128), False),
    (256, (512, 512), True), (256, (513, 512), True), (256, (512, 256), False), (255, (512, 256), False),
    (2195, (1024, 960), True), (2194, (1024, 960), True), (2300, (1025, 960), True),
])
def test_parity(ctx, hlib, n, size, clustered):
    check(ctx, hlib, n, size, clustered)


@pytest.mark.parametrize("sizes", [
    [(3, (64, 64)), (100, (512, 512)), (15, (128, 128))], [(100, (512, 512))],
    [(16, (128, 128)), (256, (512, 512))], [(256, (512, 512)), (255, (512, 512)), (0, (64, 64))],
])
def test_batch_equals_single(ctx, hlib, sizes):
    print(f"[forward rule] batch {sizes}", flush=True)
    scenes = [make(n, *size, seed=k) for k, (n, size) in enumerate(sizes)]
    pool = np.concatenate([sc.lights for sc in scenes])
    firsts = np.cumsum([0] + [len(sc.lights) for sc in scenes])
    views = []
    for sc, first in zip(scenes, firsts):
        ids = np.arange(first, first + len(sc.lights), dtype=np.uint32)
        views.append(BatchView(scene=upload_scene(ctx, sc), subset=ctx.upload(ids) if len(ids) else ctx.alloc(16),
                               num_lights=len(ids), out=ctx.alloc(sc.width * sc.height * 16)))
    pool_d = ctx.upload(pool)  # the plan reads it at every launch
    plan = BatchPlan(ctx, pool_d, len(pool), views)
    try:
        refs = [single_view(ctx, hlib, v, plan.config(i))["out"] for i, v in enumerate(views)]
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
