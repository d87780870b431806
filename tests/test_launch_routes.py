"""Which launches the host code takes for a call (CPU only, hip_routes)."""
import pytest

from hip_routes import routes

SHARED = 16  # kModeShared: four waves to a wave tile


def test_forward_shares_wave_tiles_only_where_that_is_faster():
    """Sharing repeats a tile's set-up and walk four times: sizes and light counts on both sides of where the
    two forms took the same time, on clusters and on tile lists (which end at 64 lights)."""
    cases = [  # width, height, lights, shared on clusters, on tiles
        (64, 64, 4, False, False), (32, 32, 15, False, False), (64, 64, 16, True, True),
        (128, 128, 31, True, False), (128, 128, 64, True, True), (256, 256, 16, False, False),
        (256, 256, 64, True, False), (256, 256, 128, True, True), (333, 177, 16, False, False),
        (352, 352, 512, True, True), (512, 512, 128, False, False), (512, 512, 256, True, False),
        (720, 720, 1024, False, False), (720, 720, 4096, True, False), (1300, 731, 2048, False, False),
        (1300, 731, 2554, True, False), (1024, 1024, 749, False, False), (1024, 1024, 16384, False, False),
    ]
    got = routes(f"""
for w, h, n, _, _ in {cases!r}:
    row = []
    for grid in ((4, 4, 24), None):
        ds, cull = cull_pass(scene(n, w, h), grid)
        sh = DeferredLightPass(ctx, w, h)
        sh.prepare(ds)
        mode = [v[3] for k, v, _ in calls(lambda: sh.execute(ds, cull.publish())) if k == "k_shade"]
        row.append(mode == [{SHARED}])
    result.append(row)
""")
    for c, g in zip(cases, got):
        assert g == list(c[3:]), c


def test_batched_launch_has_class_sums_only_for_a_view_that_needs_them():
    """The class sums of shared wave tiles cost LDS, a test and a ballot per light class: plans without a shared
    view do not pay for them; a plan with one still has one forward launch."""
    own, shared = (1, 2, 0), (1, 2, SHARED)
    plans = [([(512, 288, 64)], [own]), ([(640, 360, 100)] * 3, [own]), ([(128, 128, 256)] * 2, [shared]),
             ([(512, 288, 64), (128, 128, 256), (128, 128, 256)], [shared])]
    got = routes(f"""
for views, _ in {plans!r}:
    made = []
    for w, h, n in views:
        sc = scene(n, w, h)
        made.append(BatchView(scene=upload_scene(ctx, sc), subset=ctx.upload(np.arange(n, dtype=np.uint32)),
                              num_lights=n, out=ctx.alloc(w * h * 16)))
    plan = BatchPlan(ctx, made[-1].scene.lights, views[-1][2], made)
    result.append([v for k, v, _ in calls(plan.launch) if k == "k_shade_batch"])
""")
    for (views, want), g in zip(plans, got):
        assert [tuple(v) for v in g] == want, views


def test_cluster_paths():
    """Small problems (cells x lights up to 2^22) on grids past 2048 columns or 128 a side: two brute-force
    launches where the grid has few slices, else the column path; larger ones take the mark path."""
    col2, col3 = ["k_col_count", "k_col_fill"], ["k_col_prep", "k_col_count", "k_col_fill"]
    brute, mark = ["k_cluster_bf_count", "k_cluster_bf_fill"], ["k_cluster_geom", "k_cluster_mark"]
    cases = [((16, 9, 24), 200, col2), ((16, 9, 24), 2000, col3), ((128, 16, 4), 600, col3),
             ((256, 144, 1), 100, brute), ((80, 45, 1), 1000, brute), ((80, 45, 3), 300, brute),
             ((80, 45, 1), 1200, mark), ((64, 36, 8), 200, col3), ((129, 8, 4), 600, col3),
             ((255, 255, 2), 8, col3), ((200, 1, 1), 5000, col3), ((200, 1, 1), 300, col2),
             ((64, 36, 24), 900, mark), ((80, 45, 24), 500, mark)]
    got = routes(f"""
for grid, n, _ in {cases!r}:
    ds, cull = cull_pass(scene(n, 640, 360), grid)
    result.append([k for k, _, _ in calls(lambda: cull.execute(ds))])
""")
    for (grid, n, want), g in zip(cases, got):
        assert g[:len(want)] == want and (want == mark or len(g) == len(want)), (grid, n, g)


def test_a_cull_without_memory_for_the_column_scratch_takes_the_mark_path():
    """The column path reserves 12 bytes per (block, light), 398 MB for 45x45x24 cells and 16384 lights, the mark
    path's bitmask takes 100: where the first allocation fails the call goes on with the second, and takes the
    column path again when there is memory."""
    single, plan = routes("""
ds, cull = cull_pass(scene(16384, 640, 360), (45, 45, 24))
row = []
for limit in (200 << 20, NO_LIMIT):
    row.append([k for k, _, _ in calls(lambda: cull.execute(ds), limit)])
row.append(ctx.lib.raw["hl_last_error"](ctx.h).decode())
result.append(row)
sc = scene(16384, 640, 360)
dv = upload_scene(ctx, sc)
params = synth.cluster_params(ctx.lib, sc, grid=(45, 45, 24))
view = BatchView(scene=dv, subset=ctx.upload(np.arange(16384, dtype=np.uint32)), num_lights=16384,
                 out=ctx.alloc(640 * 360 * 16), clusters=params)
row = []
for limit in (200 << 20, NO_LIMIT):
    stub.stub_reset(limit)
    p = BatchPlan(ctx, dv.lights, 16384, [view])
    row.append([k for k, _, _ in calls(p.launch)])
    p.destroy()
result.append(row)
""")
    assert single[0][:2] == ["k_cluster_geom", "k_cluster_mark"]
    assert single[1] == ["k_col_prep", "k_col_count", "k_col_fill"]
    assert single[2] == ""
    assert plan[0][:2] == ["k_batch_geom", "k_batch_mark"]
    assert plan[1][:3] == ["k_batch_col_prep", "k_batch_col_count", "k_batch_col_fill"]


def test_backward_shares_heavy_tiles_on_large_views():
    """One wave to a wave tile on large views with few lights only: its chain over a long list is what bounds
    the call (1280x720 with 8192 lights 1975 us, 1612 with four waves)."""
    cases = [  # width, height, lights, items per block tile
        (512, 512, 64, 2), (512, 512, 1024, 4), (1280, 720, 64, 1), (1280, 720, 1100, 1), (1280, 720, 1300, 2),
        (1600, 900, 1024, 1), (1600, 900, 4096, 2), (1920, 1080, 4096, 1),
    ]
    got = routes(f"""
from helio_amd.device import AdjointBuffers
for w, h, n, _ in {cases!r}:
    sc = synth.make_scene("c4_512_adj", width=w, height=h, num_lights=n)
    ds = upload_scene(ctx, sc)
    cull = LightCullPass(ctx, w, h)
    sh = DeferredLightPass(ctx, w, h)
    sh.prepare(ds)
    gr = AdjointBuffers(ctx, w, h, n)
    d_out = ctx.alloc(16 * w * h)
    items = [b for k, v, b in calls(lambda: sh.backward(ds, cull.publish(), d_out, gr)) if k == "k_shade"]
    result.append([b / (-(-w // 32) * -(-h // 8)) for b in items])
""")
    for c, g in zip(cases, got):
        assert g == [c[3]], c


def test_batched_column_blocks():
    """More column blocks than the chip holds at 512 threads are launched at 256; a view of few columns and many
    lights has a block per 512 lights while every view can."""
    few, many, deep, deeps = routes("""
def view(n, w, h, grid):
    sc = scene(n, w, h)
    ds = upload_scene(ctx, sc)
    return BatchView(scene=ds, subset=ctx.upload(np.arange(n, dtype=np.uint32)), num_lights=n,
                     out=ctx.alloc(w * h * 16), clusters=synth.cluster_params(ctx.lib, sc, grid=grid))

for views in ([(64, 640, 360, (10, 6, 24))] * 2, [(64, 640, 360, (10, 6, 24))] * 18,
              [(16384, 640, 360, (30, 17, 24)), (16384, 64, 64, (1, 1, 24))],
              [(16384, 640, 360, (30, 17, 24))] + [(16384, 64, 64, (1, 1, 24))] * 63):
    made = {v: view(*v) for v in views}
    pool = max(made.values(), key=lambda v: v.num_lights)
    plan = BatchPlan(ctx, pool.scene.lights, pool.num_lights, [made[v] for v in views])
    result.append([(v, b) for k, v, b in calls(plan.launch) if k == "k_batch_col_count"])
    plan.destroy()
""")
    assert [v for v, _ in few] == [[512]] and [v for v, _ in many] == [[256]]
    assert many[0][1] == 18 * 60
    assert deep[0][1] == 2 * 510 + 24  # 511 aimed at and 32, a block per slice
    assert deeps[0][1] == 510 + 63 * 8
