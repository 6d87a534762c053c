"""The batched form: many independent jobs in one launch sequence.  Every job's image must be
identical to what the plain per-job renderer draws, for every tuning (tile shape, persistent
tile queue, graph replay), and match the CPU oracle to the parity bar."""
import numpy as np
import pytest

try:
    import torch  # noqa: F401
except ImportError:  # pragma: no cover
    torch = None

from dfpsr_amd import scenes as S
from oracle import harness as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    import torch
    assert torch.cuda.is_available()
    from dfpsr_amd import api
    jobs = S.batch_jobs(48, seed=5, max_tris=6000)
    g = api.GpuJobs(jobs)
    r = api.renderer_create()
    g.clear()
    g.render_plain(r)
    torch.cuda.synchronize()
    plain = [g.image(i) for i in range(len(jobs))]
    return api, jobs, g, plain


TUNINGS = [(0, 0, False, 0), (1, 0, False, 0), (2, 0, False, 0), (0, 4, False, 0), (2, 2, True, 0), (0, 8, True, 0),
           (0, 0, False, 1), (1, 4, True, 1)]


@pytest.mark.parametrize("tile_config,persistent,graph,path", TUNINGS)
def test_batch_equals_plain_loop(setup, tile_config, persistent, graph, path):
    api, jobs, g, plain = setup
    print(f"[gpu] batch tile_config={tile_config} persistent={persistent} graph={graph} raster_path={path}", flush=True)
    b = api.Batch()
    t = api.tuning(tile_config, persistent, graph, clear=True, raster_path=path)
    for rep in range(2 if graph else 1):  # a replayed graph must give the same images
        g.clear()
        b.render(g.jobs, t)
        for i in range(len(jobs)):
            c, d = g.image(i)
            assert np.array_equal(c, plain[i][0]), f"job {i} colour (rep {rep})"
            assert np.array_equal(d.view(np.uint32), plain[i][1].view(np.uint32)), f"job {i} depth (rep {rep})"
    assert b.stats()[0] > 0


def test_batch_jobs_match_oracle(setup):
    api, jobs, g, plain = setup
    for i in range(0, len(jobs), 6):
        rc, rd = H.oracle_render(jobs[i])
        c, d = plain[i]
        assert np.array_equal(d.view(np.uint32), rd.view(np.uint32)), f"job {i} depth"
        a = c.view(np.uint8).reshape(-1, 4).astype(int)
        b = rc.view(np.uint8).reshape(-1, 4).astype(int)
        bad = np.any(np.abs(a - b) > 1, axis=1)
        assert bad.sum() <= int(0.001 * bad.size), f"job {i}: {bad.sum()} pixels beyond 1 LSB"


def test_renderer_tuning_does_not_change_results(setup):
    api, jobs, g, plain = setup
    sc = S.terrain(width=400, height=300, grid=64, texture_size=256, resolutions=9)
    ref = api.render_scene(sc)
    for cfg in [(1, 0, False), (2, 4, True), (0, 2, True)]:
        r = api.renderer_create()
        api.renderer_setTuning(r, api.tuning(*cfg))
        for _ in range(2):
            got = api.render_scene(sc, r)
            assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1].view(np.uint32), ref[1].view(np.uint32)), cfg


def test_jobs_after_a_refused_call(setup):
    """A call that is refused for its first job leaves nothing behind: the jobs drawn before it are drawn
    again by the next call."""
    api, jobs, g, plain = setup
    b = api.Batch()
    t = api.tuning(clear=True)
    b.render(g.jobs, t)
    refused = (api.Job * 2)(g.jobs[0], g.jobs[1])
    refused[0].color.stride_bytes = 2
    with pytest.raises(api.DfpsrError):
        b.render(refused, t)
    g.clear()
    print("[gpu] batch after a refused call", flush=True)
    b.render(g.jobs, t)
    for i in range(len(jobs)):
        c, d = g.image(i)
        assert np.array_equal(c, plain[i][0]) and np.array_equal(d.view(np.uint32), plain[i][1].view(np.uint32)), f"job {i}"


def test_frames_that_show_nothing_are_cleared(setup):
    """With the fill on, a frame without any visible task still fills its canvases, and a frame after it
    draws as ever: the renderer with and without a task out of view, and a batch."""
    api, jobs, g, plain = setup
    sc = S.cube_soup(width=50, height=34, triangles=40, seed=3)
    scene = api.GpuScene(sc)
    behind = S.identity_transform()
    behind[2] = -50.0
    print("[gpu] frames that show nothing", flush=True)
    r = api.renderer_create()
    api.renderer_setTuning(r, api.tuning(clear=True, clear_color=0x01020304, clear_depth=0.5))
    want = api.render_scene(sc, r)
    for tasks in (0, 1):
        color, depth = np.full((34, 50), 7, np.uint32), np.full((34, 50), 7, np.float32)
        api.renderer_begin(r, api.host_image(color), api.host_image(depth))
        for _ in range(tasks):
            api.renderer_giveTask(r, scene.model, behind, scene.camera)
        api.renderer_end(r)
        assert (color == 0x01020304).all() and (depth == 0.5).all()
        again = api.render_scene(sc, r)
        assert np.array_equal(again[0], want[0]) and np.array_equal(again[1], want[1])
    b = api.Batch()
    two = (api.Job * 2)(g.jobs[0], g.jobs[1])
    for j in two:
        j.transform[:] = [float(v) for v in behind]
    g.colors[0].fill_(7)
    g.depths[1].fill_(7.0)
    b.render(two, api.tuning(clear=True, clear_color=0x01020304, clear_depth=0.5))
    for i in range(2):
        c, d = g.image(i)
        assert (c == 0x01020304).all() and (d == 0.5).all()
    g.clear()
    b.render(g.jobs, api.tuning(clear=True))
    for i in range(len(jobs)):
        c, d = g.image(i)
        assert np.array_equal(c, plain[i][0]) and np.array_equal(d.view(np.uint32), plain[i][1].view(np.uint32)), f"job {i}"


def test_autotune_picks_a_swept_setting_and_keeps_images(setup):
    api, jobs, g, plain = setup
    b = api.Batch()
    g.clear()
    best, ms = b.autotune(g.jobs, 2, api.tuning(clear=True))
    assert ms.shape == (3, 5) and np.all(ms > 0)
    steps = [0, 1, 2, 4, 8]
    assert 0 <= best.tile_config < 3 and best.persistent_per_cu in steps and best.use_graph == 1 and best.clear == 1
    assert ms[best.tile_config, steps.index(best.persistent_per_cu)] == ms.min()
    for i in range(len(jobs)):
        c, d = g.image(i)
        assert np.array_equal(c, plain[i][0]) and np.array_equal(d.view(np.uint32), plain[i][1].view(np.uint32)), i


def test_stage_timing_inside_graph_replay(setup):
    """With timing on, a graph-replayed frame is launched as two graphs with events between them:
    stages before the raster as one figure, then the raster, then the whole."""
    api, jobs, g, plain = setup
    sc = S.terrain(width=320, height=240, grid=48, texture_size=128, resolutions=8)
    ref = api.render_scene(sc)
    r = api.renderer_create()
    api.renderer_setTuning(r, api.tuning(use_graph=True))
    r.set_timing(True)
    for _ in range(3):
        got = api.render_scene(sc, r)
        assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1].view(np.uint32), ref[1].view(np.uint32))
        t = r.timing()
        assert t[0] == 0 and t[1] == 0 and t[2] > 0 and t[3] > 0 and t[4] >= t[3]


def test_config2_full_batch_equals_plain_loop_and_oracle():
    """Config 2 at full size: 4,096 uneven jobs (seed 2, as the benchmark draws them).  The
    batched form with the direct per-tile bins (binning 0) and with the counted, scanned and
    filled lists (binning 1), both graph-replayed over persistent workgroups, gives every job's
    image bit for bit as the per-job loop of the plain renderer does; a seeded sample of jobs
    meets the oracle's bar."""
    import torch
    assert torch.cuda.is_available()
    from dfpsr_amd import api
    jobs = S.batch_jobs(4096, seed=2)
    print(f"[gpu] config 2: {len(jobs)} jobs, {sum(s.indices.shape[0] for s in jobs)} polygons", flush=True)
    g = api.GpuJobs(jobs)
    r = api.renderer_create()
    g.clear()
    g.render_plain(r)
    torch.cuda.synchronize()
    plain_c = [c.clone() for c in g.colors]
    plain_d = [d.clone() for d in g.depths]
    for binning in (0, 1):
        b = api.Batch()
        t = api.tuning(1, 8, True, clear=True, binning=binning)
        for rep in range(2):
            g.clear()
            b.render(g.jobs, t)
            torch.cuda.synchronize()
            bad = [i for i in range(len(jobs)) if not (torch.equal(g.colors[i], plain_c[i]) and torch.equal(g.depths[i], plain_d[i]))]
            assert not bad, f"binning {binning} rep {rep}: jobs {bad[:8]} differ from the per-job loop"
        print(f"[gpu] config 2 binning {binning}: {b.stats()[0]} commands, {b.stats()[1]} tile pairs, identical", flush=True)
    sample = np.random.default_rng(2).choice(len(jobs), 12, replace=False)
    for i in sorted(sample.tolist()):
        rc, rd = H.oracle_render(jobs[i])
        c = plain_c[i].cpu().numpy().view(np.uint32)
        d = plain_d[i].cpu().numpy()
        assert np.array_equal(d.view(np.uint32), rd.view(np.uint32)), f"job {i} depth"
        a = c.view(np.uint8).reshape(-1, 4).astype(int)
        w = rc.view(np.uint8).reshape(-1, 4).astype(int)
        bad = np.any(np.abs(a - w) > 1, axis=1)
        assert bad.sum() <= int(0.001 * bad.size), f"job {i}: {bad.sum()} pixels beyond 1 LSB"
