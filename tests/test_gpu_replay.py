"""Captured launch sequences over changing frames.  A captured sequence is replayed while nothing that
picks its kernels changes; the height of a canvas, the projection of a camera and the mix of both on a
canvas pick the raster kernel, also where the number of tiles, triangles and buffers stays the same.
Every frame on an object that replays must be the frame a fresh object draws in submission order."""
import numpy as np
import pytest

try:
    import torch
except ImportError:  # pragma: no cover
    torch = None

from dfpsr_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    assert torch is not None and torch.cuda.is_available()
    from dfpsr_amd import api as A
    A.lib()
    return A


def soup(width, height, orthogonal, seed=3):
    """Triangles in front of and behind distance 1, so that a canvas of depth 1 shows half of them under
    either projection."""
    sc = S.cube_soup(width=width, height=height, triangles=150, seed=seed, spread=0.6, cam_distance=1.0)
    sc.points *= np.float32(0.5)
    sc.perspective = not orthogonal
    return sc


def same(a, b):
    return all(np.array_equal(x.view(np.uint32), y.view(np.uint32)) for x, y in zip(a, b))


# (width, height, projections of the two tasks).  Neighbours differ in the raster they need and in nothing
# that sizes a launch; each is drawn twice, so that every one is captured and replayed.
EVEN, ODD = (96, 64), (96, 63)
FRAMES = [(EVEN, "pp"), (ODD, "pp"), (EVEN, "pp"), (EVEN, "oo"), (EVEN, "pp"), (EVEN, "po"), (EVEN, "oo"), (ODD, "oo"), (ODD, "po"), (ODD, "pp")]


@pytest.mark.parametrize("timing", [False, True])
@pytest.mark.parametrize("clear", [False, True])
@pytest.mark.parametrize("tile_config,persistent", [(0, 0), (1, 0), (2, 2)])
def test_renderer_replays_frames_of_changing_form(api, tile_config, persistent, clear, timing):
    print(f"[gpu] replay renderer tiles {tile_config} persistent {persistent} clear {clear} timing {timing}", flush=True)
    models = [api.GpuScene(soup(*EVEN, False, seed)) for seed in (3, 4)]
    replaying = api.renderer_create()
    replaying.set_timing(timing)
    options = dict(tile_config=tile_config, clear=clear, clear_color=0x01020304, clear_depth=1.0)
    api.renderer_setTuning(replaying, api.tuning(persistent_per_cu=persistent, use_graph=True, **options))

    def draw(renderer, size, projections):
        color, depth = np.full(size[::-1], 9, np.uint32), np.ones(size[::-1], np.float32)
        api.renderer_begin(renderer, api.host_image(color), api.host_image(depth))
        for g, p in zip(models, projections):
            sc = soup(*size, p == "o")
            camera = api.camera_create(sc.perspective, sc.cam_location, *size, sc.width_slope, sc.near_clip, sc.far_clip)
            api.renderer_giveTask(renderer, g.model, S.identity_transform(), camera)
        api.renderer_end(renderer)
        return color, depth

    wanted = {}
    for frame in FRAMES:
        fresh = api.renderer_create()
        api.renderer_setTuning(fresh, api.tuning(raster_path=1, **options))
        wanted[frame] = draw(fresh, *frame)
        assert (wanted[frame][1] != 1.0).mean() > 0.1
    for k, frame in enumerate(FRAMES + FRAMES):
        for repeat in range(2):
            assert same(draw(replaying, *frame), wanted[frame]), f"frame {k} {frame} repeat {repeat}"


def test_renderer_replays_a_canvas_that_grows_past_16_bit_columns(api):
    """32,767 and 32,768 columns have the same tiles; the visibility raster holds only the narrower."""
    options = dict(clear=True, clear_depth=1.0)
    replaying = api.renderer_create()
    api.renderer_setTuning(replaying, api.tuning(use_graph=True, **options))
    print("[gpu] replay wide canvases", flush=True)
    for width in (32767, 32768, 32767, 32768):
        model = api.GpuScene(soup(width, 16, False))
        fresh = api.renderer_create()
        api.renderer_setTuning(fresh, api.tuning(raster_path=1, **options))
        out = []
        for r in (replaying, fresh):
            color, depth = np.zeros((16, width), np.uint32), np.zeros((16, width), np.float32)
            api.renderer_begin(r, api.host_image(color), api.host_image(depth))
            model.give(r)
            api.renderer_end(r)
            out.append((color, depth))
        assert (out[1][1] != 1.0).any() and same(*out), width


def test_batch_replays_jobs_of_changing_form(api):
    batch = api.Batch()
    options = dict(clear=True, clear_depth=1.0)
    print("[gpu] replay batch", flush=True)
    for k, (size, orthogonal) in enumerate([(EVEN, False), (ODD, False), (EVEN, False), (EVEN, True), (ODD, True), (EVEN, False)] * 2):
        jobs = [soup(*EVEN, False, 5), soup(*size, orthogonal, 6), soup(*EVEN, orthogonal, 7)]
        g = api.GpuJobs(jobs)
        batch.render(g.jobs, api.tuning(tile_config=1, persistent_per_cu=4, use_graph=True, **options))
        got = [g.image(i) for i in range(len(jobs))]
        g.clear()
        api.Batch().render(g.jobs, api.tuning(raster_path=1, **options))
        for i in range(len(jobs)):
            assert same(got[i], g.image(i)), f"call {k} job {i}"


@pytest.mark.parametrize("clear", [False, True])
@pytest.mark.parametrize("tile_config", [0, 1])
def test_differentiable_forward_replays_views_of_changing_form(api, tile_config, clear):
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    replaying = api.DiffRenderer()
    print(f"[gpu] replay differentiable views tiles {tile_config} clear {clear}", flush=True)
    for k, (height, orthogonal) in enumerate([(64, False), (63, False), (64, False), (64, True), (63, True), (64, False)] * 2):
        views = S.sphere_views(6, 2, 96, height, seed=8)
        for v in views:  # near enough that the surface reaches every row and lies around distance 0.8
            v.cam_location = S.look_at(np.asarray(v.cam_location[:3], np.float64) * (1.3 / 3.0))
            v.perspective = not orthogonal
        out = []
        for renderer, graph, path in ((replaying, True, 0), (api.DiffRenderer(), False, 1)):
            gv = api.GpuViews(views)
            for d in gv.depth:
                d.fill_(0.8)
            renderer.forward(gv.model, gv.views, tex, None, api.tuning(tile_config=tile_config, clear=clear, clear_depth=0.8, use_graph=graph, raster_path=path))
            torch.cuda.synchronize()
            out.append([x.cpu().numpy() for i in range(len(views)) for x in (gv.color[i], gv.visibility[i], gv.depth[i])])
        assert (out[1][1] >= 0).mean() > 0.1
        assert same(*out), f"call {k}"
