"""Parity of the gfx950 renderer (libdfpsr_hip.so, through its C ABI) with the CPU oracle.

The bar: coverage and depth bit-exact; RGBA8 within 1 LSB per channel on at least 99.9% of
pixels (colours go through a reciprocal estimate that differs between the reference's SSE
rcpps and the GPU).  Id-colour scenes use the single-colour shader, which involves no
reciprocal, so there every colour must match exactly.
"""
import numpy as np
import pytest

try:  # import torch at collection time: the first import on a fresh machine is slow
    import torch  # noqa: F401
except ImportError:  # pragma: no cover
    torch = None

from dfpsr_amd import scenes as S
from oracle import harness as H
import fixture_scenes

pytestmark = pytest.mark.gpu

COLOR_TOLERANCE_LSB = 1
COLOR_MIN_FRACTION = 0.999


@pytest.fixture(scope="module")
def api():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from dfpsr_amd import api as A
    A.lib()
    return A


@pytest.fixture(scope="module")
def renderer(api):
    return api.renderer_create()


def color_mismatch(got, want):
    a = got.view(np.uint8).reshape(-1, 4).astype(np.int32)
    b = want.view(np.uint8).reshape(-1, 4).astype(np.int32)
    return np.any(np.abs(a - b) > COLOR_TOLERANCE_LSB, axis=1)


def assert_parity(scene, gpu, ref, exact_color=False):
    gc, gd = gpu
    rc, rd = ref
    if scene.has_depth:
        bad = gd.view(np.uint32) != rd.view(np.uint32)
        assert not bad.any(), f"{scene.name}: {int(bad.sum())} depth pixels differ, first at {np.argwhere(bad)[:3].tolist()}"
    if scene.has_color:
        if exact_color:
            bad = gc != rc
            assert not bad.any(), f"{scene.name}: {int(bad.sum())} colour pixels differ, first at {np.argwhere(bad)[:3].tolist()}"
        else:
            bad = color_mismatch(gc, rc)
            allowed = int(np.floor((1.0 - COLOR_MIN_FRACTION) * bad.size))
            assert int(bad.sum()) <= allowed, f"{scene.name}: {int(bad.sum())} pixels beyond 1 LSB (allowed {allowed})"


@pytest.mark.parametrize("scene", fixture_scenes.fixture_scenes(), ids=lambda s: s.name)
def test_fixture_scene(api, renderer, scene):
    print(f"[gpu] fixture {scene.name} {scene.width}x{scene.height}", flush=True)
    gpu = api.render_scene(scene, renderer)
    ref = H.oracle_render(scene)
    assert_parity(scene, gpu, ref, exact_color=scene.name.endswith("_id"))


def test_config0(api, renderer):
    print("[gpu] config0 640x480", flush=True)
    sc = S.cube_soup()
    gpu = api.render_scene(sc, renderer)
    ref = H.oracle_render(sc, threads=8)
    assert_parity(sc, gpu, ref)
    gid = api.render_scene(fixture_scenes.id_color(sc), renderer)
    rid = H.oracle_render(fixture_scenes.id_color(sc), threads=8)
    assert_parity(sc, gid, rid, exact_color=True)


def test_config1(api, renderer):
    print("[gpu] config1 1920x1080", flush=True)
    sc = S.terrain()
    gpu = api.render_scene(sc, renderer)
    ref = H.oracle_render(sc, threads=8)
    assert_parity(sc, gpu, ref)
    covered = np.mean(gpu[1] > 0)
    assert covered > 0.99
    gid = api.render_scene(fixture_scenes.id_color(sc), renderer)
    rid = H.oracle_render(fixture_scenes.id_color(sc), threads=8)
    assert_parity(sc, gid, rid, exact_color=True)


def test_pyramid_matches_golden(api):
    import os
    g = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "texture_vectors.npz"))
    t = api.texture_create_RgbaU8(64, 64, 7)
    api.texture_write_level0(t, g["level0"])
    api.texture_generatePyramid(t)
    assert np.array_equal(t.read(), g["pyramid"])
    assert t.info()[:3] == tuple(int(v) for v in g["log2"])


def test_give_triangles_matches_model_path(api, renderer):
    """renderer_giveTask_triangle with camera-space corners draws what the model path draws."""
    sc = S.cube_soup(width=160, height=120, triangles=300, seed=21, cam_distance=1.2, spread=0.5)
    model_color, model_depth = api.render_scene(sc, renderer)
    cs, _, _ = H.oracle_project(sc, S.identity_transform(), sc.points)
    n = sc.polygon_count
    tri_cs = cs.reshape(n, 3, 3)
    color = np.zeros((sc.height, sc.width), np.uint32)
    depth = np.zeros((sc.height, sc.width), np.float32)
    cam = api.camera_create(True, sc.cam_location, sc.width, sc.height, sc.width_slope, sc.near_clip, sc.far_clip)
    api.renderer_begin(renderer, api.host_image(color), api.host_image(depth))
    api.renderer_giveTask_triangles(renderer, tri_cs, sc.colors[:, :3, :], sc.texcoords[:, :3, :], None, None, 0, cam)
    api.renderer_end(renderer)
    assert np.array_equal(depth.view(np.uint32), model_depth.view(np.uint32))
    assert np.array_equal(color, model_color)


def projected_by_oracle(sc):
    """The scene's triangles as ProjectedPoint records that the oracle's cameraToScreen makes
    from their camera-space corners (bit-exact to the reference's own projection)."""
    import copy
    cs, is_, flat = H.oracle_project(sc, S.identity_transform(), sc.points)
    n = sc.polygon_count
    rec = np.zeros((n, 3), fixture_scenes.H_PROJECTED)
    rec["cs"], rec["is"], rec["flat"] = cs.reshape(n, 3, 3), is_.reshape(n, 3, 2), flat.reshape(n, 3, 2)
    out = copy.copy(sc)
    out.projected = rec
    return out


def test_give_triangles_matches_oracle(api, renderer):
    """renderer_giveTask_triangle with camera-space corners (the device projects them) draws
    what the oracle's renderer_giveTask_triangle draws from the reference's projection of the
    same corners; the ProjectedPoint entry given those projections draws the same canvases."""
    n = 300
    sc = S.cube_soup(width=160, height=120, triangles=n, seed=21, cam_distance=1.2, spread=0.5)
    sc.textures = [S.noise_checker_texture(64, 21, 7, check=8)]
    sc.parts = [S.Part(0, n, diffuse=0)]
    sc.texcoords[:, :3, :2] = S.Rng(22).uniform(n * 6, -1, 2).reshape(n, 3, 2)
    ref = projected_by_oracle(sc)
    want = H.oracle_render(ref)
    g = api.GpuScene(sc)
    cam = api.camera_create(True, sc.cam_location, sc.width, sc.height, sc.width_slope, sc.near_clip, sc.far_clip)
    for entry in ("camera_space", "projected"):
        color = np.zeros((sc.height, sc.width), np.uint32)
        depth = np.zeros((sc.height, sc.width), np.float32)
        api.renderer_begin(renderer, api.host_image(color), api.host_image(depth))
        if entry == "camera_space":
            api.renderer_giveTask_triangles(renderer, ref.projected["cs"], sc.colors[:, :3, :], sc.texcoords[:, :3, :],
                                            g.textures[0], None, 0, cam)
        else:
            api.renderer_giveTask_projected(renderer, ref.projected, sc.colors[:, :3, :], sc.texcoords[:, :3, :],
                                            g.textures[0], None, 0, cam)
        api.renderer_end(renderer)
        assert (depth > 0).mean() > 0.2
        assert_parity(sc, (color, depth), want)


def test_device_canvases_match_host_canvases(api, renderer):
    import torch
    sc = fixture_scenes.clip_scenes()[2]
    hc, hd = api.render_scene(sc, renderer)
    g = api.GpuScene(sc)
    color = torch.zeros((sc.height, sc.width + 5), dtype=torch.int32, device="cuda")[:, :sc.width]
    depth = torch.zeros((sc.height, sc.width), dtype=torch.float32, device="cuda")
    api.renderer_begin(renderer, api.device_image(color), api.device_image(depth))
    g.give(renderer)
    api.renderer_end(renderer)
    torch.cuda.synchronize()
    assert np.array_equal(color.cpu().numpy().view(np.uint32), hc)
    assert np.array_equal(depth.cpu().numpy().view(np.uint32), hd.view(np.uint32))


def test_repeated_frames_identical(api, renderer):
    sc = fixture_scenes.variant(1)
    a = api.render_scene(sc, renderer)
    b = api.render_scene(sc, renderer)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_call_order_errors(api):
    r = api.renderer_create()
    with pytest.raises(api.DfpsrError) as e:
        api.renderer_end(r)
    assert e.value.code == -2
    color = np.zeros((8, 8), np.uint32)
    api.renderer_begin(r, api.host_image(color), api.host_image(None))
    assert api.renderer_takesTriangles(r)
    with pytest.raises(api.DfpsrError) as e:
        api.renderer_begin(r, api.host_image(color), api.host_image(None))
    assert e.value.code == -2
    api.renderer_end(r)
    assert not api.renderer_takesTriangles(r)
    with pytest.raises(api.DfpsrError):
        api.renderer_begin(r, api.host_image(color), api.host_image(np.zeros((4, 8), np.float32)))


def even_height(scene):
    """The scene on a canvas one row taller when its height is odd (initial canvases padded
    with a copy of their last row), so that frames of Solid perspective scenes qualify for the
    visibility raster."""
    import copy
    if scene.height % 2 == 0:
        return scene
    sc = copy.copy(scene)
    sc.height = scene.height + 1
    if scene.initial_color is not None:
        sc.initial_color = np.vstack([scene.initial_color, scene.initial_color[-1:]])
    if scene.initial_depth is not None:
        sc.initial_depth = np.vstack([scene.initial_depth, scene.initial_depth[-1:]])
    sc.name = scene.name + "_even"
    return sc


PATH_SCENES = [even_height(s) for s in fixture_scenes.fixture_scenes()] + [S.cube_soup(width=320, height=240, triangles=3000, seed=9)]


@pytest.mark.parametrize("scene", PATH_SCENES, ids=lambda s: s.name)
def test_visibility_raster_equals_in_order_raster(api, scene):
    """The visibility raster (atomic-max winner per pixel, shaded once) gives bit-identical
    canvases to the in-order walk, for every tile shape and both ways of building the tile
    lists, and all meet the oracle's bar."""
    print(f"[gpu] raster paths {scene.name} {scene.width}x{scene.height}", flush=True)
    results = []
    for tile_config in (0, 1, 2):
        for path in (0, 1):
            for binning in (0, 1):
                r = api.renderer_create()
                api.renderer_setTuning(r, api.tuning(tile_config=tile_config, raster_path=path, binning=binning))
                results.append(api.render_scene(scene, r))
    for c, d in results[1:]:
        assert np.array_equal(c, results[0][0]) and np.array_equal(d.view(np.uint32), results[0][1].view(np.uint32))
    assert_parity(scene, results[0], H.oracle_render(scene), exact_color=scene.name.endswith("_id") or
                  scene.name.endswith("_id_even"))


def odd_scene(width, height, orthogonal, canvases, seed):
    """Large overlapping triangles, whose spans' unclipped quads reach the odd canvas's last row, over
    a depth canvas that holds ordinary values, infinities and NaN."""
    sc = S.cube_soup(width=width, height=height, triangles=120, seed=seed, spread=0.9, cam_distance=2.0,
                     name=f"odd_{width}x{height}_{'ortho' if orthogonal else 'persp'}_{canvases}")
    sc.perspective = not orthogonal
    sc.has_color, sc.has_depth = "c" in canvases, "d" in canvases
    held = S.Rng(seed + 5).uniform(width * height, 0.0, 0.6 if not orthogonal else 4.0).reshape(height, width)
    held.reshape(-1)[::7] = np.inf if orthogonal else 0.0
    held.reshape(-1)[3::11] = np.nan
    held.reshape(-1)[5::13] = -np.inf
    sc.initial_depth = held
    return sc


@pytest.mark.parametrize("orthogonal", [False, True])
@pytest.mark.parametrize("canvases", ["cd", "c", "d"])
@pytest.mark.parametrize("size", [(1, 1), (61, 17), (33, 33), (130, 47), (64, 32)])
def test_visibility_raster_of_odd_heights_and_orthogonal_cameras(api, size, canvases, orthogonal):
    """The visibility raster walks an odd canvas's last row in order and reverses its depth order under
    an orthogonal camera: the same canvases as the in-order raster, bit for bit, for every tile shape,
    with and without persistent workgroups; and the oracle's."""
    sc = odd_scene(size[0], size[1], orthogonal, canvases, seed=size[0] * 7 + size[1])
    print(f"[gpu] odd rows {sc.name}", flush=True)
    results = []
    for tile_config in (0, 1, 2):
        for path, persistent in ((1, 0), (0, 0), (0, 2)):
            r = api.renderer_create()
            api.renderer_setTuning(r, api.tuning(tile_config=tile_config, raster_path=path, persistent_per_cu=persistent))
            results.append(api.render_scene(sc, r))
    for c, d in results[1:]:
        assert np.array_equal(c, results[0][0]) and np.array_equal(d.view(np.uint32), results[0][1].view(np.uint32))
    assert_parity(sc, results[0], H.oracle_render(sc))


@pytest.mark.parametrize("orthogonal", [False, True])
@pytest.mark.parametrize("canvases", ["cd", "c", "d"])
@pytest.mark.parametrize("size", [(50, 31), (96, 64)])
def test_alpha_runs_between_solid_runs(api, size, canvases, orthogonal):
    """Solid and Alpha models taking turns on one canvas (runs within one chunk of a tile, and across
    chunks and rounds): the visibility raster with its blended runs gives the in-order raster's canvases
    bit for bit, over held colours and depths, for every tile shape."""
    parts = []
    for k in range(5):
        sc = odd_scene(size[0], size[1], orthogonal, canvases, seed=50 + k)
        sc.filter = k % 2
        n = [3, 4, 120, 120, 5][k]
        sc.indices, sc.colors, sc.texcoords, sc.parts = sc.indices[:n], sc.colors[:n], sc.texcoords[:n].copy(), [S.Part(0, n, diffuse=0)]
        sc.colors[:, :, 3] = S.Rng(60 + k).uniform(n * 4).reshape(n, 4)
        sc.texcoords[:, :3, :2] = S.Rng(70 + k).uniform(n * 6, -1.0, 2.0).reshape(n, 3, 2)
        sc.textures = [S.noise_checker_texture(32, k, 6, check=4)]
        parts.append(api.GpuScene(sc))
    held_color = S.Rng(5).u64(size[0] * size[1]).astype(np.uint32).reshape(size[1], size[0])
    results = []
    for tile_config in (0, 1, 2):
        for path, persistent in ((1, 0), (0, 0), (0, 2)):
            r = api.renderer_create()
            api.renderer_setTuning(r, api.tuning(tile_config=tile_config, raster_path=path, persistent_per_cu=persistent))
            color, depth = held_color.copy(), parts[0].scene.initial_depth.copy()
            api.renderer_begin(r, api.host_image(color if "c" in canvases else None), api.host_image(depth if "d" in canvases else None))
            for g in parts + parts[:2]:
                g.give(r)
            api.renderer_end(r)
            results.append((color, depth))
    for c, d in results[1:]:
        assert np.array_equal(c, results[0][0]) and np.array_equal(d.view(np.uint32), results[0][1].view(np.uint32))
    if "c" in canvases:
        assert (results[0][0] != held_color).mean() > 0.1


def test_canvas_with_both_projections(api):
    """A frame whose tasks mix perspective and orthogonal cameras on one canvas changes the direction of
    the depth test between commands: both raster settings draw it in order."""
    persp, ortho = odd_scene(90, 41, False, "cd", 3), odd_scene(90, 41, True, "cd", 4)
    a, b = api.GpuScene(persp), api.GpuScene(ortho)
    out = []
    for path in (0, 1):
        color, depth = np.zeros((41, 90), np.uint32), persp.initial_depth.copy()
        r = api.renderer_create()
        api.renderer_setTuning(r, api.tuning(raster_path=path))
        api.renderer_begin(r, api.host_image(color), api.host_image(depth))
        for g in (a, b, a):
            g.give(r)
        api.renderer_end(r)
        out.append((color, depth))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1].view(np.uint32), out[1][1].view(np.uint32))
    assert (out[0][0] != 0).any()


@pytest.mark.parametrize("log2_reach", [12, 19, 23, 24, 27])
def test_rows_of_far_corners(api, renderer, log2_reach):
    """Corners up to 2^27 sub-pixels away, some edges nearly horizontal or vertical: below 2^24 a row's
    sides come from doubles, beyond that from 64-bit integers, and both give the oracle's rows."""
    n = 150
    sc = projected_by_oracle(S.cube_soup(width=120, height=75, triangles=n, seed=log2_reach, cam_distance=2.0, spread=0.6))
    rng = S.Rng(1000 + log2_reach)
    reach = 1 << log2_reach
    flat = rng.integers(n * 6, -reach, reach).reshape(n, 3, 2) + np.array([60, 37]) * 256
    flat[::3, 1, 1] = flat[::3, 0, 1] + rng.integers((n + 2) // 3, -1, 2)   # an edge of at most 1 / 256 row
    flat[1::3, 2, 0] = flat[1::3, 0, 0] + rng.integers((n + 1) // 3, -1, 2)
    sc.projected = sc.projected.copy()
    sc.projected["flat"] = flat
    print(f"[gpu] far corners 2^{log2_reach}", flush=True)
    ref = H.oracle_render(sc)
    assert (ref[1] > 0).any()
    for path in (0, 1):
        r = api.renderer_create()
        api.renderer_setTuning(r, api.tuning(tile_config=1, raster_path=path))
        assert_parity(sc, api.render_scene(sc, r), ref)


def test_direct_bins_grow_to_the_longest_tile_list(api):
    """Tiles holding more commands than the direct bins' starting size (64) make the first frame
    overflow them: the renderer grows the bins to the longest list and draws the frame again
    (two passes); the next frame fits in one.  Canvases and pair counts equal those of the
    scanned lists, and the oracle's bar holds."""
    sc = S.cube_soup(width=48, height=32, triangles=900, seed=5, spread=0.3, cam_distance=2.0, name="dense_bins")
    print(f"[gpu] dense bins {sc.width}x{sc.height}", flush=True)
    scanned_renderer = api.renderer_create()
    api.renderer_setTuning(scanned_renderer, api.tuning(binning=1))
    scanned = api.render_scene(sc, scanned_renderer)
    scanned_stats = scanned_renderer.stats()
    r = api.renderer_create()
    api.renderer_setTuning(r, api.tuning(binning=0))
    first = api.render_scene(sc, r)
    first_stats = r.stats()
    second = api.render_scene(sc, r)
    second_stats = r.stats()
    assert first_stats[3] == 2 and second_stats[3] == 1
    for got in (first, second):
        assert np.array_equal(got[0], scanned[0]) and np.array_equal(got[1].view(np.uint32), scanned[1].view(np.uint32))
    assert list(first_stats[:3]) == list(scanned_stats[:3]) == list(second_stats[:3])
    assert_parity(sc, first, H.oracle_render(sc))


@pytest.mark.parametrize("width,height,triangles,spread,distance,orthogonal", [
    (37, 23, 3000, 0.02, 2.5, False),    # below a pixel: most cover no pixel centre
    (37, 23, 3000, 0.02, 2.5, True),
    (97, 40, 2500, 1.2, 0.7, False),     # long slivers far outside the canvas, clipped near the camera
    (64, 33, 1500, 0.3, 1.6, False),     # a few tiles each, column 0 and the last row among them
])
def test_dense_canvas_pairs(api, width, height, triangles, spread, distance, orthogonal):
    """On canvases with few pixels per triangle the setup drops the (command, tile) pairs that no row
    covers: every tile shape, both ways of building the lists and both rasters still give the oracle's
    depth bit for bit, and so does the depth-only draw."""
    sc = S.cube_soup(width=width, height=height, triangles=triangles, seed=triangles + width, spread=spread, cam_distance=distance)
    sc.perspective = not orthogonal
    if orthogonal:
        sc.initial_depth = np.full((height, width), np.inf, np.float32)
    assert width * height < 8 * triangles
    print(f"[gpu] dense pairs {width}x{height} {triangles} spread {spread}", flush=True)
    ref = H.oracle_render(sc, threads=4)
    pairs = set()
    for tile_config in (0, 1, 2):
        for path, binning in ((0, 0), (0, 1), (1, 0)):
            r = api.renderer_create()
            api.renderer_setTuning(r, api.tuning(tile_config=tile_config, raster_path=path, binning=binning))
            assert_parity(sc, api.render_scene(sc, r), ref)
            pairs.add((tile_config, int(r.stats()[1])))
    assert len(pairs) == 3  # the same pairs whatever the lists and the raster
    depth = api.render_scene_depth(sc)
    want = H.oracle_render_depth(sc)
    assert np.array_equal(depth.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("triangles", [120, 300, 600, 2600, 12000])
def test_tile_lists_longer_than_a_round(api, triangles):
    """A canvas of one tile whose triangles all reach it: lists below and above the 128, 256 and 1,024
    commands that the rasters sort per round, in several rounds, against the oracle."""
    sc = S.cube_soup(width=30, height=16, triangles=triangles, seed=triangles, spread=0.7, cam_distance=2.2)
    # A second cluster of command indices far from the first: the middle half faces away.
    a, b = triangles // 4, 3 * triangles // 4
    sc.indices[a:b, :3] = sc.indices[a:b, 2::-1]
    print(f"[gpu] long lists {triangles}", flush=True)
    ref = H.oracle_render(sc, threads=4)
    for tile_config, path in ((1, 0), (1, 1), (0, 0), (2, 1)):
        r = api.renderer_create()
        api.renderer_setTuning(r, api.tuning(tile_config=tile_config, raster_path=path))
        assert_parity(sc, api.render_scene(sc, r), ref)
    depth, want = api.render_scene_depth(sc), H.oracle_render_depth(sc)
    assert np.array_equal(depth.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("triangles", [100, 400, 1500])
def test_persistent_grid_draws_long_lists_first(api, triangles):
    """Tiles whose lists are short, long (over 128 commands) and longest (over 512) on one canvas: the
    persistent grid's order of tiles changes nothing, with and without the fused fill, and no tile is
    drawn twice or left out."""
    near = S.cube_soup(width=200, height=70, triangles=triangles, seed=triangles, spread=0.15, cam_distance=3.0)
    wide = S.cube_soup(width=200, height=70, triangles=200, seed=9, spread=1.2, cam_distance=3.0)
    a, b = api.GpuScene(near), api.GpuScene(wide)
    print(f"[gpu] persistent long lists {triangles}", flush=True)
    for clear in (False, True):
        out = []
        for persistent, binning, path, tile_config in ((0, 0, 0, 1), (1, 0, 0, 1), (4, 1, 0, 1), (2, 1, 0, 0), (1, 1, 1, 2)):
            r = api.renderer_create()
            api.renderer_setTuning(r, api.tuning(persistent_per_cu=persistent, binning=binning, raster_path=path, tile_config=tile_config,
                                                 clear=clear, clear_color=0x11223344, clear_depth=0.0))
            for _ in range(2):
                color, depth = np.full((70, 200), 7, np.uint32), np.zeros((70, 200), np.float32)
                api.renderer_begin(r, api.host_image(color), api.host_image(depth))
                a.give(r)
                b.give(r)
                api.renderer_end(r)
                out.append((color, depth))
        assert (out[0][1] > 0).any()
        for color, depth in out[1:]:
            assert np.array_equal(color, out[0][0]) and np.array_equal(depth.view(np.uint32), out[0][1].view(np.uint32))


def test_packed_lists_grow_past_their_first_pair_capacity(api):
    """Commands whose bounds span the whole canvas touch every tile, so the frame makes more
    (tile, command) pairs than the packed lists' first capacity (four per command slot): the
    setup kernel's pair records stop at the capacity, the frame is drawn again with room for its
    pair count (two passes), and the next frame fits in one.  Canvases and pair counts equal
    those of the direct bins, and the oracle's bar holds."""
    w, h = 640, 480
    tris = []
    for k in range(12):
        if k % 2 == 0:
            tris.append([(-20.0, -20.0), (w + 20.0, -20.0), (-20.0, h + 20.0)])
        else:
            tris.append([(w + 20.0, -20.0), (w + 20.0, h + 20.0), (-20.0, h + 20.0)])
    sc = S.single_triangles(w, h, tris, depth=np.linspace(2.0, 3.0, 12), name="wide_pairs")
    print(f"[gpu] packed pair capacity {sc.width}x{sc.height}", flush=True)
    direct = api.renderer_create()
    api.renderer_setTuning(direct, api.tuning(binning=0))
    want = api.render_scene(sc, direct)
    want_stats = direct.stats()
    r = api.renderer_create()
    api.renderer_setTuning(r, api.tuning(binning=1))
    first = api.render_scene(sc, r)
    first_stats = r.stats()
    second = api.render_scene(sc, r)
    second_stats = r.stats()
    assert first_stats[1] > 4 * (len(tris) + 1024)
    assert first_stats[3] == 2 and second_stats[3] == 1
    for got in (first, second):
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32))
    assert list(first_stats[:3]) == list(want_stats[:3]) == list(second_stats[:3])
    assert_parity(sc, first, H.oracle_render(sc))


def test_every_buffer_of_a_dense_frame_grows(api):
    """Thin triangles from behind the camera on a small dense canvas beside a large, nearly empty one: the
    setup's blocks make more commands than their slots (first pass), then the bins overflow and, grown,
    pass their bound (second pass), and the lists are packed, whose records include the many pairs that a
    bound touches and no row covers (third pass, and a fourth with room for them)."""
    count, w, h = 4096, 160, 128
    rng = S.Rng(12)
    ends = rng.uniform(count * 2, -1.0, 1.0).reshape(count, 2)
    starts = rng.uniform(count * 2, -3.0, 3.0).reshape(count, 2)
    pts = np.zeros((count, 3, 3), np.float32)
    pts[:, 0, :2], pts[:, 0, 2] = starts, -0.5
    pts[:, 1, :2], pts[:, 1, 2] = ends * 2.0, 2.0
    pts[:, 2] = pts[:, 1] + rng.uniform(count * 3, -0.002, 0.002).reshape(count, 3)
    away = (np.cross(pts[:, 1] - pts[:, 0], pts[:, 2] - pts[:, 0]) * pts[:, 0]).sum(1) > 0
    pts[away] = pts[away][:, [0, 2, 1]]  # every triangle faces the camera
    thin = clip_heavy_scene(count)
    thin.width, thin.height, thin.points = w, h, pts.reshape(-1, 3)
    large = S.single_triangles(8192, 8192, [[(10.0, 10.0), (10.0, 60.0), (60.0, 10.0)], [(10.0, 10.0), (60.0, 10.0), (10.0, 60.0)]])
    g = api.GpuJobs([thin])
    depth = torch.zeros((8192, 8192), device="cuda")
    model = api.GpuScene(large)
    jobs = (api.Job * 2)()
    jobs[0] = g.jobs[0]
    jobs[1].depth, jobs[1].model, jobs[1].camera = api.device_image(depth), model.model.handle, model.camera
    jobs[1].transform[:] = [float(v) for v in S.identity_transform()]
    print("[gpu] every buffer grows", flush=True)
    b = api.Batch()
    b.render(jobs, api.tuning())
    assert b.stats()[3] == 4
    got = g.image(0)
    assert (depth > 0).any()
    g.clear()
    r = api.renderer_create()
    api.renderer_setTuning(r, api.tuning(raster_path=1, binning=1))
    g.render_plain(r)
    want = g.image(0)
    assert (want[1] > 0).mean() > 0.2
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32))


def test_setup_offsets_scanned_for_many_fan_triangles(api):
    """Above 2048 setup blocks (524288 fan triangles) the command offsets come from the block
    scan kernel instead of each block summing the totals before it; both give the oracle's
    canvases."""
    sc = S.cube_soup(width=64, height=48, triangles=540000, seed=3, spread=0.02, cam_distance=2.5, name="many_triangles")
    print(f"[gpu] many fan triangles {sc.indices.shape[0]}", flush=True)
    got = api.render_scene(sc)
    assert_parity(sc, got, H.oracle_render(sc))


def clip_heavy_scene(triangles=256, seed=31):
    """Large triangles around the camera: each crosses the near plane and several sides of the
    clip frustum, so clipping splits it into several draw commands and one setup block (256 fan
    triangles) makes far more than the 512 commands its block-wide binning table holds."""
    rng = S.Rng(seed)
    jitter = rng.uniform(triangles * 9, -0.3, 0.3).reshape(triangles, 3, 3).astype(np.float32)
    base = np.array([[-4.0, -3.0, -0.5], [4.0, -3.0, 3.0], [0.0, 4.0, 3.0]], dtype=np.float32)
    tri = base[None, :, :] + jitter
    tri = tri[:, ::-1]  # clockwise on screen: every triangle faces the camera
    pts = tri.reshape(-1, 3)
    idx = np.full((triangles, 4), -1, dtype=np.int32)
    idx[:, :3] = np.arange(triangles * 3, dtype=np.int32).reshape(triangles, 3)
    colors = np.ones((triangles, 4, 4), dtype=np.float32)
    colors[:, :3, :3] = rng.uniform(triangles * 9, 0.0, 1.0).reshape(triangles, 3, 3).astype(np.float32)
    return S.Scene(name="clip_heavy", width=96, height=64, points=pts, indices=idx, colors=colors,
                   texcoords=np.zeros((triangles, 4, 4), dtype=np.float32), parts=[S.Part(0, triangles)], textures=[],
                   cam_location=S.identity_transform(), width_slope=1.0, far_clip=100.0, seed=seed)


def test_setup_block_with_more_commands_than_its_binning_table(api):
    """A setup block whose fan triangles make more than 512 draw commands bins them thread by
    thread instead of block-wide; the canvases still meet the oracle's bar and match the packed
    lists bit for bit."""
    sc = clip_heavy_scene()
    print(f"[gpu] clip-heavy block {sc.width}x{sc.height}", flush=True)
    r = api.renderer_create()
    got = api.render_scene(sc, r)
    assert r.stats()[0] > 512
    packed = api.renderer_create()
    api.renderer_setTuning(packed, api.tuning(binning=1))
    ref = api.render_scene(sc, packed)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1].view(np.uint32), ref[1].view(np.uint32))
    assert_parity(sc, got, H.oracle_render(sc))


@pytest.mark.parametrize("sizes", [(1,), (3, 1, 64, 2), (200, 40, 7)])
def test_tasks_smaller_than_a_wavefront(api, sizes):
    """Triangles given in tasks of a few at a time, clipped ones among whole ones, share the setup's
    wavefronts and blocks: the canvases are those of one task bit for bit, and the oracle's."""
    sc = clip_heavy_scene(triangles=300)
    whole = S.cube_soup(width=96, height=64, triangles=300, seed=6, cam_distance=2.0, spread=0.6)
    moved = sc.points.reshape(300, 3, 3)
    keep = np.arange(300) % 5 != 0
    # Whole triangles in front of the camera: the soup's, moved along the view axis.
    moved[keep] = whole.points.reshape(300, 3, 3)[keep] + np.array([0.0, 0.0, 2.5], np.float32)
    ref = projected_by_oracle(sc)
    print(f"[gpu] tasks of {sizes}", flush=True)
    want = H.oracle_render(ref)
    cam = api.camera_create(True, sc.cam_location, sc.width, sc.height, sc.width_slope, sc.near_clip, sc.far_clip)
    out = []
    for split in ((300,), sizes):
        r = api.renderer_create()
        color, depth = np.zeros((sc.height, sc.width), np.uint32), np.zeros((sc.height, sc.width), np.float32)
        api.renderer_begin(r, api.host_image(color), api.host_image(depth))
        at = k = 0
        while at < 300:
            end = min(at + split[k % len(split)], 300)
            api.renderer_giveTask_triangles(r, ref.projected["cs"][at:end], sc.colors[at:end, :3, :], sc.texcoords[at:end, :3, :], None, None, 0, cam)
            at, k = end, k + 1
        api.renderer_end(r)
        out.append((color, depth, r.stats()[0]))
    assert out[0][2] == out[1][2] > 300  # some triangles are split, some whole
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1].view(np.uint32), out[1][1].view(np.uint32))
    assert_parity(sc, out[1][:2], want)


def test_points_replaced_by_fewer_are_refused_by_every_draw(api):
    """A model whose points were replaced by fewer after its polygons were added is refused with
    an argument error by renderer_giveTask, the batch and the differentiable forward, and the
    canvases stay untouched."""
    import torch
    sc = S.cube_soup(width=32, height=24, triangles=20, seed=4)
    jobs = api.GpuJobs([sc])
    model = jobs.gpu[0]
    api.model_setPoints(model, sc.points[:-3])
    r = api.renderer_create()
    color = np.zeros((sc.height, sc.width), np.uint32)
    api.renderer_begin(r, api.host_image(color), api.host_image(None))
    cam = api.camera_create(sc.perspective, sc.cam_location, sc.width, sc.height, sc.width_slope, sc.near_clip, sc.far_clip)
    with pytest.raises(api.DfpsrError) as e:
        api.renderer_giveTask(r, model, sc.instances[0], cam)
    assert e.value.code == -1 and "does not have" in str(e.value)
    api.renderer_end(r)
    assert not color.any()
    batch = api.Batch()
    with pytest.raises(api.DfpsrError) as e:
        batch.render(jobs.jobs, api.tuning())
    assert e.value.code == -1
    torch.cuda.synchronize()
    assert not jobs.colors[0].any().item()
    views = api.GpuViews([sc])
    api.model_setPoints(views.model, sc.points[:-3])
    diff = api.DiffRenderer()
    tex = torch.full((8, 8, 4), 0.5, dtype=torch.float32, device="cuda")
    with pytest.raises(api.DfpsrError) as e:
        diff.forward(views.model, views.views, tex)
    assert e.value.code == -1


@pytest.mark.parametrize("scene", fixture_scenes.occlusion_scenes(), ids=lambda s: s.name)
def test_occlusion_queries_commands_and_grid(api, scene):
    """The renderer's occluder calls: box-query answers, the draw commands left after
    completeOcclusion and the final grid equal the oracle's, and the canvases meet the bar."""
    print(f"[gpu] occlusion {scene.name}", flush=True)
    r = api.renderer_create()
    g = api.GpuScene(scene)
    color = np.zeros((scene.height, scene.width), np.uint32)
    depth = scene.initial_depth.copy() if scene.initial_depth is not None else np.zeros((scene.height, scene.width), np.float32)
    api.renderer_begin(r, api.host_image(color), api.host_image(depth))
    assert not api.renderer_hasOccluders(r)
    g.give(r)
    assert api.renderer_hasOccluders(r)
    api.renderer_end(r)
    oc, od, visible = H.oracle_render_queries(scene)
    assert [int(v) for v in g.visible] == visible.tolist()
    assert int(r.stats()[0]) == len(H.oracle_commands(scene)[0])
    grid, _ = H.oracle_occlusion_grid(scene)
    assert np.array_equal(api.renderer_occlusionGrid(r).view(np.uint32), grid.view(np.uint32))
    assert_parity(scene, (color, depth), (oc, od))


def test_occlusion_grid_outlives_the_frame(api):
    """A box query before the frame's first occluder call reads the grid the previous frame
    left (the reference keeps its grid image); a renderer that never had a grid reads 0."""
    sc = fixture_scenes.occlusion_scenes()[0]
    g = api.GpuScene(sc)
    box = ((-0.5, -0.5, -0.5), (0.5, 0.5, 0.5))
    r = api.renderer_create()
    color = np.zeros((sc.height, sc.width), np.uint32)
    api.renderer_begin(r, api.host_image(color), api.host_image(None))
    answers_fresh = [api.renderer_isBoxVisible(r, *box, _translate(x), g.camera) for x in (-6.0, 0.0, 6.0)]
    g.give(r)
    answers_end = [api.renderer_isBoxVisible(r, *box, _translate(x), g.camera) for x in (-6.0, 0.0, 6.0)]
    api.renderer_end(r)
    api.renderer_begin(r, api.host_image(color), api.host_image(None))
    answers_next = [api.renderer_isBoxVisible(r, *box, _translate(x), g.camera) for x in (-6.0, 0.0, 6.0)]
    assert not api.renderer_hasOccluders(r)
    api.renderer_end(r)
    assert answers_fresh == [False, False, False]
    assert answers_next == answers_end and True in answers_end and False in answers_end


def _translate(x):
    t = S.identity_transform().copy()
    t[0], t[2] = x, 2.0
    return t


def test_occlusion_calls_need_begin_and_a_depth_canvas(api):
    r = api.renderer_create()
    cam = api.camera_create(True, S.identity_transform(), 32, 32, 1.0)
    with pytest.raises(api.DfpsrError) as e:
        api.renderer_occludeFromExistingTriangles(r)
    assert e.value.code == -2
    color = np.zeros((32, 32), np.uint32)
    api.renderer_begin(r, api.host_image(color), api.host_image(None))
    with pytest.raises(api.DfpsrError) as e:
        api.renderer_occludeFromTopRows(r, cam)
    assert e.value.code == -2 and "depth buffer" in str(e.value)
    api.renderer_end(r)


def test_consecutive_frames_on_one_renderer(api):
    """Frames drawn one after another on one renderer (the counts one frame's raster leaves
    zeroed are the next frame's starting counts) equal frames drawn on fresh renderers: scenes
    of different sizes, a crowded one whose tile bins overflow and are redrawn, and repeats."""
    small = S.cube_soup(width=160, height=120, triangles=400, seed=31, spread=0.3, cam_distance=1.5, name="small")
    wide = S.cube_soup(width=400, height=240, triangles=1500, seed=32, spread=0.4, cam_distance=1.8, name="wide")
    crowded = S.cube_soup(width=96, height=64, triangles=6000, seed=33, spread=0.6, cam_distance=1.6, name="crowded")
    textured = fixture_scenes.shader_branch_scenes()[0]
    order = [small, wide, small, crowded, small, textured, wide, wide, crowded, small]
    r = api.renderer_create()
    for i, sc in enumerate(order):
        print(f"[gpu] frame {i}: {sc.name} {sc.width}x{sc.height}", flush=True)
        got = api.render_scene(sc, r)
        want = api.render_scene(sc, api.renderer_create())
        assert np.array_equal(got[0], want[0]), f"frame {i} ({sc.name}): colour differs from a fresh renderer's"
        assert np.array_equal(got[1].view(np.uint32), want[1].view(np.uint32)), f"frame {i} ({sc.name}): depth differs"
    assert_parity(small, api.render_scene(small, r), H.oracle_render(small))
