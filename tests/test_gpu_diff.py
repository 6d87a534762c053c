"""The differentiable form: forward on the reference raster with a float shader, adjoint with
visibility fixed from the forward.

Checks: the forward against the CPU oracle (visibility and depth bit-exact, colour to float
rounding); the adjoint against the oracle's float64 adjoint built on the same coverage and
against the dot-product identity <g, F(T)> = <F^T g, T> (the colour is linear in the texture
and in the multipliers); central finite differences on the full 8-view 1280x720 fit; the Adam
fit itself; and the 256-view batched form against the per-view form.
"""
import numpy as np
import pytest

try:
    import torch
except ImportError:  # pragma: no cover
    torch = None

from dfpsr_amd import scenes as S
from oracle import harness as H

pytestmark = pytest.mark.gpu

# Tolerances written into the checks below.
FORWARD_RTOL = 1e-5          # colour vs oracle: weights differ only by the reciprocal estimate ...
FORWARD_FLIP_FRACTION = 1e-3  # ... except where u or v sits on an 8-bit sub-texel boundary and the
FORWARD_FLIP_ATOL = 1.0 / 128  # tap weights move by one step of 1/256 (texels and multipliers < 2);
                               # the same 99.9% bar as the RGBA8 path's colours
ADJOINT_RTOL = 1e-3          # GPU float32 atomics vs the oracle's float64 adjoint
FD_RTOL = 1e-3               # analytic gradient vs central finite differences (h = 1e-3), no floor
BATCHED_GRAD_RTOL = 1e-4     # 256-view batched adjoint vs the sum of per-view adjoints


@pytest.fixture(scope="module")
def api():
    assert torch is not None and torch.cuda.is_available()
    from dfpsr_amd import api as A
    A.lib()
    return A


class RenderFunction(torch.autograd.Function if torch is not None else object):
    """torch.autograd wrapper of the C ABI, for these tests only."""

    @staticmethod
    def forward(ctx, texture, multipliers, renderer, gv, tuning):
        renderer.forward(gv.model, gv.views, texture, multipliers, tuning)
        ctx.renderer, ctx.gv, ctx.tuning = renderer, gv, tuning
        ctx.shapes = (texture.shape, multipliers.shape)
        return torch.stack([c.clone() for c in gv.color])

    @staticmethod
    def backward(ctx, grad):
        gv = ctx.gv
        for i, g in enumerate(gv.grad):
            g.copy_(grad[i])
        gt = torch.zeros(ctx.shapes[0], dtype=torch.float32, device="cuda")
        gm = torch.zeros(ctx.shapes[1], dtype=torch.float32, device="cuda")
        ctx.renderer.backward(gt, gm, ctx.tuning)
        return gt, gm, None, None, None


def small_views():
    return S.sphere_views(12, 3, 320, 180, seed=4)


def test_forward_matches_oracle(api):
    views = small_views()
    gv = api.GpuViews(views)
    tex = S.float_texture(64, 1)
    mul = (1.0 + 0.3 * S.Rng(8).uniform(views[0].points.shape[0] * 3, -1, 1)).reshape(-1, 3).astype(np.float32)
    r = api.DiffRenderer()
    r.forward(gv.model, gv.views, torch.from_numpy(tex).cuda(), torch.from_numpy(mul).cuda(), api.tuning(clear=True))
    torch.cuda.synchronize()
    for i, sc in enumerate(views):
        col, vis, dep, w = H.oracle_diff_forward(sc, tex, mul)
        assert np.array_equal(gv.visibility[i].cpu().numpy(), vis), f"view {i} visibility"
        assert np.array_equal(gv.depth[i].cpu().numpy().view(np.uint32), dep.view(np.uint32)), f"view {i} depth"
        got = gv.color[i].cpu().numpy()
        close = np.isclose(got, col, rtol=FORWARD_RTOL, atol=1e-6)
        assert 1.0 - close.mean() <= FORWARD_FLIP_FRACTION, f"view {i}: {int((~close).sum())} values differ"
        assert np.max(np.abs(got - col)) <= FORWARD_FLIP_ATOL
        assert (vis >= 0).mean() > 0.3


def test_forward_of_clipped_triangles(api):
    """Differentiable frames whose near plane cuts the object: clipped and whole triangles in the
    setup's two passes give the oracle's visibility and depth."""
    views = S.sphere_views(10, 3, 96, 64, seed=5)
    for v in views:
        v.near_clip = float(np.linalg.norm(np.asarray(v.cam_location[:3], np.float64))) - 0.8
    gv = api.GpuViews(views)
    tex = S.float_texture(64, 2)
    print("[gpu] clipped differentiable views", flush=True)
    r = api.DiffRenderer()
    r.forward(gv.model, gv.views, torch.from_numpy(tex).cuda(), None, api.tuning(clear=True))
    torch.cuda.synchronize()
    for i, sc in enumerate(views):
        col, vis, dep, _ = H.oracle_diff_forward(sc, tex, None)
        assert np.array_equal(gv.visibility[i].cpu().numpy(), vis), f"view {i} visibility"
        assert np.array_equal(gv.depth[i].cpu().numpy().view(np.uint32), dep.view(np.uint32)), f"view {i} depth"
        close = np.isclose(gv.color[i].cpu().numpy(), col, rtol=FORWARD_RTOL, atol=1e-6)
        assert 1.0 - close.mean() <= FORWARD_FLIP_FRACTION
        assert (vis >= 0).any()


def test_forward_visibility_raster_equals_in_order_raster(api):
    """The differentiable forward through the visibility raster (winner per pixel by atomic max,
    shaded once) writes the same float colours, visibility ids and depths, bit for bit, as the
    in-order tile walk, for every tile shape.  The canvases hold other values before each
    forward, so that the fill of the undrawn pixels (a kernel of its own, or the visibility
    raster's write-back on 32-pixel-wide tiles) is compared too."""
    views = small_views()
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    mul = torch.from_numpy((1.0 + 0.3 * S.Rng(10).uniform(views[0].points.shape[0] * 3, -1, 1)).reshape(-1, 3)
                           .astype(np.float32)).cuda()
    out = []
    for tile_config in (0, 1, 2):
        for path in (0, 1):
            gv = api.GpuViews(views)
            for i in range(len(views)):
                gv.color[i].fill_(7.0)
                gv.visibility[i].fill_(12345)
                gv.depth[i].fill_(3.0)
            r = api.DiffRenderer()
            r.forward(gv.model, gv.views, tex, mul, api.tuning(clear=True, raster_path=path, tile_config=tile_config))
            torch.cuda.synchronize()
            out.append([(gv.color[i].cpu().numpy(), gv.visibility[i].cpu().numpy(), gv.depth[i].cpu().numpy())
                        for i in range(len(views))])
    for k in range(1, len(out)):
        for i in range(len(views)):
            for a, b in zip(out[0][i], out[k][i]):
                assert np.array_equal(a.view(np.uint32) if a.dtype == np.float32 else a,
                                      b.view(np.uint32) if b.dtype == np.float32 else b), f"run {k} view {i}"


def test_forward_on_odd_heights_equals_in_order_raster(api):
    """The same equality on canvases of odd height, whose last row the visibility raster walks in
    submission order."""
    views = S.sphere_views(6, 2, 75, 45, seed=8)
    for v in views:  # near enough that the object reaches the last row
        v.cam_location = S.look_at(np.asarray(v.cam_location[:3], np.float64) * 0.55)
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    out = []
    for tile_config in (0, 1, 2):
        for path in (0, 1):
            gv = api.GpuViews(views)
            r = api.DiffRenderer()
            r.forward(gv.model, gv.views, tex, None, api.tuning(clear=True, raster_path=path, tile_config=tile_config))
            torch.cuda.synchronize()
            out.append([(gv.color[i].cpu().numpy(), gv.visibility[i].cpu().numpy(), gv.depth[i].cpu().numpy())
                        for i in range(len(views))])
    assert all((o[1][-1] >= 0).any() for o in out[0])
    for k in range(1, len(out)):
        for i in range(len(views)):
            for a, b in zip(out[0][i], out[k][i]):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"run {k} view {i}"


def test_adjoint_of_kept_and_changed_visibility(api):
    """The adjoint takes a pixel's weights from the forward's record only where the pixel still shows what
    that forward drew there, and derives them again otherwise.  Masked pixels are left out; two pixels of
    one quad that trade their ids and gradients, and canvases kept from an earlier forward (not cleared,
    so that the second forward draws nothing), give the gradients they gave before.  Sums of some 10^4
    single-precision terms in any order differ by about 1e-6 of their norm; the bound is 2e-5."""
    views = small_views()
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    gv = api.GpuViews(views)
    for i, g in enumerate(gv.grad):
        g.copy_(torch.from_numpy(S.Rng(100 + i).uniform(g.numel(), -1.0, 1.0).reshape(tuple(g.shape))))
    r = api.DiffRenderer()

    def adjoint():
        gt, gm = torch.zeros_like(tex), torch.zeros((gv.point_count, 3), device="cuda")
        r.backward(gt, gm)
        torch.cuda.synchronize()
        return gt.cpu().double(), gm.cpu().double()

    def assert_close(got, want, what):
        for a, b in zip(got, want):
            assert float((a - b).norm()) <= 2e-5 * float(b.norm()), what

    for path in (0, 1):
        r.forward(gv.model, gv.views, tex, None, api.tuning(clear=True, raster_path=path))
        base = adjoint()
        vis, grad = [v.clone() for v in gv.visibility], [g.clone() for g in gv.grad]
        swapped = 0
        for v, g in zip(gv.visibility, gv.grad):  # columns 2k and 2k + 1 of one command
            left, right = v[:, 0::2].clone(), v[:, 1::2].clone()
            trade = (left >= 0) & (right >= 0) & ((left >> 2) == (right >> 2))
            v[:, 0::2], v[:, 1::2] = torch.where(trade, right, left), torch.where(trade, left, right)
            gl, gr = g[:, 0::2].clone(), g[:, 1::2].clone()
            g[:, 0::2], g[:, 1::2] = torch.where(trade[..., None], gr, gl), torch.where(trade[..., None], gl, gr)
            swapped += int(trade.sum())
        assert swapped > 1000
        assert_close(adjoint(), base, "traded ids")
        for i, v in enumerate(gv.visibility):
            v.copy_(vis[i])
            gv.grad[i].copy_(grad[i])
            v[::3, ::2] = -1
        masked = adjoint()
        for i, v in enumerate(gv.visibility):
            v.copy_(vis[i])
            gv.grad[i][::3, ::2] = 0.0
        assert_close(masked, adjoint(), "masked pixels")
        for i, g in enumerate(gv.grad):
            g.copy_(grad[i])
        r.forward(gv.model, gv.views, tex, None, api.tuning(raster_path=path))
        assert all(torch.equal(a, b) for a, b in zip(vis, gv.visibility))
        assert_close(adjoint(), base, "kept canvases")


def test_views_after_a_refused_forward(api):
    """A forward that is refused for its first view leaves nothing behind: the views drawn before it are
    drawn again by the next one."""
    gv = api.GpuViews(small_views())
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    r = api.DiffRenderer()
    t = api.tuning(clear=True)
    print("[gpu] forward after a refused one", flush=True)
    r.forward(gv.model, gv.views, tex, None, t)
    want = [v.clone() for v in gv.visibility]
    refused = (api.View * 1)(gv.views[0])
    refused[0].width = 0
    with pytest.raises(api.DfpsrError):
        r.forward(gv.model, refused, tex, None, t)
    for v in gv.visibility:
        v.fill_(-1)
    r.forward(gv.model, gv.views, tex, None, t)
    torch.cuda.synchronize()
    for v, w in zip(gv.visibility, want):
        assert torch.equal(v, w) and bool((w >= 0).any())


@pytest.mark.parametrize("tile_config", [0, 1])
def test_views_that_see_nothing(api, tile_config):
    """A forward whose views all turned away still clears them, and its adjoint adds nothing, also after a
    forward that drew."""
    views = small_views()[:2]
    gv = api.GpuViews(views)
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    for g in gv.grad:
        g.fill_(1.0)
    r = api.DiffRenderer()
    print("[gpu] views that see nothing", flush=True)
    r.forward(gv.model, gv.views, tex, None, api.tuning(clear=True, tile_config=tile_config))
    assert all(bool((v >= 0).any()) for v in gv.visibility)
    for i, sc in enumerate(views):
        position = np.asarray(sc.cam_location[:3], np.float64)
        gv.views[i].camera = api.camera_create(True, S.look_at(position, position * 2.0), sc.width, sc.height, sc.width_slope)
    r.forward(gv.model, gv.views, tex, None, api.tuning(clear=True, clear_depth=0.25, tile_config=tile_config))
    gt = torch.zeros_like(tex)
    r.backward(gt, None)
    torch.cuda.synchronize()
    assert not bool(gt.any())
    for i in range(len(views)):
        assert bool((gv.visibility[i] == -1).all()) and not bool(gv.color[i].any()) and bool((gv.depth[i] == 0.25).all())


def test_adjoint_of_ids_that_name_no_command(api):
    """Canvases kept from an earlier forward whose view the last one draws nothing in (turned away), and ids
    past the last command: their pixels are left out, and the other view's gradients are what it gives
    alone.  The bound is that of test_adjoint_of_kept_and_changed_visibility."""
    views = small_views()[:2]
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    gv = api.GpuViews(views)
    for i, g in enumerate(gv.grad):
        g.copy_(torch.from_numpy(S.Rng(200 + i).uniform(g.numel(), -1.0, 1.0).reshape(tuple(g.shape))))
    r = api.DiffRenderer()

    def adjoint(renderer):
        gt, gm = torch.zeros_like(tex), torch.zeros((gv.point_count, 3), device="cuda")
        renderer.backward(gt, gm)
        torch.cuda.synchronize()
        return gt.cpu().double(), gm.cpu().double()

    def assert_close(got, want):
        for a, b in zip(got, want):
            assert float((a - b).norm()) <= 2e-5 * float(b.norm())

    print("[gpu] ids that name no command", flush=True)
    alone = (api.View * 1)(gv.views[0])
    r.forward(gv.model, alone, tex, None, api.tuning(clear=True))
    want = adjoint(r)
    r.forward(gv.model, gv.views, tex, None, api.tuning(clear=True))
    kept = gv.visibility[1].clone()
    assert int((kept >= 0).sum()) > 1000
    position = np.asarray(views[1].cam_location[:3], np.float64)
    gv.views[1].camera = api.camera_create(True, S.look_at(position, position * 2.0), views[1].width, views[1].height, views[1].width_slope)
    r.forward(gv.model, gv.views, tex, None, api.tuning())
    assert torch.equal(gv.visibility[1], kept)
    assert_close(adjoint(r), want)
    for far in (0x7FFFFFFF, 4 * int(r.stats()[0])):
        r.forward(gv.model, alone, tex, None, api.tuning(clear=True))
        gv.visibility[0][gv.visibility[0] < 0] = far
        assert_close(adjoint(r), want)


def test_adjoint_without_memory_for_records(api):
    """Views with more pixels than the card has room for records of (1,250 of 4096x4096 that see nothing
    and share their buffers): the forward draws, and its adjoint, which derives every weight, adds what the
    visible view alone gives with records.  The next forward on the same object, without those views, keeps
    records again.  The bound is that of test_adjoint_of_kept_and_changed_visibility."""
    seen = small_views()[:1]
    tex = torch.from_numpy(S.float_texture(64, 5)).cuda()
    gv = api.GpuViews(seen)
    gv.grad[0].copy_(torch.from_numpy(S.Rng(9).uniform(gv.grad[0].numel(), -1.0, 1.0).reshape(tuple(gv.grad[0].shape))))
    side, count = 4096, 1250
    assert count * side * side * 16 > torch.cuda.mem_get_info()[1]
    color, grad = (torch.zeros((side, side, 4), device="cuda") for _ in range(2))
    depth, vis = torch.zeros((side, side), device="cuda"), torch.full((side, side), -1, dtype=torch.int32, device="cuda")
    position = np.asarray(seen[0].cam_location[:3], np.float64)
    views = (api.View * (1 + count))()
    views[0] = gv.views[0]
    for i in range(1, count + 1):
        v = views[i]
        v.color, v.visibility, v.depth, v.grad_color = color.data_ptr(), vis.data_ptr(), depth.data_ptr(), grad.data_ptr()
        v.width, v.height, v.stride_pixels = side, side, side
        v.transform[:] = list(gv.views[0].transform)
        v.camera = api.camera_create(True, S.look_at(position, position * 2.0), side, side, seen[0].width_slope)
    t = api.tuning(tile_config=2, persistent_per_cu=4)

    def adjoint(renderer, which):
        gv.visibility[0].fill_(-1)
        gv.depth[0].zero_()
        renderer.forward(gv.model, which, tex, None, t)
        gt, gm = torch.zeros_like(tex), torch.zeros((gv.point_count, 3), device="cuda")
        renderer.backward(gt, gm, t)
        torch.cuda.synchronize()
        return gt.cpu().double(), gm.cpu().double()

    print(f"[gpu] no room for records {count} x {side}^2", flush=True)
    r = api.DiffRenderer()
    want = adjoint(api.DiffRenderer(), gv.views)
    assert float(want[0].norm()) > 0.0 and float(want[1].norm()) > 0.0
    for which in (views, gv.views):
        for a, b in zip(adjoint(r, which), want):
            assert float((a - b).norm()) <= 2e-5 * float(b.norm())
    assert int((vis >= 0).sum()) == 0


def test_adjoint_same_for_every_tile_shape(api):
    """The adjoint walks whatever tiles the forward used: texture and multiplier gradients agree
    across tile shapes up to the order of the float atomics."""
    views = small_views()
    tex = torch.from_numpy(S.float_texture(64, 6)).cuda()
    mul = torch.from_numpy((1.0 + 0.3 * S.Rng(11).uniform(views[0].points.shape[0] * 3, -1, 1)).reshape(-1, 3)
                           .astype(np.float32)).cuda()
    rng = np.random.default_rng(5)
    grads = [torch.from_numpy(rng.standard_normal((v.height, v.width, 4)).astype(np.float32)) for v in views]
    results = []
    for tile_config in (0, 1, 2):
        gv = api.GpuViews(views)
        for g, buf in zip(grads, gv.grad):
            buf.copy_(g)
        r = api.DiffRenderer()
        r.forward(gv.model, gv.views, tex, mul, api.tuning(clear=True, tile_config=tile_config))
        gt, gm = torch.zeros_like(tex), torch.zeros_like(mul)
        r.backward(gt, gm, api.tuning())
        torch.cuda.synchronize()
        results.append((gt.cpu().numpy().astype(np.float64), gm.cpu().numpy().astype(np.float64)))
    for gt, gm in results[1:]:
        assert np.linalg.norm(gt - results[0][0]) <= 1e-5 * np.linalg.norm(results[0][0])
        assert np.linalg.norm(gm - results[0][1]) <= 1e-5 * np.linalg.norm(results[0][1])


def test_adjoint_matches_oracle_and_dot_product(api):
    views = small_views()
    gv = api.GpuViews(views)
    tex = S.float_texture(64, 2)
    mul = (1.0 + 0.3 * S.Rng(9).uniform(views[0].points.shape[0] * 3, -1, 1)).reshape(-1, 3).astype(np.float32)
    r = api.DiffRenderer()
    tex_d, mul_d = torch.from_numpy(tex).cuda(), torch.from_numpy(mul).cuda()
    r.forward(gv.model, gv.views, tex_d, mul_d, api.tuning(clear=True))
    rng = np.random.default_rng(3)
    grads = [rng.standard_normal((v.height, v.width, 4)).astype(np.float32) for v in views]
    for g, buf in zip(grads, gv.grad):
        buf.copy_(torch.from_numpy(g))
    gt = torch.zeros_like(tex_d)
    gm = torch.zeros_like(mul_d)
    r.backward(gt, gm, api.tuning())
    torch.cuda.synchronize()
    ref_t = np.zeros(tex.shape)
    ref_m = np.zeros(mul.shape)
    dot = 0.0
    for i, sc in enumerate(views):
        col, vis, dep, w = H.oracle_diff_forward(sc, tex, mul)
        a, b = H.oracle_diff_backward(sc, tex, mul, vis, w, grads[i], mul.shape[0])
        ref_t += a
        ref_m += b
        dot += float((grads[i].astype(np.float64) * gv.color[i].cpu().numpy()).sum())
    got_t, got_m = gt.cpu().numpy().astype(np.float64), gm.cpu().numpy().astype(np.float64)
    # Relative L2 error: the few pixels whose sub-texel weights flip (see the forward test) move
    # a little gradient between neighbouring texels.
    assert np.linalg.norm(got_t - ref_t) <= ADJOINT_RTOL * np.linalg.norm(ref_t)
    assert np.linalg.norm(got_m - ref_m) <= ADJOINT_RTOL * np.linalg.norm(ref_m)
    # Dot-product identities: colour is linear in the texture, and its RGB in the multipliers.
    assert abs(dot - float((got_t * tex).sum())) <= 1e-4 * abs(dot)
    dot_rgb = sum(float((grads[i][..., :3].astype(np.float64) * gv.color[i].cpu().numpy()[..., :3]).sum())
                  for i in range(len(views)))
    assert abs(dot_rgb - float((got_m * mul).sum())) <= 1e-4 * abs(dot_rgb)


def test_adjoint_matches_oracle_on_ragged_canvases(api):
    """Canvases of odd width and of height that is no multiple of the tile height: the pixel
    pairs at the right edge hold one pixel only, and edge tiles hold partial rows.  Every tile
    shape's adjoint meets the oracle's bar."""
    views = S.sphere_views(12, 2, 203, 118, seed=6, radius=1.8)  # the sphere fills the edge columns and rows
    tex = S.float_texture(64, 8)
    mul = (1.0 + 0.3 * S.Rng(12).uniform(views[0].points.shape[0] * 3, -1, 1)).reshape(-1, 3).astype(np.float32)
    rng = np.random.default_rng(8)
    grads = [rng.standard_normal((v.height, v.width, 4)).astype(np.float32) for v in views]
    ref_t = np.zeros(tex.shape)
    ref_m = np.zeros(mul.shape)
    for i, sc in enumerate(views):
        col, vis, dep, w = H.oracle_diff_forward(sc, tex, mul)
        a, b = H.oracle_diff_backward(sc, tex, mul, vis, w, grads[i], mul.shape[0])
        ref_t += a
        ref_m += b
    tex_d, mul_d = torch.from_numpy(tex).cuda(), torch.from_numpy(mul).cuda()
    for tile_config in (0, 1, 2):
        print(f"[gpu] ragged adjoint 203x118 tile_config {tile_config}", flush=True)
        gv = api.GpuViews(views)
        for g, buf in zip(grads, gv.grad):
            buf.copy_(torch.from_numpy(g))
        r = api.DiffRenderer()
        r.forward(gv.model, gv.views, tex_d, mul_d, api.tuning(clear=True, tile_config=tile_config))
        gt, gm = torch.zeros_like(tex_d), torch.zeros_like(mul_d)
        r.backward(gt, gm, api.tuning())
        torch.cuda.synchronize()
        got_t, got_m = gt.cpu().numpy().astype(np.float64), gm.cpu().numpy().astype(np.float64)
        assert np.linalg.norm(got_t - ref_t) <= ADJOINT_RTOL * np.linalg.norm(ref_t)
        assert np.linalg.norm(got_m - ref_m) <= ADJOINT_RTOL * np.linalg.norm(ref_m)


@pytest.fixture(scope="module")
def fit_setup(api):
    """Config 3: 8 views at 1280x720 of a 50,000-triangle displaced geodesic sphere (frequency 50),
    a 512x512 RGBA float texture and per-point RGB multipliers."""
    views = S.sphere_views(50, 8, 1280, 720, seed=3)
    gv = api.GpuViews(views)
    hidden = torch.from_numpy(S.float_texture(512, 77, smooth=16)).cuda()
    ones = torch.ones((gv.point_count, 3), dtype=torch.float32, device="cuda")
    r = api.DiffRenderer()
    t = api.tuning(clear=True, persistent_per_cu=4, use_graph=True)
    r.forward(gv.model, gv.views, hidden, ones, t)
    target = torch.stack([c.clone() for c in gv.color])
    return gv, r, t, target


def test_config3_finite_differences(api, fit_setup):
    """Texture gradients of the config-3 loss against central finite differences on 1,000
    seeded (texel, channel) pairs, h = 1e-3.  The colour is linear in the texture and
    visibility does not depend on it, so the loss is exactly quadratic along each pair: the
    only error left is float32 rounding of the rendered images.  The step is the stored
    difference of the perturbed texel values.  Every pair with a non-zero gradient must agree
    to 1e-3 relative error, with no floor; texels that no pixel samples must give exactly zero
    on both sides."""
    gv, r, t, target = fit_setup
    texture = torch.full((512, 512, 4), 0.5, dtype=torch.float32, device="cuda")
    mul = torch.ones((gv.point_count, 3), dtype=torch.float32, device="cuda")

    def render():
        r.forward(gv.model, gv.views, texture, mul, t)
        return torch.stack(gv.color).clone()

    img = render()
    for i, g in enumerate(gv.grad):
        g.copy_(2.0 * (img[i] - target[i]))
    gt = torch.zeros_like(texture)
    r.backward(gt, None, api.tuning())
    analytic = gt.cpu().numpy().reshape(-1).astype(np.float64)
    rng = np.random.default_rng(1000)
    texels = rng.integers(0, 512 * 512, 1000)
    channels = rng.integers(0, 4, 1000)
    h = 1e-3
    target64 = target.double()
    errors, zeros = [], 0
    flat = texture.view(-1)
    for tx, ch in zip(texels, channels):
        k = int(tx) * 4 + int(ch)
        flat[k] = 0.5 + h
        plus = float(flat[k].item())
        ip = render()
        flat[k] = 0.5 - h
        minus = float(flat[k].item())
        im = render()
        flat[k] = 0.5
        # L(T+h) - L(T-h) = sum (ip - im)(ip + im - 2 target): exactly zero where nothing changed.
        num = float(((ip.double() - im.double()) * (ip.double() + im.double() - 2.0 * target64)).sum())
        fd = num / (plus - minus)
        an = float(analytic[k])
        if an == 0.0:
            assert fd == 0.0, f"texel {tx} channel {ch}: no analytic gradient but a finite difference of {fd}"
            zeros += 1
            continue
        errors.append(abs(fd - an) / abs(an))
    errors = np.array(errors)
    print(f"[gpu] texel fd: max rel err {errors.max():.2e}, median {np.median(errors):.2e}, "
          f"{len(errors)} of 1000 texels sampled ({zeros} not sampled by any pixel)", flush=True)
    assert len(errors) > 100
    assert errors.max() <= FD_RTOL


def test_config3_multiplier_finite_differences(api, fit_setup):
    """Per-point RGB multiplier gradients of the config-3 loss (8 views at 1280x720, texture
    0.5, multipliers 1) against central finite differences on 1,000 seeded (point, channel)
    pairs.  The colour is linear in the multipliers and visibility does not depend on them, so
    the loss is exactly quadratic along each pair and the central difference is the
    derivative: the only error left is float32 rounding of the rendered images.  The step is
    the stored difference of the perturbed multipliers (h = 1e-3 before rounding to float32).
    Every pair with a non-zero gradient must agree to 1e-3 relative error; pairs whose point no
    view draws must give exactly zero on both sides."""
    gv, r, t, target = fit_setup
    texture = torch.full((512, 512, 4), 0.5, dtype=torch.float32, device="cuda")
    mul = torch.ones((gv.point_count, 3), dtype=torch.float32, device="cuda")

    def render():
        r.forward(gv.model, gv.views, texture, mul, t)
        return torch.stack(gv.color).clone()

    img = render()
    for i, g in enumerate(gv.grad):
        g.copy_(2.0 * (img[i] - target[i]))
    gm = torch.zeros_like(mul)
    r.backward(None, gm, api.tuning())
    analytic = gm.cpu().numpy().reshape(-1).astype(np.float64)
    rng = np.random.default_rng(2000)
    points = rng.integers(0, gv.point_count, 1000)
    channels = rng.integers(0, 3, 1000)
    h = 1e-3
    target64 = target.double()
    flat = mul.view(-1)
    errors, zeros = [], 0
    for p, ch in zip(points, channels):
        k = int(p) * 3 + int(ch)
        flat[k] = 1.0 + h
        plus = float(flat[k].item())
        ip = render()
        flat[k] = 1.0 - h
        minus = float(flat[k].item())
        im = render()
        flat[k] = 1.0
        num = float(((ip.double() - im.double()) * (ip.double() + im.double() - 2.0 * target64)).sum())
        fd = num / (plus - minus)
        an = float(analytic[k])
        if an == 0.0:
            assert fd == 0.0, f"point {p} channel {ch}: no analytic gradient but a finite difference of {fd}"
            zeros += 1
            continue
        errors.append(abs(fd - an) / abs(an))
    errors = np.array(errors)
    print(f"[gpu] multiplier fd: max rel err {errors.max():.2e}, median {np.median(errors):.2e}, "
          f"{len(errors)} of 1000 pairs drawn ({zeros} not drawn in any view)", flush=True)
    assert len(errors) > 500
    assert errors.max() <= FD_RTOL


def test_config3_adam_fit(api, fit_setup):
    gv, r, t, target = fit_setup
    texture = torch.full((512, 512, 4), 0.5, dtype=torch.float32, device="cuda", requires_grad=True)
    mul = torch.ones((gv.point_count, 3), dtype=torch.float32, device="cuda", requires_grad=True)
    opt = torch.optim.Adam([texture, mul], lr=1e-2)
    losses = []
    for step in range(200):
        opt.zero_grad()
        img = RenderFunction.apply(texture, mul, r, gv, t)
        loss = ((img - target) ** 2).sum()
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    print(f"[gpu] fit: loss {losses[0]:.2f} -> {losses[-1]:.2f}", flush=True)
    assert losses[-1] < 0.1 * losses[0]


def test_config4_batched_equals_per_view(api):
    """Config 4: 256 views of 256x256, a 20,480-triangle sphere, a shared 1024x1024 texture.
    One persistent, graph-captured launch per pass against the per-view form."""
    views = S.sphere_views(32, 256, 256, 256, seed=11)
    gv = api.GpuViews(views)
    tex = torch.from_numpy(S.float_texture(1024, 5, smooth=32)).cuda()
    rng = np.random.default_rng(4)
    for g in gv.grad:
        g.copy_(torch.from_numpy(rng.standard_normal((256, 256, 4)).astype(np.float32)))
    batched = api.DiffRenderer()
    t = api.tuning(clear=True, persistent_per_cu=4, use_graph=True)
    batched.forward(gv.model, gv.views, tex, None, t)
    images = [c.clone() for c in gv.color]
    vis = [v.clone() for v in gv.visibility]
    g_batched = torch.zeros_like(tex)
    batched.backward(g_batched, None, t)
    single = api.DiffRenderer()
    g_sum = torch.zeros_like(tex)
    for i in range(len(views)):
        one = (type(gv.views[0]) * 1)(gv.views[i])
        single.forward(gv.model, one, tex, None, api.tuning(clear=True))
        assert torch.equal(gv.color[i], images[i]), f"view {i} image"
        assert torch.equal(gv.visibility[i], vis[i]), f"view {i} visibility"
        single.backward(g_sum, None, api.tuning())
    torch.cuda.synchronize()
    diff = (g_batched - g_sum).abs().max().item()
    assert diff <= BATCHED_GRAD_RTOL * g_sum.abs().max().item()
