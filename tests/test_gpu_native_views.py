"""Views through the native host layer (one C++ call and one autograd node per render, record slots handed out by regions
of 256-surfel blocks instead of a prefix scan) against the same view on the operators: equal maps, equal gradients.
Sizes: one, around a block, around one turn of the 64 regions (16 384 surfels), ragged images."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scene(P, W, H, seed, scale=-4.2):
    from fast_sp_gs_amd import scenes
    g = torch.Generator().manual_seed(seed)
    s = scenes._surfels(g, P, 'cube', scale, 0.7, 0.0, 1.5)
    return s, scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])), g


def _leaves(device, *tensors):
    return [t.to(device).requires_grad_(True) for t in tensors]


@pytest.mark.parametrize('P,W,H,mode', [(1, 16, 16, 'sh'), (255, 49, 31, 'split'), (256, 49, 31, 'colors'),
                                        (257, 64, 48, 'culling'), (16_384, 161, 99, 'sh'), (16_385, 161, 99, 'flow'),
                                        (40_000, 250, 130, 'accum')])
def test_surfel_view_equals_operators(P, W, H, mode, device):
    from fast_sp_gs_amd.renderer import gs_2d_render as m
    s, cam_h, g = _scene(P, W, H, P + 1)
    cam = cam_h.to(device)
    params = _leaves(device, s.means3D, s.scales, s.rotations, s.opacities)
    rest = None
    if mode == 'split':
        sh, rest = _leaves(device, s.shs[:, :1].contiguous(), s.shs[:, 1:].contiguous())
    elif mode == 'colors':
        sh, = _leaves(device, s.shs[:, 0].contiguous())
    else:
        sh, = _leaves(device, s.shs)
    culling = (torch.rand(P, generator=g) < 0.3).to(device) if mode == 'culling' else None
    t2 = torch.randn(P, 3, 3, generator=g).to(device) if mode == 'flow' else None
    accum = lambda: ([torch.zeros(P, dtype=torch.int32, device=device), torch.zeros(P, device=device),
                      torch.zeros(P, dtype=torch.int32, device=device)] if mode == 'accum' else [None] * 3)
    a1, a2 = accum(), accum()
    out = m.GS_2D_render(*params, (W, H), cam.Tw2v, cam.Tv2c, campos=cam.campos, sh_degree=3, near=0.2, far=100.0,
                         colors=sh if mode == 'colors' else None, sh_features=None if mode == 'colors' else sh,
                         sh_features_rest=rest, culling=culling, trans_mat_t2=t2, accum_max_count=a1[0],
                         accum_weights_p=a1[1], accum_weights_count=a1[2])
    m2 = torch.zeros(P, 2, device=device, requires_grad=True)
    img, opac, extras, flow, n_contrib, radii, buf = m._GS_2D_Render.apply(
        *params, sh, rest, cam.Tw2v, cam.Tv2c, cam.campos, (W, H), -1 if mode == 'colors' else 3, False, 0.2, 100.0, False,
        None, m2, t2, culling, *a2)
    same = lambda a, b: a.shape == b.shape and torch.equal(a, b)
    assert same(out['images'], img) and same(out['opacity'], opac) and same(out['distortion'], extras[5:6])
    assert same(out['radii'], radii) and same(out['visibility_filter'], radii > 0)
    assert same(out['depths'], torch.nan_to_num(extras[4:5], 0, 0))
    assert same(out['viewspace_points'], m2) and same(out['buffer'].n_contribed, n_contrib)
    assert same(out['buffer'].tile_ranges, buf.tile_ranges) and out['buffer'].R == buf.R
    used = int((buf.tile_ranges[:, 1] - buf.tile_ranges[:, 0]).sum())
    assert torch.equal(out['buffer'].point_list[:used], buf.point_list[:used])
    for x, y in zip(a1[::2], a2[::2]):
        assert x is None or torch.equal(x, y)
    g_img, g_op, g_dist = (torch.randn(t.shape, generator=g).to(device) for t in (img, opac, extras[5:6]))
    wrt = params + [sh] + ([rest] if rest is not None else [])
    maps, ups = [out['images'], out['opacity'], out['distortion']], [g_img, g_op, g_dist]
    o_maps = [img, opac, extras[5:6]]
    if mode == 'flow':
        assert same(out['flow'], flow)
        g_flow = torch.randn(flow.shape, generator=g).to(device) * (flow.abs() < 1e3)
        maps, o_maps, ups = maps + [out['flow']], o_maps + [flow], ups + [g_flow]
    got = torch.autograd.grad(maps, wrt + [out['viewspace_points']], ups, allow_unused=True)
    want = torch.autograd.grad(o_maps, wrt + [m2], ups, allow_unused=True)
    for x, y in zip(got, want):
        assert (x is None) == (y is None) and (x is None or torch.equal(torch.nan_to_num(x), torch.nan_to_num(y)))


def test_surfel_views_on_two_streams_and_threads(device):
    """Views of two host threads on two streams at once give what they give alone (counters are per stream and call)."""
    import threading

    from fast_sp_gs_amd.renderer import GS_2D_render
    jobs = []
    for k, P in enumerate((3_000, 9_000)):
        s, cam_h, _ = _scene(P, 200, 120, k)
        jobs.append((s.to(device), cam_h.to(device)))

    def view(job):
        s, cam = job
        with torch.no_grad():
            return GS_2D_render(s.means3D, s.scales, s.rotations, s.opacities, (cam.W, cam.H), cam.Tw2v, cam.Tv2c,
                                campos=cam.campos, sh_degree=3, sh_features=s.shs)['images']

    want = [view(j) for j in jobs]
    torch.cuda.synchronize()
    bad = []

    def loop(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                if not torch.equal(view(jobs[k]), want[k]):
                    bad.append(k)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=loop, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize('P,W,H,mode', [(1, 16, 16, 'sh'), (257, 49, 31, 'split'), (256, 64, 48, 'colors'),
                                        (300, 49, 31, 'partial'), (16_385, 161, 99, 'culling'), (20_000, 250, 130, 'flow')])
def test_fast_surfel_view_equals_operators(P, W, H, mode, device):
    """The fused tail's maps to the rounding of its 3x3 inverses; everything else bit for bit."""
    from fast_sp_gs_amd.renderer import gs_2d_fast_render as m
    from fast_sp_gs_amd.renderer.gs_2d_render import depth_to_normal
    s, cam_h, g = _scene(P, W, H, P + 2)
    cam = cam_h.to(device)
    params = _leaves(device, s.means3D, s.scales, s.rotations, s.opacities)
    rest, degree = None, 2 if mode == 'partial' else 3
    if mode == 'split':
        sh, rest = _leaves(device, s.shs[:, :1].contiguous(), s.shs[:, 1:].contiguous())
    else:
        sh, = _leaves(device, s.shs[:, 0].contiguous() if mode == 'colors' else s.shs)
    culling = (torch.rand(P, generator=g) < 0.3).to(device) if mode == 'culling' else None
    t2 = torch.randn(P, 3, 3, generator=g).to(device) if mode == 'flow' else None
    out = m.GS_2D_fast_render(*params, (W, H), cam.Tw2v, cam.Tv2c, cam.Tv2s, campos=cam.campos, sh_degree=degree,
                              colors=sh if mode == 'colors' else None, sh_features=None if mode == 'colors' else sh,
                              sh_features_rest=rest, culling=culling, trans_mat_t2=t2)
    m2 = torch.zeros(P, 2, device=device, requires_grad=True)
    img, opac, extras, flow, n_contrib, radii = m._Fast_Render.apply(
        *params, sh, rest, cam.Tw2v, cam.Tv2c, cam.Tv2s, cam.campos, (W, H), -1 if mode == 'colors' else degree, False, 0.2,
        100.0, False, None, m2, t2, culling, None, None, None)
    depth = torch.nan_to_num(extras[4:5], 0, 0)  # depth_ratio = 1
    normals = (extras[1:4].permute(1, 2, 0) @ cam.Tw2v[:3, :3]).permute(2, 0, 1)
    surf_normal = depth_to_normal(cam.Tw2v, cam.Tv2c, (W, H), depth).permute(2, 0, 1) * opac.detach()
    same = lambda a, b: a.shape == b.shape and torch.equal(a, b)
    assert same(out['images'], img) and same(out['opacity'], opac) and same(out['distortion'], extras[5:6])
    assert same(out['radii'], radii) and same(out['visibility_filter'], radii > 0)
    assert same(out['viewspace_points'], m2) and same(out['surf_depth'], depth)
    assert torch.allclose(out['normals'], normals, atol=1e-6)
    assert (out['surf_normal'] - surf_normal).norm() <= 2e-3 * surf_normal.norm() + 1e-6
    assert (out['flows'] is None and flow is None) or same(out['flows'], flow)
    up = [torch.randn(t.shape, generator=g).to(device) for t in (img, opac, extras[5:6], normals, depth)]
    wanted = params + [sh] + ([rest] if rest is not None else [])
    got = torch.autograd.grad([out[k] for k in ('images', 'opacity', 'distortion', 'normals', 'surf_depth')] +
                              ([out['flows']] if flow is not None else []), wanted + [out['viewspace_points']],
                              up + ([torch.ones_like(flow)] if flow is not None else []))
    ref = torch.autograd.grad([img, opac, extras[5:6], normals, depth] + ([flow] if flow is not None else []), wanted + [m2],
                              up + ([torch.ones_like(flow)] if flow is not None else []))
    for a, b in zip(got, ref):
        assert (a - b).norm() <= 1e-5 * b.norm() + 1e-7


@pytest.mark.parametrize('P,W,H,mode', [(1, 16, 16, 'sh'), (257, 49, 31, 'split'), (256, 64, 48, 'colors'),
                                        (300, 49, 31, 'extras'), (16_385, 161, 99, 'culling'), (3_000, 120, 90, 'opengl'),
                                        (3_000, 120, 90, 'later')])
def test_gaussian_view_equals_operators(P, W, H, mode, device):
    """Maps bit for bit; gradients to the order of the sums over a Gaussian's tiles. 'later': a further table blended with
    the view's weights, whose gradient reaches the geometry through the buffer."""
    import math

    from fast_sp_gs_amd.renderer import gaussian_render as m
    s, cam_h, g = _scene(P, W, H, P + 3)
    cam = cam_h.to(device)
    third = torch.exp(torch.randn(P, 1, generator=g) * 0.5 - 4.2)
    params = _leaves(device, s.means3D, torch.cat([s.scales, third], dim=1), s.rotations, s.opacities)
    rest = extras = table = None
    if mode == 'split':
        sh, rest = _leaves(device, s.shs[:, :1].contiguous(), s.shs[:, 1:].contiguous())
    else:
        sh, = _leaves(device, s.shs[:, 0].contiguous() if mode == 'colors' else s.shs)
    if mode == 'extras':
        extras, = _leaves(device, torch.randn(P, 3, generator=g))
    if mode == 'later':
        table, = _leaves(device, torch.randn(P, 6, generator=g))
    culling = (torch.rand(P, generator=g) < 0.3).to(device) if mode == 'culling' else None
    tan = (math.tan(math.radians(25.0)), math.tan(math.radians(25.0)) * H / W)
    out = m.render(cam.Tw2v, cam.Tv2c, (W, H), params[0], params[3], params[1], params[2], campos=cam.campos,
                   FoV=tuple(2 * math.atan(t) for t in tan), sh_degree=3, is_opengl=mode == 'opengl', culling=culling,
                   colors=sh if mode == 'colors' else None, sh_features=None if mode == 'colors' else sh,
                   sh_features_rest=rest, **({} if extras is None else {'feature': extras}))
    m2 = torch.zeros(P, 2, device=device, requires_grad=True)
    img, opac, maps, radii, buf, visible = m._rasterize_operators(
        params[0], m2, sh, rest, params[3], params[1], params[2], None, None, extras, (W, H), -1 if mode == 'colors' else 3,
        cam.Tw2v, cam.Tv2c, cam.campos, tan, mode == 'opengl', culling, None, None, None)
    same = lambda a, b: a.shape == b.shape and torch.equal(a, b)
    assert same(out['images'], img) and same(out['opacity'], opac) and same(out['radii'], radii)
    assert same(out['visibility_filter'], visible) and same(out['viewspace_points'], m2)
    assert same(out['buffer'].conic_opacity, buf.conic_opacity) and same(out['buffer'].n_contribed, buf.n_contribed)
    got_maps, ref_maps = [out['images'], out['opacity']], [img, opac]
    wanted = params + [sh] + [t for t in (rest, extras, table) if t is not None]
    if extras is not None:
        assert same(out['feature'], maps)
        got_maps, ref_maps = got_maps + [out['feature']], ref_maps + [maps]
    if table is not None:
        got_maps, ref_maps = got_maps + [m.render_extra(out['buffer'], table)], ref_maps + [m.render_extra(buf, table)]
    up = [torch.randn(t.shape, generator=g).to(device) for t in got_maps]
    got = torch.autograd.grad(got_maps, wanted + [out['viewspace_points']], up)
    ref = torch.autograd.grad(ref_maps, wanted + [m2], up)
    for a, b in zip(got, ref):
        assert (a - b).norm() <= 1e-4 * b.norm() + 1e-7


@pytest.mark.parametrize('split', [False, True])
@pytest.mark.parametrize('table', [False, True])
@pytest.mark.parametrize('given', ['cov3D', 'cov2D'])
def test_gaussian_view_with_given_covariance(given, split, table, device):
    """Pre-computed covariances with and without the optional inputs in front of and behind them, through `.backward()` and
    as the only gradient asked for, with the caller's screen positions and without."""
    import math

    from fast_sp_gs_amd.renderer import gaussian_render as m
    P, W, H = 300, 49, 31
    s, cam_h, g = _scene(P, W, H, 7)
    cam = cam_h.to(device)
    third = torch.exp(torch.randn(P, 1, generator=g) * 0.5 - 4.2)
    means, scales, rot, opac = _leaves(device, s.means3D, torch.cat([s.scales, third], dim=1), s.rotations, s.opacities)
    tan = (math.tan(math.radians(25.0)), math.tan(math.radians(25.0)) * H / W)
    cov = m.compute_cov3D(scales, rot).detach()
    if given == 'cov2D':
        cov = m.compute_cov2D(means, cov, cam.Tw2v, W / (2 * tan[0]), H / (2 * tan[1]), *tan).detach()
    cov.requires_grad_(True)
    sh, rest = (_leaves(device, s.shs[:, :1].contiguous(), s.shs[:, 1:].contiguous()) if split else
                (*_leaves(device, s.shs), None))
    extras = _leaves(device, torch.randn(P, 3, generator=g))[0] if table else None
    args = (sh, rest, opac, scales, rot, *((cov, None) if given == 'cov3D' else (None, cov)), extras, (W, H), 3, cam.Tw2v,
            cam.Tv2c, cam.campos, tan, False, None, None, None, None)
    up = [torch.randn(n, H, W, generator=g).to(device) for n in (3, 1, 3)]
    loss = lambda o: (o[0] * up[0]).sum() + (o[1] * up[1]).sum() + ((o[2] * up[2]).sum() if table else 0)
    screen = lambda: torch.zeros(P, 2, device=device, requires_grad=True)
    wanted = [cov, means, opac, sh] + ([rest] if split else []) + ([extras] if table else [])
    want = torch.autograd.grad(loss(m._rasterize_operators(means, screen(), *args)), wanted)
    for m2 in (screen(), None):
        value = loss(m.RasterizeGaussians(means, m2, *args))
        alone, = torch.autograd.grad(value, [cov], retain_graph=True)
        value.backward()
        for t, w in zip([alone] + [t.grad for t in wanted], [want[0], *want]):
            assert t is not None and (t - w).norm() <= 1e-4 * w.norm() + 1e-7
        assert scales.grad is None and rot.grad is None
        for t in wanted:
            t.grad = None


@pytest.mark.parametrize('split', [False, True])
@pytest.mark.parametrize('view', ['surfel', 'fast_surfel', 'gaussian'])
def test_colours_of_a_wrong_shape_are_refused(view, split, device):
    """On the host, before anything is launched: pre-computed colours beside a table of further coefficients or not, and
    fewer first coefficients than points beside such a table."""
    from fast_sp_gs_amd.renderer import GS_2D_render
    from fast_sp_gs_amd.renderer.gaussian_render import render
    from fast_sp_gs_amd.renderer.gs_2d_fast_render import GS_2D_fast_render
    P, W, H = 300, 49, 31
    s, cam_h, _ = _scene(P, W, H, 7)
    s, cam = s.to(device), cam_h.to(device)
    rest = s.shs[:, 1:].contiguous() if split else None

    def picture(**kw):
        kw.update(campos=cam.campos, sh_degree=3, sh_features_rest=rest)
        if view == 'gaussian':
            scales = torch.cat([s.scales, s.scales[:, :1]], dim=1)
            return render(cam.Tw2v, cam.Tv2c, (W, H), s.means3D, s.opacities, scales, s.rotations, FoV=(0.8, 0.6), **kw)
        args = (s.means3D, s.scales, s.rotations, s.opacities, (W, H), cam.Tw2v, cam.Tv2c)
        return GS_2D_render(*args, **kw) if view == 'surfel' else GS_2D_fast_render(*args, cam.Tv2s, **kw)

    for shape in ((P - 1, 3), (P + 1, 3), (P, 4), (P, 1, 3), (3 * P,)):
        with pytest.raises(RuntimeError, match='shs must have shape'):
            picture(colors=torch.zeros(shape, device=device))
    if split:
        with pytest.raises(RuntimeError, match='Error shape for sh features'):
            picture(sh_features=s.shs[1:, :1].contiguous())
        assert torch.isfinite(picture(sh_features=s.shs[:, :1].contiguous())['images']).all()
    assert torch.isfinite(picture(colors=torch.zeros(P, 3, device=device))['images']).all()


def _tail_in_double(Tw2v, Tv2c, size, extras, opacity, depth_ratio):
    """normals, depths, surf_depth, surf_normal of the blend's maps in 64 bits, and per pixel how far single precision
    throws the pseudo normal: the points p carry about eight roundings each, the unit normal of the differences a and b
    turns by their error times (|a| + |b|) / |a x b|."""
    Tw2v, Tv2c, (W, H) = Tw2v.double(), Tv2c.double(), size
    pixels = torch.tensor([[W / 2, 0, 0, W / 2], [0, H / 2, 0, H / 2], [0, 0, 0, 1]], dtype=torch.float64, device=Tw2v.device)
    y, x = torch.meshgrid(torch.arange(H, device=Tw2v.device), torch.arange(W, device=Tw2v.device), indexing='ij')
    at = torch.stack([x, y, torch.ones_like(x)], dim=-1).double()
    rays = at @ ((pixels @ Tv2c)[:, :3].inverse().T @ Tw2v[:3, :3].inverse().T)
    normals = (extras[1:4].permute(1, 2, 0) @ Tw2v[:3, :3]).permute(2, 0, 1)
    depths, median = torch.nan_to_num(extras[0:1], 0, 0), torch.nan_to_num(extras[4:5], 0, 0)
    surf_depth = depths * (1 - depth_ratio) + depth_ratio * median
    p = surf_depth.reshape(H, W, 1) * rays + Tw2v.inverse()[:3, 3]
    a, b = p[2:, 1:-1] - p[:-2, 1:-1], p[1:-1, 2:] - p[1:-1, :-2]
    c = torch.cross(a, b, dim=-1)
    surf_normal = torch.nn.functional.pad(torch.nn.functional.normalize(c, dim=-1).permute(2, 0, 1), (1, 1, 1, 1))
    far = p.norm(dim=-1)
    far = torch.stack([far[2:, 1:-1], far[:-2, 1:-1], far[1:-1, 2:], far[1:-1, :-2]]).amax(0)
    turn = 8 * 2.0 ** -24 * far * (a.norm(dim=-1) + b.norm(dim=-1)) / c.norm(dim=-1)
    turn = torch.nn.functional.pad(torch.nan_to_num(turn.detach(), nan=1.0, posinf=1.0), (1, 1, 1, 1), value=0.0)
    return normals, median, surf_depth, surf_normal * opacity, turn


@pytest.mark.parametrize('P,W,H,mode', [(1, 16, 16, 'sh'), (257, 49, 31, 'split'), (256, 64, 48, 'colors'),
                                        (300, 49, 31, 'partial'), (3_000, 161, 99, 'culling'), (4_000, 120, 90, 'ratio')])
@pytest.mark.parametrize('view', ['surfel', 'fast_surfel'])
def test_surfel_tails_against_double(view, P, W, H, mode, device):
    """Surfels of several pixels, so that the small pictures are covered too. Every map of the fused tail and the gradients
    of all of them together, surf_normal among them, against the tail in 64 bits around the operators."""
    from fast_sp_gs_amd.renderer import gs_2d_fast_render, gs_2d_render
    s, cam_h, g = _scene(P, W, H, P + 4, scale=-2.0 if P < 1000 else -3.0)
    cam = cam_h.to(device)
    params = _leaves(device, s.means3D, s.scales, s.rotations, s.opacities)
    rest, degree, ratio = None, 2 if mode == 'partial' else 3, 0.25 if mode == 'ratio' else 1.0
    if mode == 'split':
        sh, rest = _leaves(device, s.shs[:, :1].contiguous(), s.shs[:, 1:].contiguous())
    else:
        sh, = _leaves(device, s.shs[:, 0].contiguous() if mode == 'colors' else s.shs)
    culling = (torch.rand(P, generator=g) < 0.3).to(device) if mode == 'culling' else None
    kw = dict(campos=cam.campos, sh_degree=degree, colors=sh if mode == 'colors' else None,
              sh_features=None if mode == 'colors' else sh, sh_features_rest=rest, culling=culling, depth_ratio=ratio)
    m2, size, cams = torch.zeros(P, 2, device=device, requires_grad=True), (W, H), (cam.Tw2v, cam.Tv2c)
    drawn = (cam.campos, size, -1 if mode == 'colors' else degree, False, 0.2, 100.0, False, None, m2, None, culling, None, None,
             None)
    background = None
    if view == 'surfel':
        background = torch.rand(3, generator=g).to(device)
        out = gs_2d_render.GS_2D_render(*params, size, *cams, background=background, **kw)
        img, opac, extras, *_ = gs_2d_render._GS_2D_Render.apply(*params, sh, rest, *cams, *drawn)
    else:
        out = gs_2d_fast_render.GS_2D_fast_render(*params, size, *cams, cam.Tv2s, **kw)
        img, opac, extras, *_ = gs_2d_fast_render._Fast_Render.apply(*params, sh, rest, *cams, cam.Tv2s, *drawn)
    assert mode == 'sh' or float((opac > 0.1).float().mean()) > 0.2

    maps64 = extras.detach().double().requires_grad_(True)
    normals, median, surf_depth, surf_normal, turn = _tail_in_double(*cams, size, maps64, opac.detach().double(), ratio)
    for name, want in (('normals', normals), ('depths', median), ('surf_depth', surf_depth)):
        assert name not in out or torch.allclose(out[name].double(), want, rtol=1e-6, atol=1e-6), name
    steady = turn < 1e-4
    assert mode == 'sh' or float((steady & (opac > 0.1)).float().mean()) > 0.1
    off = (out['surf_normal'].detach().double() - surf_normal.detach()).norm(dim=0)
    assert bool((off <= turn + 1e-6)[steady].all())

    names = [k for k in ('images', 'opacity', 'normals', 'depths', 'surf_depth', 'surf_normal', 'distortion') if k in out]
    up = {k: torch.randn(out[k].shape, generator=g).to(device) for k in names}
    up['surf_normal'] = up['surf_normal'] * steady
    wanted = params + [sh] + ([rest] if rest is not None else [])
    keep = [k for k in names if k not in ('images', 'opacity')]
    of64 = {'normals': normals, 'depths': median, 'surf_depth': surf_depth, 'surf_normal': surf_normal,
            'distortion': maps64[5:6]}
    for some in (keep, ['surf_normal']):
        got = torch.autograd.grad([out[k] for k in ['images', 'opacity'] + some], wanted + [out['viewspace_points']],
                                  [up[k] for k in ['images', 'opacity'] + some], retain_graph=True, allow_unused=True)
        g_maps, = torch.autograd.grad([of64[k] for k in some], [maps64], [up[k].double() for k in some], retain_graph=True)
        g_opac = up['opacity'] if background is None else up['opacity'] - (background[:, None, None] * up['images']).sum(0)
        ref = torch.autograd.grad([img, opac, extras], wanted + [m2], [up['images'], g_opac.reshape(opac.shape), g_maps.float()],
                                  retain_graph=True, allow_unused=True)
        for k, (a, b) in enumerate(zip(got, ref)):
            assert (a is None) == (b is None)
            if a is not None:
                # a pixel's part is off by its turn, once for the direction and twice for the two differences' lengths
                assert (a - b).norm() <= 3e-4 * b.norm() + 1e-7
