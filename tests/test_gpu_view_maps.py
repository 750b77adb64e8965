"""The maps that a view's blend writes itself, and the pseudo normal behind it, against the raw maps of the same view put through
the epilogue operator, with and without what a backward needs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('W,H', [(1, 1), (2, 3), (16, 16), (63, 17), (64, 16), (65, 33), (131, 77)])
@pytest.mark.parametrize('kind,ratio,background', [('surfel', 1.0, True), ('surfel', 0.3, True), ('surfel', 0.0, False),
                                                   ('fast', 1.0, False), ('fast', 0.3, False)])
def test_view_maps_equal_the_epilogue(kind, ratio, background, W, H, device):
    """Every map that is one pixel's own bit for bit. The pseudo normal: both kernels fuse products and sums as they like."""
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd._C import get_C_function
    from fast_sp_gs_amd.lib import host
    print(f'[view maps] {kind} {W}x{H} ratio={ratio}', flush=True)
    g = torch.Generator().manual_seed(W)
    P = 400
    points, scales, rotations, opacities, shs = [t.to(device) for t in (
        (torch.rand(P, 3, generator=g) - 0.5) * 2, torch.exp(torch.randn(P, 2, generator=g) * 0.4 - 2.2),
        torch.nn.functional.normalize(torch.randn(P, 4, generator=g), dim=-1), torch.sigmoid(torch.randn(P, 1, generator=g)),
        torch.randn(P, 16, 3, generator=g) * 0.2)]
    cam = scenes.pinhole(W, H, 45.0, torch.tensor([0.3, -0.2, 3.5])).to(device)
    bg = torch.tensor([0.2, 0.5, 0.9], device=device) if background else None

    def view(points, epilogue):
        m2, none = torch.empty(P, 2, device=device), [None] * 5
        if kind == 'surfel':
            return host.surfel_render(points, scales, rotations, opacities, shs, None, m2, cam.Tw2v, cam.Tv2c, cam.campos,
                                      bg if epilogue else None, *none, W, H, 3, 0.2, 100.0, ratio, epilogue, True)[0]
        return host.fast_surfel_render(points, scales, rotations, opacities, shs, None, m2, cam.Tw2v, cam.Tv2c, cam.Tv2s,
                                       cam.campos, *none, W, H, 3, 0.2, 100.0, ratio, epilogue)[0]

    with torch.no_grad():
        image, opacity, extras = view(points, False)
        plain = view(points, True)
    for a, b in zip(plain, view(points.clone().requires_grad_(True), True)):
        assert torch.equal(a, b.detach())
    nine = torch.cat([extras, extras[:9 - extras.shape[0]]])
    normals, depths, surf_depth, surf_normal, composited = get_C_function('gs_2d_epilogue_forward')(
        W, H, ratio, cam.Tw2v, cam.Tv2c, nine, opacity, image if background else None, bg)
    want = {'surfel': [composited if background else image, opacity, normals, depths, surf_depth, surf_normal, extras[5:6]],
            'fast': [image, opacity, normals, surf_depth, surf_normal, extras[5:6]]}[kind]
    for k, (a, b) in enumerate(zip(plain, want)):
        a, b = a.reshape(-1), b.reshape(-1)
        if b.data_ptr() != surf_normal.data_ptr():
            assert torch.equal(a, b), k
        else:
            # a normal turns by the rounding of world coordinates (2^-23 of about 4, a few operations each way) against the length
            # of their differences, two pixels (a pixel is 2 tan(22.5 deg) 3.5 / W) at least
            turn = 16 * 2.0 ** -23 * 4 / (2 * 2 * 0.414 * 3.5 / W)
            assert float((a - b).abs().max()) <= turn, (k, float((a - b).abs().max()), turn)


@pytest.mark.parametrize('visible', [True, False])
@pytest.mark.parametrize('kind,maps', [('surfel', ('images',)), ('surfel', ('images', 'normals')), ('fast', ('images',)),
                                       ('fast', ('images', 'distortion'))])
def test_absent_opacity_gradient_is_a_zero_one(kind, maps, visible, device):
    """A loss that does not use the opacity map gives the gradients of one that uses it times zero, bit for bit (the sums are
    records, added in a fixed order), also for a view that sees nothing."""
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd.renderer import GS_2D_render
    from fast_sp_gs_amd.renderer.gs_2d_fast_render import GS_2D_fast_render
    print(f'[view maps] {kind} {maps} visible={visible}', flush=True)
    scene, cam = scenes.config0(P=3000, size=100, seed=3)
    scene, cam = scene.to(device), cam.to(device)
    centres = scene.means3D if visible else scene.means3D - 100.0 * cam.Tw2v[2, :3]
    params = [t.clone().requires_grad_(True) for t in (centres, scene.scales, scene.rotations, scene.opacities, scene.shs)]
    g = torch.Generator(device=device).manual_seed(1)
    up = {k: torch.randn(n, 100, 100, generator=g, device=device) for k, n in (('images', 3), ('normals', 3), ('distortion', 1))}

    def grads(with_opacity):
        render, view = (GS_2D_render, (cam.Tw2v, cam.Tv2c)) if kind == 'surfel' else \
            (GS_2D_fast_render, (cam.Tw2v, cam.Tv2c, cam.Tv2s))
        out = render(*params[:4], (100, 100), *view, campos=cam.campos, sh_degree=3, sh_features=params[4])
        assert bool(out['visibility_filter'].any()) == visible
        used = [out[k] for k in maps] + ([out['opacity']] if with_opacity else [])
        return torch.autograd.grad(used, params, [up[k] for k in maps] +
                                   ([torch.zeros_like(out['opacity'])] if with_opacity else []))

    for a, b in zip(grads(False), grads(True)):
        assert torch.isfinite(a).all() and torch.equal(a, b)
        assert bool(a.any()) == visible
