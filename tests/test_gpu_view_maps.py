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
