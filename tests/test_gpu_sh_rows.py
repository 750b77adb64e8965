"""Rows of SH coefficients that a wavefront moves as 16-byte pieces (rows of 48, 45, 27, 16, 12 and 9 floats), against the
path of tensors that start off a 16-byte boundary, around the sizes of a wavefront and a block. Both form the same sums in
the same order; contraction may differ between two instantiations, hence a few units in the last place of the largest term."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 63, 64, 65, 127, 255, 257, 1000]


def off_boundary(t):
    """The same values one float behind a 16-byte boundary."""
    room = torch.empty(t.numel() + 4, device=t.device)
    return room[1:1 + t.numel()].view(t.shape).copy_(t)


def close(a, b, what):
    assert a.shape == b.shape, what
    if a.is_floating_point():
        assert torch.isfinite(a).all(), what
        assert (a - b).abs().max() <= 1e-5 * max(float(b.abs().max()), 1e-6), what
    else:
        assert torch.equal(a, b), what


@pytest.mark.parametrize('P', SIZES)
@pytest.mark.parametrize('degree', [1, 2, 3])
def test_encoders(P, degree, device):
    from fast_sp_gs_amd.ops import SH_to_RGB, sh_encode
    print(f'[sh rows] encoders P={P} degree={degree}', flush=True)
    g = torch.Generator(device=device).manual_seed(P)
    n = (degree + 1) ** 2
    normal = lambda *s: torch.randn(*s, generator=g, device=device)
    dirs, sh, campos = torch.nn.functional.normalize(normal(P, 3), dim=-1), normal(P, n, 3), normal(3)
    g_basis, g_rgb = normal(P, n), normal(P, 3)

    def both(move):
        d, s = dirs.clone().requires_grad_(True), move(sh).requires_grad_(True)
        basis, rgb = sh_encode(d, degree), SH_to_RGB(s, dirs, campos, degree, True)
        return [basis, rgb, *torch.autograd.grad([basis, rgb], [d, s], [move(g_basis), g_rgb])]

    for a, b in zip(both(torch.clone), both(off_boundary)):
        close(a, b, (P, degree))


@pytest.mark.parametrize('P', SIZES)
@pytest.mark.parametrize('path', ['surfel', 'fast', 'gauss'])
@pytest.mark.parametrize('split', [False, True])
def test_renders(P, path, split, device):
    import math

    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd.renderer import GS_2D_render
    from fast_sp_gs_amd.renderer.gaussian_render import render
    from fast_sp_gs_amd.renderer.gs_2d_fast_render import GS_2D_fast_render
    print(f'[sh rows] {path} P={P} split={split}', flush=True)
    g = torch.Generator(device=device).manual_seed(P)
    normal = lambda *s: torch.randn(*s, generator=g, device=device)
    cam = scenes.pinhole(100, 75, 50.0, torch.tensor([0.0, 0.0, 2.0])).to(device)
    xyz = normal(P, 3) * 1.5  # some behind the camera, some outside the picture
    scales = torch.exp(normal(P, 3 if path == 'gauss' else 2) * 0.5 - 3.0)
    rot = torch.nn.functional.normalize(normal(P, 4), dim=-1)
    opacity, sh = torch.sigmoid(normal(P, 1)), normal(P, 16, 3) * 0.3
    upstream = normal(3, 75, 100)

    def both(move):
        p = {'points': xyz, 'scales': scales, 'rotations': rot, 'opacity': opacity}
        if split:
            p.update(sh_features=sh[:, :1].contiguous(), sh_features_rest=move(sh[:, 1:].contiguous()))
        else:
            p.update(sh_features=move(sh))
        p = {k: v.detach().requires_grad_(True) for k, v in p.items()}
        size = (cam.W, cam.H)
        if path == 'surfel':
            out = GS_2D_render(size=size, Tw2v=cam.Tw2v, Tv2c=cam.Tv2c, campos=cam.campos, near=cam.near, far=cam.far,
                               sh_degree=3, **p)
        elif path == 'fast':
            out = GS_2D_fast_render(size=size, Tw2v=cam.Tw2v, Tv2c=cam.Tv2c, Tv2s=cam.Tv2s, campos=cam.campos,
                                    near=cam.near, far=cam.far, sh_degree=3, **p)
        else:
            fov = math.radians(50.0)
            out = render(cam.Tw2v, cam.Tv2c, size, campos=cam.campos,
                         FoV=(fov, 2 * math.atan(math.tan(fov / 2) * 75 / 100)), sh_degree=3, **p)
        return [out['images'], *torch.autograd.grad(out['images'], list(p.values()), upstream)]

    for a, b in zip(both(torch.clone), both(off_boundary)):
        close(a, b, (P, path, split))


@pytest.mark.parametrize('P', SIZES)
@pytest.mark.parametrize('path', ['surfel', 'fast', 'gauss'])
@pytest.mark.parametrize('split', [False, True])
def test_preprocess_rows(P, path, split, device):
    """Every output row of the preprocess operators, those that leave a wavefront together and those that a lane stores itself,
    and, as the outputs are allocated uninitialised, the rows of what is not rendered."""
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd._C import get_C_function
    print(f'[preprocess rows] {path} P={P} split={split}', flush=True)
    g = torch.Generator(device=device).manual_seed(P)
    normal = lambda *s: torch.randn(*s, generator=g, device=device)
    cam = scenes.pinhole(100, 75, 50.0, torch.tensor([0.0, 0.0, 2.0])).to(device)
    shape = [normal(P, 3) * 1.5, torch.exp(normal(P, 3 if path == 'gauss' else 2) * 0.5 - 3.0),
             torch.nn.functional.normalize(normal(P, 4), dim=-1), torch.sigmoid(normal(P, 1))]
    sh = normal(P, 16, 3) * 0.3

    def outputs(move):
        rows = [sh[:, :1].contiguous(), move(sh[:, 1:].contiguous())] if split else [move(sh), None]
        view = [cam.Tw2v, cam.Tv2c]
        if path == 'surfel':
            return get_C_function('gs_2d_preprocess_forward')(100, 75, 3, False, *shape, *rows, *view, cam.campos,
                                                              return_records=True, return_masks=True)
        if path == 'fast':
            return get_C_function('gs_2d_fast_preprocess_forward')(100, 75, 3, False, *shape, *rows, *view, cam.Tv2s, cam.campos)
        return get_C_function('gs_preprocess_forward')(100, 75, 3, False, *shape, *rows, *view, cam.campos, (0.5, 0.4))

    for k, (a, b) in enumerate(zip(outputs(torch.clone), outputs(off_boundary))):
        if path == 'surfel' and k == 7:  # the records: 18 numbers, then the radius and the first slot as integers
            close(a[:, 18:].contiguous().view(torch.int32), b[:, 18:].contiguous().view(torch.int32), (path, k))
            a, b = a[:, :18], b[:, :18]
        close(a, b, (path, k))
