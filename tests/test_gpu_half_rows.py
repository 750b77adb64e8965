"""The preprocess kernels' rows of coefficients reach their lanes 32 at a time: colours against the rows themselves in double precision, at
the edges of half wavefronts, with one half, all of one half but a lane, or nothing of a wavefront on the screen."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _basis(d):  # real spherical harmonics to degree 3 of unit directions, in double precision
    x, y, z = d.unbind(-1)
    xx, yy, zz = x * x, y * y, z * z
    return torch.stack([
        0.28209479177387814 + 0 * x, -0.48860251190291987 * y, 0.48860251190291987 * z, -0.48860251190291987 * x,
        1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.31539156525252005 * (3 * zz - 1), -1.0925484305920792 * x * z,
        0.5462742152960396 * (xx - yy), 0.5900435899266435 * y * (-3 * xx + yy), 2.890611442640554 * x * y * z,
        0.4570457994644657 * y * (1 - 5 * zz), 0.3731763325901154 * z * (5 * zz - 3), 0.4570457994644657 * x * (1 - 5 * zz),
        1.445305721320277 * z * (xx - yy), 0.5900435899266435 * x * (-xx + 3 * yy)], -1)


HIDDEN = {'none': lambda r: r < 0, 'first half': lambda r: r < 32, 'second half': lambda r: r >= 32, 'all but 31': lambda r: r != 31,
          'all but 32': lambda r: r != 32, 'every other': lambda r: r % 2 == 0, 'all': lambda r: r >= 0}


@pytest.mark.parametrize('P', [1, 31, 32, 33, 63, 65, 96, 97, 255, 289])
@pytest.mark.parametrize('path', ['surfel', 'fast', 'gauss'])
@pytest.mark.parametrize('split', [False, True])
def test_colors(P, path, split, device):
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd._C import get_C_function
    print(f'[half rows] {path} P={P} split={split}', flush=True)
    g = torch.Generator(device=device).manual_seed(P)
    normal = lambda *s: torch.randn(*s, generator=g, device=device)
    cam = scenes.pinhole(100, 75, 50.0, torch.tensor([0.0, 0.0, 2.0])).to(device)
    shape = [torch.exp(normal(P, 3 if path == 'gauss' else 2) * 0.3 - 3.0), torch.nn.functional.normalize(normal(P, 4), dim=-1),
             torch.sigmoid(normal(P, 1))]
    sh = normal(P, 16, 3)
    rows = [sh[:, :1].contiguous(), sh[:, 1:].contiguous()] if split else [sh, None]
    at = torch.arange(P, device=device) % 64
    for name, hidden in HIDDEN.items():
        points = normal(P, 3) * 0.2
        points[hidden(at)] = 2.0 * cam.campos  # behind the camera
        if path == 'surfel':
            out = get_C_function('gs_2d_preprocess_forward')(100, 75, 3, False, points, *shape, *rows, cam.Tw2v, cam.Tv2c, cam.campos)
            colors, radii = out[1], out[5]
        elif path == 'fast':
            out = get_C_function('gs_2d_fast_preprocess_forward')(100, 75, 3, False, points, *shape, *rows, cam.Tw2v, cam.Tv2c, cam.Tv2s,
                                                                  cam.campos)
            colors, radii = out[1], out[6]
        else:
            out = get_C_function('gs_preprocess_forward')(100, 75, 3, False, points, *shape, *rows, cam.Tw2v, cam.Tv2c, cam.campos, (0.5, 0.4))
            colors = next(t for t in out if t.shape == (P, 3) and t.dtype == torch.float32)
            radii = next(t for t in out if t.shape == (P,) and t.dtype == torch.int32)
        seen = radii > 0
        assert not seen[hidden(at)].any() and (name != 'none' or seen.sum() >= 0.9 * P)
        Y = _basis(torch.nn.functional.normalize(points.double() - cam.campos.double(), dim=-1))
        want = (Y[:, :, None] * sh.double()).sum(1) + 0.5
        # sixteen terms of at most 2.9 |c| a summand: each is formed and added with a rounding, its direction and basis with some ten more
        bound = 26 * 2.0 ** -24 * ((Y.abs() + 1.0)[:, :, None] * sh.double().abs()).sum(1) + 2.0 ** -23
        assert ((colors.double() - want.clamp_min(0)).abs() <= bound)[seen].all(), name


@pytest.mark.parametrize('P', [1, 31, 32, 33, 63, 65, 97, 255, 289])
@pytest.mark.parametrize('grad', [False, True])
def test_sh_to_rgb(P, grad, device):
    from fast_sp_gs_amd.ops import SH_to_RGB
    print(f'[half rows] SH_to_RGB P={P} grad={grad}', flush=True)
    g = torch.Generator(device=device).manual_seed(P)
    sh, points = torch.randn(P, 16, 3, generator=g, device=device), torch.randn(P, 3, generator=g, device=device)
    campos = torch.tensor([0.3, -0.2, 5.0], device=device)
    Y = _basis(torch.nn.functional.normalize(points.double() - campos.double(), dim=-1))
    want = (Y[:, :, None] * sh.double()).sum(1) + 0.5
    bound = 26 * 2.0 ** -24 * ((Y.abs() + 1.0)[:, :, None] * sh.double().abs()).sum(1) + 2.0 ** -23  # as above
    got = SH_to_RGB(sh.requires_grad_(grad), points.requires_grad_(grad), campos, 3, True)
    assert ((got.double() - want.clamp_min(0)).abs() <= bound).all()
