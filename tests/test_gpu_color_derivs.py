"""The colours' derivatives by the view direction that a view's forward keeps for its backward (instead of its reading the coefficients
again): the same gradients, bit for bit, as from the coefficients, which the backward reads where their rows do not allow it. At the
edges of wavefronts and half wavefronts, with the first coefficient apart and not, with points beside the picture."""
import pytest
import torch

pytestmark = pytest.mark.gpu

KINDS = ['surfel', 'fast', 'gaussian']


def _view(kind, P, split, device, hooks=None):
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd.renderer import GS_2D_render
    from fast_sp_gs_amd.renderer.gaussian_render import render
    from fast_sp_gs_amd.renderer.gs_2d_fast_render import GS_2D_fast_render
    g = torch.Generator().manual_seed(P)
    s = scenes._surfels(g, P, 'cube', -3.0, 0.5, 0.0, 1.0, 1.0)
    s.means3D.mul_(1.5)  # a few of them beside the picture
    s = s.to(device)
    cam = scenes.pinhole(61, 45, 40.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    scales = torch.cat([s.scales, s.scales[:, :1]], 1) if kind == 'gaussian' else s.scales
    wrt = [t.clone().requires_grad_(True) for t in (s.means3D, scales, s.rotations, s.opacities)]
    sh = [s.shs[:, :1].contiguous(), s.shs[:, 1:].contiguous()] if split else [s.shs.clone()]
    wrt += [t.requires_grad_(True) for t in sh]
    pts, sc, rot, op = wrt[:4]
    rest = wrt[5] if split else None
    common = dict(campos=cam.campos, sh_degree=3, sh_features=wrt[4], sh_features_rest=rest)
    with torch.autograd.graph.saved_tensors_hooks(*hooks) if hooks else torch.enable_grad():
        if kind == 'surfel':
            out = GS_2D_render(pts, sc, rot, op, (cam.W, cam.H), cam.Tw2v, cam.Tv2c, near=cam.near, far=cam.far, **common)
        elif kind == 'fast':
            out = GS_2D_fast_render(pts, sc, rot, op, (cam.W, cam.H), cam.Tw2v, cam.Tv2c, cam.Tv2s, near=cam.near, far=cam.far, **common)
        else:
            out = render(cam.Tw2v, cam.Tv2c, (cam.W, cam.H), points=pts, scales=sc, rotations=rot, opacity=op, FoV=(0.7, 0.52), **common)
    up = torch.randn(out['images'].shape, generator=torch.Generator().manual_seed(1)).to(device)
    return torch.autograd.grad(out['images'], wrt, up)


def _move(t):  # the same values four bytes off a 16-byte boundary: no complete rows then
    if t.dtype != torch.float32 or t.dim() != 3 or t.numel() == 0:
        return t
    room = torch.empty(t.numel() + 1, device=t.device)
    return room[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize('P', [1, 31, 32, 33, 64, 65, 255, 257, 1500])
@pytest.mark.parametrize('split', [False, True])
@pytest.mark.parametrize('kind', KINDS)
def test_kept_or_formed_again(kind, split, P, device):
    kept = _view(kind, P, split, device)
    again = _view(kind, P, split, device, hooks=(lambda t: t, _move))
    for a, b in zip(kept, again):
        if kind == 'gaussian':  # its blend adds by atomics, in any order: a few roundings of sums of at most 1e4 terms
            assert (a - b).abs().max() <= 1e-5 * b.abs().max() + 1e-30
        else:
            assert torch.equal(a, b)


@pytest.mark.parametrize('P', [1, 31, 33, 64, 255, 257, 1500])
@pytest.mark.parametrize('camera', [False, True])
def test_sh_to_rgb_kept_or_formed_again(P, camera, device):
    """The operator pair on its own: every choice of gradients, from the forward's derivatives (and, without a gradient of the direction,
    from nothing of the coefficients) against gradients from the coefficients, which rows off a 16-byte boundary are given."""
    from fast_sp_gs_amd.ops import SH_to_RGB
    print(f'[colour derivatives] SH_to_RGB P={P} camera={camera}', flush=True)
    g = torch.Generator().manual_seed(P)
    normal = lambda *s: torch.randn(*s, generator=g).to(device)
    sh, pos, cam, up = normal(P, 16, 3) * 0.4, normal(P, 3), normal(3) * 3.0, normal(P, 3)
    if not camera:
        pos = torch.nn.functional.normalize(pos, dim=-1)
    for wants in range(1, 8 if camera else 4):
        def run(move):
            p = [move(sh), pos.clone(), cam.clone() if camera else None]
            wrt = [t.requires_grad_(True) for k, t in enumerate(p) if t is not None and wants >> k & 1]
            rgb = SH_to_RGB(*p, 3, True)
            return [rgb, *torch.autograd.grad(rgb, wrt, up)]
        for k, (a, b) in enumerate(zip(run(torch.clone), run(_move))):
            if a.shape == (3,):  # the camera's: sums over blocks of 256 points, one atomic each, in any order
                assert (a - b).abs().max() <= 1e-6 * P ** 0.5 * max(float(b.abs().max()), 1.0)
            elif k == 0:  # the colours: contraction may differ between the two kernels, 16 terms of at most a few units
                assert (a - b).abs().max() <= 16 * 2 ** -23
            else:
                assert torch.equal(a, b), (wants, k)
