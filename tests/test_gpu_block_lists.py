"""Work lists per pixel block of the blend kernels (csrc/block_lists.hpp): a block's list holds every staged entry that can
reach alpha >= 1/255 at one of its pixels, so a render with the bound switched off (fsgs_debug_set_culling: every entry is
evaluated at every pixel) gives the same pictures bit for bit and the same gradients to the rounding of their sums. At list
lengths around the staging batches, on images that end inside a tile, for surfels of every shape: a fraction of a pixel,
several tiles, long and thin, edge-on down to a tilt of 1e-4."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = ["small", "large", "thin", "edge_on"]


def _scene(shape, P, device):
    from fast_sp_gs_amd import scenes
    g = torch.Generator().manual_seed(P)
    scene = scenes._surfels(g, P, 'cube', {'small': -6.5, 'large': -1.5}.get(shape, -3.0), 0.5, 0.0, 1.5, 1.0)
    scene.means3D.mul_(0.4)
    if shape == "thin":
        scene.scales[:, 1] *= 0.01
    if shape == "edge_on":  # turned about a random axis across the view until the camera sees the rim, to within a tilt
        tilt = 10.0 ** (-4.0 + 3.0 * torch.rand(P, generator=g))
        half, roll = (math.pi / 2 - tilt) / 2, torch.rand(P, generator=g) * 2 * math.pi
        scene.rotations = torch.stack([half.sin() * roll.cos(), half.sin() * roll.sin(), torch.zeros(P), half.cos()], 1)
    return scene.to(device), scenes.pinhole(61, 45, 40.0, torch.tensor([0.0, 0.0, 4.0])).to(device)


def _culling(on):
    from fast_sp_gs_amd import lib
    lib.check(lib.load().fsgs_debug_set_culling(int(on)), 'debug_set_culling')


def _both(run):
    with_lists = run()
    torch.cuda.synchronize()
    _culling(False)
    try:
        everything = run()
        torch.cuda.synchronize()
    finally:
        _culling(True)
    return with_lists, everything


@pytest.mark.parametrize("P", [1, 64, 65, 191, 192, 193, 450, 3000])
@pytest.mark.parametrize("shape", SHAPES)
def test_surfel_blend(shape, P, device):
    from fast_sp_gs_amd.renderer import render_step
    scene, cam = _scene(shape, P, device)
    g = torch.Generator().manual_seed(3)
    gi, go = torch.randn(3, cam.H, cam.W, generator=g).to(device), torch.randn(cam.H, cam.W, generator=g).to(device)
    ge = torch.cat([torch.randn(6, cam.H, cam.W, generator=g), torch.zeros(3, cam.H, cam.W)]).to(device)
    a, b = _both(lambda: render_step(scene, cam, gi, ge, go))
    for k in ('image', 'opacity', 'extras', 'n_contrib'):
        assert torch.equal(a[k], b[k]), k
    for k in a:
        if k.startswith('g_') and a[k] is not None:  # sums of at most 1e4 terms: 1e-5 of the largest is 100 roundings
            assert (a[k] - b[k]).abs().max() <= 1e-5 * b[k].abs().max(), k


def _params(scene, axes=2):
    scales = scene.scales if axes == 2 else torch.cat([scene.scales, scene.scales.mean(1, keepdim=True)], 1)
    return {k: v.clone().requires_grad_(True) for k, v in
            dict(points=scene.means3D, scales=scales, rotations=scene.rotations, opacity=scene.opacities,
                 sh_features=scene.shs).items()}


def _gradients(params, maps, seed=5):
    g = torch.Generator().manual_seed(seed)
    up = [torch.randn(m.shape, generator=g).to(m.device) for m in maps]
    return torch.autograd.grad(maps, list(params.values()), up, allow_unused=True)


@pytest.mark.parametrize("P", [1, 95, 96, 97, 700])
@pytest.mark.parametrize("shape", SHAPES)
def test_surfel_view(shape, P, device):
    """The view's backward walks the blocks that the forward noted as blended instead of bounding footprints."""
    from fast_sp_gs_amd.renderer import GS_2D_render
    scene, cam = _scene(shape, P, device)

    def run():
        params = _params(scene)
        out = GS_2D_render(size=(cam.W, cam.H), Tw2v=cam.Tw2v, Tv2c=cam.Tv2c, campos=cam.campos, near=cam.near, far=cam.far,
                           sh_degree=3, background=torch.ones(3, device=device), **params)
        maps = [out[k] for k in ('images', 'normals', 'surf_depth', 'distortion')]
        return maps, _gradients(params, maps)

    (maps, grads), (maps_all, grads_all) = _both(run)
    for a, b in zip(maps, maps_all):
        assert torch.equal(a, b)
    for a, b in zip(grads, grads_all):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()


@pytest.mark.parametrize("P", [1, 127, 128, 129, 191, 192, 193, 900])
@pytest.mark.parametrize("shape", SHAPES)
def test_gaussian_view(shape, P, device):
    from fast_sp_gs_amd.renderer.gaussian_render import render
    scene, cam = _scene(shape, P, device)
    fov = (math.radians(40.0), 2 * math.atan(math.tan(math.radians(20.0)) * cam.H / cam.W))

    def run():
        params = _params(scene, axes=3)
        out = render(cam.Tw2v, cam.Tv2c, (cam.W, cam.H), campos=cam.campos, FoV=fov, sh_degree=3, **params)
        maps = [out['images'], out['opacity']]
        return maps, _gradients(params, maps)

    (maps, grads), (maps_all, grads_all) = _both(run)
    for a, b in zip(maps, maps_all):
        assert torch.equal(a, b)
    for a, b in zip(grads, grads_all):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()


@pytest.mark.parametrize("P", [1, 127, 128, 129, 191, 192, 193, 900])
@pytest.mark.parametrize("shape", SHAPES)
def test_fast_surfel_view(shape, P, device):
    from fast_sp_gs_amd.renderer.gs_2d_fast_render import GS_2D_fast_render
    scene, cam = _scene(shape, P, device)

    def run():
        params = _params(scene)
        out = GS_2D_fast_render(size=(cam.W, cam.H), Tw2v=cam.Tw2v, Tv2c=cam.Tv2c, Tv2s=cam.Tv2s, campos=cam.campos,
                                near=cam.near, far=cam.far, sh_degree=3, **params)
        maps = [out[k] for k in ('images', 'normals', 'surf_depth', 'distortion')]
        return maps, _gradients(params, maps)

    (maps, grads), (maps_all, grads_all) = _both(run)
    for a, b in zip(maps, maps_all):
        assert torch.equal(a, b)
    for a, b in zip(grads, grads_all):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
