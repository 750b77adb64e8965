"""Backward of the blend operators on footprints that cover whole tiles: an entry then takes a place in all 16 rows of a tile and a
batch is over after 14 or 15 entries, so the staged entries are walked in several batches. Lists around the lengths where a
batch, the staging and the wavefront's half end; gradients against the oracle in float64, within 1e-4 of a tensor's largest entry:
400 entries' transmittance is a product of 400 factors rounded to 6e-8 each, 2.4e-5, and the plane gradients lose a digit more."""
import numpy as np
import pytest
import torch

from util import check_blend_gradients, f64, npy

pytestmark = pytest.mark.gpu

LENGTHS = [1, 14, 15, 16, 17, 63, 64, 65, 127, 128, 129, 143, 257, 400]


def _scene(P, device, axes=2):
    """P faint surfels (or Gaussians) over all of a picture whose sides are no multiples of a tile."""
    from fast_sp_gs_amd import scenes
    g = torch.Generator().manual_seed(P)
    scene = scenes._surfels(g, P, 'cube', -0.3, 0.3, -3.0, 0.7)
    scene.means3D.mul_(0.3)
    scene.scales = scene.scales if axes == 2 else torch.cat([scene.scales, scene.scales.mean(1, keepdim=True)], 1)
    cam = scenes.pinhole(43, 27, 40.0, torch.tensor([0.0, 0.0, 4.0]))
    return scene.to(device), cam.to(device), g


def _upstream(g, cam, device, extras):
    r = lambda *shape: torch.randn(*shape, generator=g).to(device)
    ge = torch.zeros(extras, cam.H, cam.W, device=device)
    ge[:6] = r(6, cam.H, cam.W)
    return r(3, cam.H, cam.W), r(cam.H, cam.W), ge, r(cam.H, cam.W, 2)


def _moved(scene, cam, radii, g, f):
    """Transforms of the same surfels a little elsewhere: what the optical flow is taken to."""
    to = (scene.means3D + 0.02 * torch.randn(scene.P, 3, generator=g).to(radii.device)).contiguous()
    t2 = f('gs_2d_compute_transmat_forward')(cam.W, cam.H, to, scene.scales, scene.rotations, cam.Tw2v,
                                             (cam.Tv2c @ cam.Tw2v).contiguous())[0]
    return (t2 * (radii[:, None, None] > 0)).contiguous()


def _check(tag, names, got, reference):
    rows = lambda ts: {k: np.asarray(npy(t) if isinstance(t, torch.Tensor) else t, np.float64) for k, t in zip(names, ts) if t is not None}
    check_blend_gradients(tag, rows(got), rows(reference(f64)), lambda: rows(reference(lambda a: a)), tol=1e-4)


@pytest.mark.parametrize('flow', [False, True])
@pytest.mark.parametrize('P', LENGTHS)
def test_surfels(P, flow, device, oracle_mod):
    from fast_sp_gs_amd._C import get_C_function as f
    scene, cam, g = _scene(P, device)
    print(f'[wide surfels] P={P} flow={flow}', flush=True)
    m2, col, tm, no, dep, rad, tt = f('gs_2d_preprocess_forward')(
        cam.W, cam.H, 3, False, scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs, None, cam.Tw2v, cam.Tv2c,
        cam.campos, None, None, None)
    ranges, pl, offsets = f('GS_prepare')(cam.W, cam.H, m2, dep, rad, tt, False, return_offsets=True)[:3]
    t2 = _moved(scene, cam, rad, g, f) if flow else None
    oc, oo, oe, of, nc = f('GS_2D_render_forward')(cam.W, cam.H, m2, col, no, tm, pl, ranges, cam.near, cam.far, False, t2)
    gi, go, ge, gf = _upstream(g, cam, device, 9)
    gf = gf if flow else None

    def reference(cast):
        c = lambda t: cast(npy(t))
        return oracle_mod.render_backward(c(m2), c(no), c(col), c(tm), c(t2), c(oo), c(oe), c(of), c(gi), c(go), c(ge), c(gf),
                                          npy(ranges), npy(pl), npy(nc), cam.near, cam.far)

    for ordered in (True, False):
        got = f('GS_2D_render_backward')(m2, no, col, tm, t2, oo, oe, of, gi, go, ge, gf, ranges, pl, nc, cam.near, cam.far,
                                         offsets if ordered else None, rad if ordered else None)
        _check(f'wide surfels {P} flow={flow} ordered={ordered}', ('colors', 'means2D', 'trans_mat', 'normal_opacity'), got, reference)


@pytest.mark.parametrize('flow', [False, True])
@pytest.mark.parametrize('P', LENGTHS)
def test_fast_surfels(P, flow, device, oracle_mod):
    from fast_sp_gs_amd._C import get_C_function as f
    scene, cam, g = _scene(P, device)
    print(f'[wide fast surfels] P={P} flow={flow}', flush=True)
    (m2, col, tm, inv, no, dep, rad, ranges, pl, _, _, offsets, _) = f('gs_2d_fast_preprocess_forward')(
        cam.W, cam.H, 3, False, scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs, None, cam.Tw2v, cam.Tv2c,
        cam.Tv2s, cam.campos, None, None, None, False, True, True, True)
    t2 = _moved(scene, cam, rad, g, f) if flow else None
    oc, oo, oe, of, nc = f('GS_2D_fast_render_forward')(cam.W, cam.H, cam.near, cam.far, False, m2, col, no, tm, inv, pl, ranges,
                                                        t2)[:5]
    gi, go, ge, gf = _upstream(g, cam, device, 8)
    gf = gf if flow else None

    def reference(cast):
        c = lambda t: cast(npy(t))
        return oracle_mod.fast_render_backward(cam.near, cam.far, 0, c(m2), c(no), c(col), c(tm), c(inv), c(oo), c(oe), c(gi), c(go),
                                               c(ge), npy(ranges), npy(pl), npy(nc), c(t2), c(of), c(gf))

    for ordered in (True, False):
        got = f('GS_2D_fast_render_backward')(m2, no, col, tm, inv, t2, oc, oo, oe, of, gi, go, ge, gf, ranges, pl, nc, cam.near,
                                              cam.far, None, None, None, None, None, None, offsets if ordered else None,
                                              rad if ordered else None)
        _check(f'wide fast surfels {P} flow={flow} ordered={ordered}',
               ('colors', 'means2D', 'trans_mat', 'inverse_m', 'normal_opacity'), got, reference)


@pytest.mark.parametrize('E', [0, 1, 4])
@pytest.mark.parametrize('P', LENGTHS)
def test_gaussians(P, E, device, oracle_mod):
    from fast_sp_gs_amd._C import get_C_function as f
    scene, cam, g = _scene(P, device, axes=3)
    print(f'[wide Gaussians] P={P} E={E}', flush=True)
    tan = (cam.W / 2 / float(cam.Tv2s[0, 0]), cam.H / 2 / float(cam.Tv2s[1, 1]))
    m2, dep, col, rad, tt, _, co = f('gs_preprocess_forward')(
        cam.W, cam.H, 3, False, scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs, None, cam.Tw2v, cam.Tv2c,
        cam.campos, tan, None, None, None, None)
    ranges, pl, offsets = f('GS_prepare')(cam.W, cam.H, m2, dep, rad, tt, False, return_offsets=True)[:3]
    ex = torch.randn(P, E, generator=g).to(device) if E else None
    oc, oo, oe, nc = f('gaussian_rasterize_forward')(cam.W, cam.H, m2, co, col, ex, pl, ranges)
    gi, go, ge, _ = _upstream(g, cam, device, 8)
    gx = ge[:E].contiguous() if E else None

    def reference(cast):
        c = lambda t: cast(npy(t))
        return oracle_mod.gs3d_render_backward(cam.W, cam.H, c(m2), c(co), c(col), c(ex), c(oo), npy(nc), c(gi), c(gx), c(go), npy(pl),
                                               npy(ranges))

    for ordered in (True, False):
        got = f('gaussian_rasterize_backward')(m2, co, col, ex, oo, gi, go, gx, ranges, pl, nc, offsets if ordered else None,
                                               rad if ordered else None)
        _check(f'wide Gaussians {P} E={E} ordered={ordered}', ('colors', 'extras', 'means2D', 'conic_opacity'), got, reference)
