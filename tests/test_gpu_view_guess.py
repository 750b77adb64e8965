"""Views are queued for a guessed number of list positions before their instance count is known (positions_to_guess in
csrc/host/torch_util.hpp: 16 per surfel, 65 536 at least, one per surfel and tile at most). Scenes with more instances than that
take their second half again: the same maps, lists, counts and gradients as by the operators, which wait for the count."""
import pytest
import torch

import test_gpu_native_views as views

pytestmark = pytest.mark.gpu


def _large_surfels(P, W, H, seed):
    from fast_sp_gs_amd import scenes
    g = torch.Generator().manual_seed(seed)
    return (scenes._surfels(g, P, 'cube', -0.5, 0.3, -1.0, 1.0),
            scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])), g)


# tiles 1200 (prefix and scan over the tiles) and 540 (the scatter's blocks sum the columns); one surfel: the bound by tiles
@pytest.mark.parametrize('P,W,H,more', [(700, 640, 480, True), (900, 480, 288, True), (1, 480, 288, False)])
@pytest.mark.parametrize('which', ['surfel', 'fast', 'gaussian'])
def test_more_instances_than_guessed(which, P, W, H, more, device, monkeypatch):
    from fast_sp_gs_amd.renderer import GS_2D_render
    s, cam_h, _ = _large_surfels(P, W, H, P + 1)
    s, cam = s.to(device), cam_h.to(device)
    R = GS_2D_render(s.means3D, s.scales, s.rotations, s.opacities, (W, H), cam.Tw2v, cam.Tv2c, campos=cam.campos,
                     sh_degree=3, sh_features=s.shs)['buffer'].R
    assert (R > max(16 * P, 65_536)) == more
    monkeypatch.setattr(views, '_scene', lambda P, W, H, seed, scale=None: _large_surfels(P, W, H, seed))
    if which == 'surfel':
        views.test_surfel_view_equals_operators(P, W, H, 'accum', device)
    elif which == 'fast':
        views.test_fast_surfel_view_equals_operators(P, W, H, 'sh', device)
    else:
        views.test_gaussian_view_equals_operators(P, W, H, 'sh', device)
