"""Sums of a surfel's records in the view's backward (wave_record_sums in csrc/preprocess.hip): spans of up to 32 tiles go
record by record, longer ones 64 positions at a time by the whole wavefront. Pictures one tile high, so that a surfel over all of
it has as many tiles as the picture, around both limits; bit for bit what the operators give, whose kernel adds in the same order."""
import pytest
import torch

import test_gpu_native_views as views

pytestmark = pytest.mark.gpu


def _surfels_of_all_sizes(P, W, H, seed, spread=2.0):
    from fast_sp_gs_amd import scenes
    g = torch.Generator().manual_seed(seed)
    return (scenes._surfels(g, P, 'cube', -1.0, spread, -1.0, 1.0),
            scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])), g)


@pytest.mark.parametrize('tiles', [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300])
@pytest.mark.parametrize('P,mode', [(70, 'sh'), (65, 'split'), (300, 'colors')])
def test_spans_around_the_limits(tiles, P, mode, device, monkeypatch):
    monkeypatch.setattr(views, '_scene', lambda P, W, H, seed, scale=None: _surfels_of_all_sizes(P, W, H, seed))
    views.test_surfel_view_equals_operators(P, 16 * tiles, 16, mode, device)


@pytest.mark.parametrize('tiles', [1, 31, 32, 33, 63, 64, 65, 129, 300])
@pytest.mark.parametrize('P,masks', [(19, True), (21, False), (300, True)])
def test_fast_spans_around_the_limits(tiles, P, masks, device):
    """The fast path's sums over records (20 surfels a wavefront, spans above 32 positions by all of it), with the preprocess
    kernel's masks and by the corner test, against device-scope atomics, which add the same terms in any order. A surfel has one
    term per tile, so the two differ by at most the number of tiles times 2^-24 times the sum of the terms' sizes; that sum is
    taken as 16 times the largest result, for surfels no larger than these cancel little."""
    from fast_sp_gs_amd.renderer import fast_render_step
    s, cam_h, g = _surfels_of_all_sizes(P, 16 * tiles, 16, P + tiles, spread=0.7)
    s, cam = s.to(device), cam_h.to(device)
    H, W = cam.H, cam.W
    up = [torch.randn(n, H, W, generator=g).to(device) for n in (3, 8, 1)]
    args = (s, cam, up[0], up[1] * 0.1, up[2][0])
    a = fast_render_step(*args, reuse_masks=masks)
    c = fast_render_step(*args, ordered_sums=False)
    torch.cuda.synchronize()
    assert tiles <= 32 or int(a['tiles_touched'].max()) > 32
    for k in ('g_colors', 'g_means2D_blend', 'g_trans', 'g_inv', 'g_normal_opacity'):
        ref = float(c[k].abs().max())
        assert float((a[k] - c[k]).abs().max()) <= max(tiles, 4) * 2.0 ** -24 * 16 * ref, k
