"""Sums of a surfel's records in the view's backward (wave_record_sums in csrc/preprocess.hip): spans of up to 32 tiles go
record by record, longer ones 64 positions at a time by the whole wavefront. Pictures one tile high, so that a surfel over all of
it has as many tiles as the picture, around both limits; bit for bit what the operators give, whose kernel adds in the same order."""
import pytest
import torch

import test_gpu_native_views as views

pytestmark = pytest.mark.gpu


def _surfels_of_all_sizes(P, W, H, seed):
    from fast_sp_gs_amd import scenes
    g = torch.Generator().manual_seed(seed)
    return (scenes._surfels(g, P, 'cube', -1.0, 2.0, -1.0, 1.0),
            scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])), g)


@pytest.mark.parametrize('tiles', [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300])
@pytest.mark.parametrize('P,mode', [(70, 'sh'), (65, 'split'), (300, 'colors')])
def test_spans_around_the_limits(tiles, P, mode, device, monkeypatch):
    monkeypatch.setattr(views, '_scene', lambda P, W, H, seed, scale=None: _surfels_of_all_sizes(P, W, H, seed))
    views.test_surfel_view_equals_operators(P, 16 * tiles, 16, mode, device)
