"""Binning bit for bit against the oracle around the sizes at which one block does the prefixes and the scan (1024 tiles, 65 536
surfels), around the tile counts at which the counters change places (16 384 tiles: half of a
compute unit's LDS; 40 960: all of it; beyond: global memory) and around one turn of the scan's 4096 tiles per block."""
import numpy as np
import pytest
import torch

from util import npy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('gx,gy,P', [(2, 2, 500), (4, 256, 2000), (41, 25, 1025), (32, 32, 65_536),
                                     (32, 32, 65_537), (33, 31, 8193), (64, 64, 3000), (17, 241, 2000), (128, 128, 5000), (5, 3277, 300), (256, 160, 4000),
                                     (17, 2410, 300), (240, 135, 70_000)])
def test_lists_on_wide_grids(gx, gy, P, device, oracle_mod):
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd._C import get_C_function
    W, H = 16 * gx - 3, 16 * gy - 5
    scene, _ = scenes.config0(P=P, size=max(W, H), seed=4)
    scene.scales = scene.scales * (20.0 if P < 10_000 else 3.0)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0., 0., 4.]))
    d = lambda t: t.to(device).contiguous()
    print(f"[wide grid] {gx}x{gy} tiles, P={P}", flush=True)
    m2, colors, tm, no, dep, radii, tt = get_C_function('gs_2d_preprocess_forward')(
        W, H, 3, False, d(scene.means3D), d(scene.scales), d(scene.rotations), d(scene.opacities), d(scene.shs), None,
        d(cam.Tw2v), d(cam.Tv2c), d(cam.campos), None, None, None)
    ranges, pl, keys = get_C_function('GS_prepare')(W, H, m2, dep, radii, tt, False, return_keys=True)[:3]
    r_ranges, r_pl, r_keys = oracle_mod.prepare(W, H, npy(m2), npy(dep), npy(radii), npy(tt), return_keys=True)
    assert r_pl.size > P
    assert np.array_equal(npy(ranges), r_ranges) and np.array_equal(npy(pl), r_pl) and np.array_equal(npy(keys), r_keys)
