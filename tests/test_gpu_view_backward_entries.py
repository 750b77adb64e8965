"""The views' backward entry points of the C ABI called directly, with and without the forward's notes: record slots by regions hold
what the operators' records by prefix scan hold, so the per-surfel sums are the operators' ordered sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 33, 17), (300, 61, 45), (5000, 160, 96)]


def _scene(P, W, H, device):
    from fast_sp_gs_amd import scenes
    scene, _ = scenes.config0(P=P, size=64, seed=P)
    scene.scales = scene.scales * 3
    return scene.to(device), scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)


def _by_regions(touched):
    """Slots of the prefix scan as region 0's offsets: the regions' first slots are all 0."""
    offsets = (touched.cumsum(0) - touched).int()
    return offsets, torch.zeros(64, dtype=torch.int32, device=touched.device)


def _close(a, b):  # sums of the same addends in another grouping: at most 1e4 of them, 1e-5 of the largest is 100 roundings
    return bool((a - b).abs().max() <= 1e-5 * b.abs().max() + 1e-30)


@pytest.mark.parametrize('P,W,H', SIZES)
def test_surfel_view_backward(P, W, H, device):
    from fast_sp_gs_amd import lib as L
    from fast_sp_gs_amd._C import get_C_function as f
    print(f'[view backward entries] surfels P={P} {W}x{H}', flush=True)
    lib, p = L.load(), L.ptr
    scene, cam = _scene(P, W, H, device)
    m2, col, tm, no, dep, rad, tt = f('gs_2d_preprocess_forward')(
        W, H, 3, False, scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs, None, cam.Tw2v, cam.Tv2c, cam.campos,
        None, None, None)
    ranges, pl, scan = f('GS_prepare')(W, H, m2, dep, rad, tt, False, return_offsets=True)[:3]
    records = torch.empty(P, 20, device=device)
    L.check(lib.fsgs_gs_2d_pack_records(P, p(m2), p(col), p(no), p(tm), p(rad), None, p(records), L.current_stream()), 'pack')
    R = pl.numel()
    hits = torch.zeros(max(R, 1), dtype=torch.int32, device=device)
    oc, oo, oe = (torch.empty(n, H, W, device=device) for n in (3, 1, 9))
    nc = torch.empty(2, H, W, dtype=torch.int32, device=device)
    maps = [torch.empty(n, H, W, device=device) for n in (3, 1, 1, 1)]
    L.check(lib.fsgs_gs_2d_view_forward(P, W, H, cam.near, cam.far, p(m2), p(col), p(no), p(tm), p(pl), p(ranges), None, None, None, None,
                                        p(oc), p(oo), p(oe), None, p(nc), p(records), p(hits), 0.0, p(cam.Tw2v), None,
                                        *[p(m) for m in maps], L.current_stream()), 'forward')
    g = torch.Generator().manual_seed(P)
    gi, go = torch.randn(3, H, W, generator=g).to(device), torch.randn(H, W, generator=g).to(device)
    ge = torch.cat([torch.randn(6, H, W, generator=g), torch.zeros(3, H, W)]).to(device)
    want = f('GS_2D_render_backward')(m2, no, col, tm, None, oo[0], oe, None, gi, go, ge, None, ranges, pl, nc, cam.near, cam.far, scan, rad)
    offsets, regions = _by_regions(tt)
    owner = torch.repeat_interleave(torch.arange(P, device=device), tt.long())
    got = {}
    for name, tail in (('', ()), ('_hits', (p(hits),)), ('_hits', (None,))):
        ws = torch.full((lib.fsgs_gs_2d_render_backward_workspace_bytes(R) // 4,), float('nan'), device=device)
        L.check(getattr(lib, 'fsgs_gs_2d_view_backward' + name)(
            P, W, H, cam.near, cam.far, p(m2), p(no), p(col), p(tm), None, p(oo), p(oe), None, p(gi), p(go), p(ge), None, p(ranges), p(pl),
            p(nc), R, p(offsets), p(regions), p(tt), p(rad), p(ws), ws.numel() * 4, p(records), *tail, L.current_stream()), name)
        sums = torch.zeros(P, 18, device=device).index_add_(0, owner, ws[:18 * R].view(R, 18))
        assert _close(sums[:, :3], want[0]) and _close(sums[:, 3:12], want[2].view(P, 9))
        assert _close(sums[:, 12:16], want[3]) and _close(sums[:, 16:], want[1])
        got[name, tail] = ws[:18 * R].clone()
    plain, _, without = got.values()
    assert torch.equal(plain, without)


@pytest.mark.parametrize('P,W,H', SIZES)
def test_fast_surfel_view_backward(P, W, H, device):
    from fast_sp_gs_amd import lib as L
    from fast_sp_gs_amd._C import get_C_function as f
    print(f'[view backward entries] fast surfels P={P} {W}x{H}', flush=True)
    lib, p = L.load(), L.ptr
    scene, cam = _scene(P, W, H, device)
    (m2, col, tm, inv, no, dep, rad, ranges, pl, _, tt, scan, keep) = f('gs_2d_fast_preprocess_forward')(
        W, H, 3, False, scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs, None, cam.Tw2v, cam.Tv2c, cam.Tv2s,
        cam.campos, None, None, None, False, True, True, True)
    oc, oo, oe, _, nc = f('GS_2D_fast_render_forward')(W, H, cam.near, cam.far, False, m2, col, no, tm, inv, pl, ranges)[:5]
    g = torch.Generator().manual_seed(P)
    gi, go = torch.randn(3, H, W, generator=g).to(device), torch.randn(H, W, generator=g).to(device)
    ge = torch.cat([torch.randn(6, H, W, generator=g), torch.zeros(2, H, W)]).to(device)
    want = f('GS_2D_fast_render_backward')(m2, no, col, tm, inv, None, oc, oo, oe, None, gi, go, ge, None, ranges, pl, nc, cam.near,
                                           cam.far, None, None, None, None, None, None, scan, rad, keep_masks=keep)
    R = pl.numel()
    offsets, regions = _by_regions(tt)
    for name, tail in (('', ()), ('_hits', (None,))):
        outs = [torch.full_like(t, float('nan')) for t in want]
        ws = torch.empty(lib.fsgs_gs_2d_fast_render_backward_workspace_bytes(R), dtype=torch.uint8, device=device)
        L.check(getattr(lib, 'fsgs_gs_2d_fast_view_backward' + name)(
            P, W, H, cam.near, cam.far, p(m2), p(no), p(col), p(tm), p(inv), None, p(oo), p(oe), None, p(gi), p(go), p(ge), None, p(ranges),
            p(pl), p(nc), *[p(t) for t in outs], R, p(offsets), p(regions), p(tt), p(rad), p(ws), ws.numel(), p(keep), *tail,
            L.current_stream()), name)
        assert all(torch.equal(a, b) for a, b in zip(outs, want))
