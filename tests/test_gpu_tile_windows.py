"""Views without gradients leave the tiles of large rectangles (above 32 tiles) that no pixel can blend out of their lists by a
window per surfel; views with gradients keep those rectangles whole. Maps must be equal bit for bit, a list without gradients a
subsequence of the one with them that holds every surfel the other's blend reached. Sizes: rectangles around 32 tiles, more than
16 columns or rows (a sixteenth of the window then holds several tiles), long thin ones, the whole picture, more columns than
lanes, grids beyond the counters in LDS."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('P,W,H,scale,thin', [
    (300, 97, 95, -0.6, 1.5), (500, 113, 67, -1.6, 2.5), (400, 640, 353, -2.4, 0.0), (400, 640, 353, -1.4, 3.5),
    (257, 511, 1203, -0.8, 5.0), (200, 1601, 97, 0.3, 3.0), (64, 3333, 3171, -1.5, 4.0), (1, 801, 601, -1.0, 6.0)])
def test_windows_change_no_map(P, W, H, scale, thin, device):
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd.renderer import gs_2d_render as m
    g = torch.Generator().manual_seed(P + W)
    s = scenes._surfels(g, P, 'cube', scale, 0.7, 0.0, 1.5)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])).to(device)
    scales = s.scales.clone()
    scales[:, 0] *= torch.exp(-thin * torch.rand(P, generator=g))
    opacities = s.opacities.clone()
    opacities[::7] = 0.0039  # below 1/255: no tile
    args = [t.to(device) for t in (s.means3D, scales, s.rotations, opacities)]
    shs = s.shs.to(device)

    def view(grad):
        with torch.set_grad_enabled(grad):
            return m.GS_2D_render(*args, (W, H), cam.Tw2v, cam.Tv2c, campos=cam.campos, sh_degree=3, near=0.2, far=100.0,
                                  sh_features=shs)

    whole, out = view(True), view(False)
    for k, v in whole.items():
        if torch.is_tensor(v) and k != 'viewspace_points':
            assert torch.equal(torch.nan_to_num(v), torch.nan_to_num(out[k])), k
    full, some = whole['buffer'], out['buffer']
    entries = []
    for b in (full, some):
        n = b.tile_ranges[:, 1] - b.tile_ranges[:, 0]
        tile = torch.repeat_interleave(torch.arange(n.numel(), device=device), n)
        first = torch.repeat_interleave(b.tile_ranges[:, 0] - (n.cumsum(0) - n), n)
        entries.append((tile * P + b.point_list[torch.arange(tile.numel(), device=device) + first].long()).cpu())
    at = {k: i for i, k in enumerate(entries[0].tolist())}
    places = torch.tensor([at[k] for k in entries[1].tolist()])
    assert bool((places[1:] > places[:-1]).all())  # a subsequence, tile by tile
    if thin or P == 400:
        assert entries[1].numel() < entries[0].numel()
    # the last surfel that each pixel blended is still in its list
    gx = (W + 15) // 16
    for b, name in ((full, 'whole'), (some, 'window')):
        last = b.n_contribed[0].reshape(H, W).long()
        y, x = torch.meshgrid(torch.arange(H, device=device), torch.arange(W, device=device), indexing='ij')
        start = b.tile_ranges[:, 0][(y // 16) * gx + x // 16]
        ids = torch.where(last > 0, b.point_list[(start + last - 1).clamp(min=0)].long(), -1)
        if name == 'whole':
            want = ids
    assert torch.equal(ids, want)


def test_only_views_without_a_backward_get_windows(device):
    """The C entries: without record slots, too, the masks of large rectangles have all bits set, as the sums of
    `fsgs_gs_2d_render_backward_culled` expect them; with `_no_backward` they are windows, the others' masks are the same."""
    from fast_sp_gs_amd import lib as L, scenes
    lib, stream = L.load(), L.current_stream()
    P, W, H = 400, 640, 353
    g = torch.Generator().manual_seed(7)
    s = scenes._surfels(g, P, 'cube', -1.4, 0.7, 0.0, 1.5).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])).to(device)

    def masks(entry, *slots):
        f = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device=device)
        means2D, colors, trans, normal_opacity, depths = f(P, 2), f(P, 3), f(P, 3, 3), f(P, 4), f(P)
        radii, touched, keep = f(P, dtype=torch.int32), f(P, dtype=torch.int32), f(P, dtype=torch.int32)
        counters = torch.zeros(64, dtype=torch.int64, device=device)
        L.check(entry(P, W, H, 3, 16, L.ptr(s.means3D), L.ptr(s.scales), L.ptr(s.rotations), L.ptr(s.opacities), L.ptr(s.shs), None,
                      L.ptr(cam.Tw2v), L.ptr(cam.Tv2c), L.ptr(cam.campos), None, L.ptr(means2D), L.ptr(colors), L.ptr(trans),
                      L.ptr(normal_opacity), L.ptr(depths), L.ptr(radii), None, L.ptr(touched), *slots, L.ptr(counters), None,
                      L.ptr(keep), stream), 'preprocess')
        assert int(counters.sum()) == int(touched.sum())
        return touched, keep
    offsets = torch.empty(P, dtype=torch.int32, device=device)
    touched, kept = masks(lib.fsgs_gs_2d_view_preprocess, L.ptr(offsets))
    large = touched > 32
    assert int(large.sum()) > P // 4 and bool((kept[large] == -1).all())
    assert torch.equal(masks(lib.fsgs_gs_2d_view_preprocess, None)[1], kept)
    windows = masks(lib.fsgs_gs_2d_view_preprocess_no_backward)[1]
    assert torch.equal(windows[~large], kept[~large]) and int((windows[large] != -1).sum()) > P // 8
