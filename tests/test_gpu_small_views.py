"""Lists of small views, gathered tile by tile (fsgs_gs_view_gather, fsgs_gs_view_place): against lists formed on the host from the same
rectangles, keep masks and depths, and, on both sides of the limits of fsgs_gs_view_gathers, against the operators' binning."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _host_lists(rects, masks, depths, gx, gy):
    """(tile, depth, number) of every kept pair in order, and the ranges."""
    tiles, numbers = [], []
    for i, (x0, y0, x1, y1) in enumerate(rects):
        w, h = x1 - x0, y1 - y0
        ys, xs = np.divmod(np.arange(w * h), max(w, 1))
        if masks is not None:
            kept = (masks[i] >> np.arange(w * h)) & 1 if w * h <= 32 else np.full(w * h, masks[i] != 0)
            ys, xs = ys[kept != 0], xs[kept != 0]
        tiles.append((y0 + ys) * gx + x0 + xs)
        numbers.append(np.full(len(xs), i))
    tiles, numbers = np.concatenate(tiles), np.concatenate(numbers)
    order = np.lexsort((numbers, depths.view(np.uint32)[numbers], tiles))
    tiles, numbers = tiles[order], numbers[order]
    ends = np.searchsorted(tiles, np.arange(gx * gy), side='right')
    starts = np.searchsorted(tiles, np.arange(gx * gy), side='left')
    ranges = np.stack([starts, ends], 1)
    ranges[starts == ends] = 0
    return numbers.astype(np.int32), ranges


def _gather(rects, masks, depths, gx, gy, R, device):
    from fast_sp_gs_amd import lib as L
    lib, stream = L.load(), L.current_stream()
    P, W, H = len(rects), 16 * gx - 3, 16 * gy - 5
    assert lib.fsgs_gs_view_gathers(P, W, H)
    x0, y0, x1, y1 = rects.T
    words = np.where((x1 > x0) & (y1 > y0), x0 | (128 - x1) << 8 | y0 << 16 | (128 - y1) << 24, 0x7f7f7f7f)
    words = np.concatenate([words, np.full(-P % 256, 0x7f7f7f7f)]).astype(np.uint32)
    at = lambda a: torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).to(device)
    d_words, d_depths, d_masks = at(words), at(depths), None if masks is None else at(masks.astype(np.uint32))
    counters = torch.zeros(64, dtype=torch.int64, device=device)
    counters[3], counters[62] = R - 1, 1
    regions = torch.empty(64, dtype=torch.int32, device=device)
    word = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    lists = torch.full((lib.fsgs_gs_view_gather_bytes(W, H),), 0xab, dtype=torch.uint8, device=device)
    ranges = torch.full((gx * gy, 2), -1, dtype=torch.int64, device=device)
    point_list = torch.full((R,), -5, dtype=torch.int32, device=device)
    space = torch.empty(8 * R, dtype=torch.uint8, device=device)
    L.check(lib.fsgs_gs_view_gather(P, W, H, L.ptr(d_depths), L.ptr(d_words), L.ptr(d_masks), L.ptr(counters), L.ptr(regions),
                                    word.data_ptr(), L.ptr(lists), lists.numel(), stream), 'gather')
    L.check(lib.fsgs_gs_view_wait(word.data_ptr(), stream), 'wait')
    assert int(word[0]) == R and not counters.any() and regions[4:63].eq(R - 1).all() and not regions[:4].any()
    L.check(lib.fsgs_gs_view_place(P, W, H, L.ptr(d_depths), L.ptr(d_words), L.ptr(d_masks), R, L.ptr(ranges), L.ptr(point_list),
                                   L.ptr(lists), lists.numel(), L.ptr(space), space.numel(), stream), 'place')
    return point_list.cpu().numpy(), ranges.cpu().numpy()


# numbers of surfels around a quad of words, a go of a wavefront and of a block, two of a block and the most; grids of one tile, one row
# or column as long as a word's bounds allow, and around the tiles per block of the second launch
@pytest.mark.parametrize('P,gx,gy', [(1, 1, 1), (3, 1, 127), (255, 127, 1), (256, 15, 17), (257, 16, 16), (1023, 30, 17), (1025, 73, 7),
                                     (4095, 32, 32), (4097, 20, 51), (8193, 1021, 1), (5000, 40, 51), (2049, 127, 16), (65_535, 19, 18)])
@pytest.mark.parametrize('masked', [False, True])
def test_lists_from_rectangles(P, gx, gy, masked, device):
    print(f'[small view] P={P} {gx}x{gy} masked={masked}', flush=True)
    if gx > 127:  # not for this path
        from fast_sp_gs_amd import lib as L
        assert not L.load().fsgs_gs_view_gathers(P, 16 * gx, 16 * gy)
        return
    g = np.random.default_rng(P + gx)
    x0, y0 = g.integers(0, gx, P), g.integers(0, gy, P)
    x1, y1 = np.minimum(gx, x0 + g.integers(0, 5, P)), np.minimum(gy, y0 + g.integers(1, 5, P))
    x0[::97], y0[::97], x1[::97], y1[::97] = 0, 0, gx, gy  # a few over the whole picture
    rects = np.stack([x0, y0, x1, y1], 1)
    # as the preprocess kernel leaves them: a bit per tile, or, above 32 tiles, a window, here all of the rectangle or nothing
    masks = g.integers(0, 2 ** 32, P, dtype=np.uint32) if masked else None
    if masked:
        big = (x1 - x0) * (y1 - y0) > 32
        masks[big] = np.where(g.random(big.sum()) < 0.8, 0xffffffff, 0)
    depths = np.round(g.random(P) * 200, 0).astype(np.float32) + 0.25  # many at the same depth
    want, ranges = _host_lists(rects, masks, depths, gx, gy)
    R = max(len(want), 1) + 3
    got, got_ranges = _gather(rects, masks, depths, gx, gy, R, device)
    assert np.array_equal(got_ranges, ranges) and np.array_equal(got[:len(want)], want) and (got[len(want):] == -5).all()


# lists that their own blocks cannot sort: around 2048 entries, above 4096, 8192 and 16 384, beside short ones
@pytest.mark.parametrize('P,gx,gy', [(2048, 11, 1), (2049, 1, 11), (2500, 16, 16), (5000, 5, 5), (9000, 30, 40), (17_000, 10, 9), (20_000, 25, 30),
                                     (65_535, 20, 20)])
@pytest.mark.parametrize('one_depth', [False, True])
def test_long_lists(P, gx, gy, one_depth, device):
    print(f'[small view] long lists P={P} {gx}x{gy} one_depth={one_depth}', flush=True)
    g = np.random.default_rng(P)
    tx, ty = g.integers(0, gx, P), g.integers(0, gy, P)
    rects = np.stack([tx, ty, tx + 1, ty + 1], 1)
    rects[g.random(P) < 0.97] = (gx // 2, gy // 2, gx // 2 + 1, gy // 2 + 1)  # nearly all in one tile, that and its neighbour
    rects[::2, 2] = np.minimum(gx, rects[::2, 2] + 1)
    if P == 2048:  # as long as a block sorts, twice
        rects[:] = (3, 0, 5, 1)
    depths = np.full(P, 7.5, np.float32) if one_depth else g.random(P).astype(np.float32) + 0.2
    want, ranges = _host_lists(rects, None, depths, gx, gy)
    got, got_ranges = _gather(rects, None, depths, gx, gy, len(want), device)
    assert np.array_equal(got_ranges, ranges) and np.array_equal(got, want)


# the last sizes that are gathered and the first that are not: by tiles, by numbers, by both
@pytest.mark.parametrize('gx,gy,P,small', [(40, 51, 900, True), (41, 50, 900, False), (127, 3, 500, True), (128, 3, 500, False),
                                           (32, 32, 65_535, True), (32, 32, 65_536, False), (41, 25, 46_829, True), (41, 25, 46_830, False),
                                           (5, 7, 7000, True), (5, 7, 7001, False)])
@pytest.mark.parametrize('cull', [False, True])
def test_views_at_the_limits(gx, gy, P, small, cull, device, monkeypatch):
    from fast_sp_gs_amd import lib as L, scenes
    from fast_sp_gs_amd._C import get_C_function
    from fast_sp_gs_amd.renderer import gs_2d_render as m
    print(f'[small view] limits {gx}x{gy} P={P} cull={cull}', flush=True)
    W, H = 16 * gx - 3, 16 * gy - 5
    assert bool(L.load().fsgs_gs_view_gathers(P, W, H)) == small
    s = scenes._surfels(torch.Generator().manual_seed(P), P, 'cube', -3.5 if P < 10_000 else -4.5, 0.7, 0.0, 1.5).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    monkeypatch.setattr(m, 'CULL_LISTS', cull)
    pre = get_C_function('gs_2d_preprocess_forward')(W, H, 3, False, s.means3D, s.scales, s.rotations, s.opacities, s.shs, None, cam.Tw2v,
                                                     cam.Tv2c, cam.campos, None, None, None, return_records=True, return_masks=True)
    m2, depths, radii, touched, masks = pre[0], pre[4], pre[5], pre[6], pre[8]
    if cull:
        want = get_C_function('GS_prepare')(W, H, m2, depths, radii, touched, False, cull=True, keep_masks=masks)[:2]
    else:
        want = get_C_function('GS_prepare')(W, H, m2, depths, radii, touched, False)[:2]
    b = m.GS_2D_render(s.means3D.requires_grad_(True), s.scales, s.rotations, s.opacities, (W, H), cam.Tw2v, cam.Tv2c, campos=cam.campos,
                       sh_degree=3, near=0.2, far=100.0, sh_features=s.shs)['buffer']
    assert torch.equal(b.tile_ranges, want[0])
    kept = int((want[0][:, 1] - want[0][:, 0]).sum())
    assert torch.equal(b.point_list[:kept], want[1][:kept]) and b.R == int(touched.sum())
