"""Lists of small views, gathered tile by tile (fsgs_gs_view_gather, fsgs_gs_view_place): against lists formed on the host from the same
rectangles, keep masks and depths, and, on both sides of the limits of fsgs_gs_view_gathers, against the operators' binning."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _window(word, xs, ys, w, h):
    """Which tiles of a w x h rectangle of more than 32 tiles its word keeps: column, row, column + row and column - row + h - 1, each
    from a first to a last sixteenth of its n values (four bits for 15 less the first sixteenth, then four for the last)."""
    kept = np.ones(len(xs), bool)
    for shift, at, n in ((0, xs, w), (8, ys, h), (16, xs + ys, w + h - 1), (24, xs - ys + h - 1, w + h - 1)):
        first, last = 15 - (int(word) >> shift & 15), int(word) >> shift + 4 & 15
        kept &= (at >= -(-first * n // 16)) & (at < -(-(last + 1) * n // 16))
    return kept


def _host_lists(rects, masks, depths, gx, gy):
    """(tile, depth, number) of every kept pair in order, and the ranges."""
    tiles, numbers = [], []
    for i, (x0, y0, x1, y1) in enumerate(rects):
        w, h = x1 - x0, y1 - y0
        ys, xs = np.divmod(np.arange(w * h), max(w, 1))
        if masks is not None:
            kept = (masks[i] >> np.arange(w * h)) & 1 if w * h <= 32 else _window(masks[i], xs, ys, w, h)
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


# windows of large rectangles as views without a backward get them: sides around 16 tiles (from 17 on a sixteenth holds several), one row
# or column, the whole picture; first and last sixteenths in any order (no tile where the last comes first), and around each other
@pytest.mark.parametrize('P,gx,gy', [(300, 33, 1), (300, 1, 127), (600, 17, 16), (600, 18, 15), (900, 33, 31), (700, 127, 16), (800, 45, 45)])
def test_windows_of_large_rectangles(P, gx, gy, device):
    print(f'[small view] windows P={P} {gx}x{gy}', flush=True)
    g = np.random.default_rng(P + gx)
    x0, y0 = g.integers(0, gx, P), g.integers(0, gy, P)
    x1, y1 = x0 + 1 + g.integers(0, gx, P) % (gx - x0), y0 + 1 + g.integers(0, gy, P) % (gy - y0)
    x0[::3], y0[::3], x1[::3], y1[::3] = 0, 0, gx, gy
    rects = np.stack([x0, y0, x1, y1], 1)
    assert ((x1 - x0) * (y1 - y0) > 32).sum() >= P // 3
    masks = g.integers(0, 2 ** 32, P, dtype=np.uint32)  # half of the intervals empty, and so most windows
    wide = g.random(P) < 0.7
    a, b = np.sort(g.integers(0, 16, (2, P, 4)), axis=0)
    word = sum((((15 - a[:, k]) | b[:, k] << 4) << 8 * k).astype(np.uint32) for k in range(4))
    masks[wide] = word[wide]
    masks[::11], masks[5::11] = 0xffffffff, 0
    depths = np.round(g.random(P) * 50, 0).astype(np.float32) + 0.25
    want, ranges = _host_lists(rects, masks, depths, gx, gy)
    whole = len(_host_lists(rects, None, depths, gx, gy)[0])
    assert 0 < len(want) < 0.9 * whole
    got, got_ranges = _gather(rects, masks, depths, gx, gy, len(want), device)
    assert np.array_equal(got_ranges, ranges) and np.array_equal(got, want)


def _preprocessed(kind, P, W, H, seed, scale, thin, device):
    """A view's preprocess without a backward by its C entry, with the rectangles in words and without: what the binning reads of it."""
    import math

    from fast_sp_gs_amd import lib as L, scenes
    lib, stream = L.load(), L.current_stream()
    g = torch.Generator().manual_seed(seed)
    s = scenes._surfels(g, P, 'cube', scale, 0.7, 0.0, 1.5)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])).to(device)
    scales = torch.cat([s.scales, s.scales[:, :1] * 0.5], 1) if kind == 'gaussian' else s.scales.clone()
    scales[:, 0] *= torch.exp(-thin * torch.rand(P, generator=g))
    s.opacities[::7] = 0.0039  # below 1/255: no tile
    s, scales = s.to(device), scales.to(device)
    tan = (math.tan(math.radians(25.0)), math.tan(math.radians(25.0)) * H / W)

    def run(with_rects):
        f = lambda *shape, dtype=torch.float32: torch.zeros(shape, dtype=dtype, device=device)
        out = dict(means2D=f(P, 2), depths=f(P), radii=f(P, dtype=torch.int32), masks=f(P, dtype=torch.int32),
                   counters=f(65, dtype=torch.int64), rects=f((P + 255) // 256 * 256, dtype=torch.int32),
                   word=torch.zeros(1, dtype=torch.int64, pin_memory=True))
        extra = (L.ptr(out['rects']), out['word'].data_ptr()) if with_rects else (None, None)
        colors = f(P, 3)
        if kind == 'surfel':
            trans, normal_opacity, touched = f(P, 9), f(P, 4), f(P, dtype=torch.int32)
            rc = lib.fsgs_gs_2d_view_preprocess_no_backward_rects(
                P, W, H, 3, 16, L.ptr(s.means3D), L.ptr(scales), L.ptr(s.rotations), L.ptr(s.opacities), L.ptr(s.shs), None, L.ptr(cam.Tw2v),
                L.ptr(cam.Tv2c), L.ptr(cam.campos), None, L.ptr(out['means2D']), L.ptr(colors), L.ptr(trans), L.ptr(normal_opacity),
                L.ptr(out['depths']), L.ptr(out['radii']), None, L.ptr(touched), L.ptr(out['counters']), None, L.ptr(out['masks']), *extra,
                stream)
        else:
            cov, conic = f(P, 6), f(P, 4)
            rc = lib.fsgs_gs_view_preprocess_derivs(
                P, W, H, 3, 16, 0, L.ptr(s.means3D), L.ptr(scales), L.ptr(s.rotations), L.ptr(s.opacities), L.ptr(s.shs), None,
                L.ptr(cam.Tw2v), L.ptr(cam.Tv2c), L.ptr(cam.campos), *tan, None, None, None, 0, L.ptr(out['means2D']), L.ptr(out['depths']),
                L.ptr(colors), L.ptr(out['radii']), None, L.ptr(out['counters']), L.ptr(cov), L.ptr(conic), L.ptr(out['masks']), None, *extra,
                stream)
        L.check(rc, 'preprocess')
        torch.cuda.synchronize()
        return out

    return run(True), run(False)


# windows as the preprocess kernel of the surfels leaves them, the Gaussians' masks, and both without masks: the scenes of the windows' own
# tests, where they are gathered, and small footprints
@pytest.mark.parametrize('P,W,H,scale,thin', [(500, 113, 67, -1.6, 2.5), (400, 640, 353, -1.4, 3.5), (257, 511, 1003, -0.8, 5.0), (200, 1601, 97, 0.3, 3.0),
                                              (1, 801, 601, -1.0, 6.0), (900, 801, 601, -1.0, 4.0), (20_001, 333, 211, -4.2, 0.0)])
@pytest.mark.parametrize('masked', [True, False])
@pytest.mark.parametrize('kind', ['surfel', 'gaussian'])
def test_gathered_or_scattered(kind, masked, P, W, H, scale, thin, device):
    from fast_sp_gs_amd import lib as L
    lib, stream = L.load(), L.current_stream()
    print(f'[small view] gathered or scattered: {kind} P={P} {W}x{H} masked={masked}', flush=True)
    assert lib.fsgs_gs_view_gathers(P, W, H)
    a, b = _preprocessed(kind, P, W, H, P + W, scale, thin, device)
    for k in ('means2D', 'depths', 'radii', 'masks'):
        assert torch.equal(a[k], b[k]), k
    T = ((W + 15) // 16) * ((H + 15) // 16)
    masks = lambda o: L.ptr(o['masks']) if masked else None
    bytes_of = lambda n: torch.empty(max(int(n), 1), dtype=torch.uint8, device=device)
    lists_of = lambda n: (torch.full((T, 2), -1, dtype=torch.int64, device=device), torch.full((n,), -5, dtype=torch.int32, device=device))
    # scattered
    bins, word = bytes_of(lib.fsgs_gs_prepare_bins_bytes(P, W, H)), torch.zeros(1, dtype=torch.int64, pin_memory=True)
    regions = [torch.empty(64, dtype=torch.int32, device=device) for _ in range(2)]
    ranges = torch.empty(T, 2, dtype=torch.int64, device=device)
    args = (P, W, H, L.ptr(b['means2D']), None, L.ptr(b['depths']), None, L.ptr(b['radii']), masks(b))
    L.check(lib.fsgs_gs_view_count(P, W, H, L.ptr(b['means2D']), None, None, L.ptr(b['radii']), masks(b), L.ptr(b['counters']),
                                   L.ptr(regions[1]), word.data_ptr(), L.ptr(ranges), L.ptr(bins), bins.numel(), stream), 'count')
    L.check(lib.fsgs_gs_view_wait(word.data_ptr(), stream), 'wait')
    R = int(word[0])
    assert int(a['word'][0]) == R > 0 and not b['counters'].any()
    want = torch.full((R,), -5, dtype=torch.int32, device=device)
    space = bytes_of(lib.fsgs_gs_view_lists_workspace_bytes(R))
    L.check(lib.fsgs_gs_view_scatter(*args, R, L.ptr(ranges), L.ptr(bins), bins.numel(), L.ptr(space), space.numel(), stream), 'scatter')
    L.check(lib.fsgs_gs_view_sort(*args, R, R, L.ptr(ranges), L.ptr(want), L.ptr(bins), bins.numel(), L.ptr(space), space.numel(), stream), 'sort')
    # gathered
    lists, space = bytes_of(lib.fsgs_gs_view_gather_bytes(W, H)), bytes_of(8 * R)
    got_ranges, got = lists_of(R)
    L.check(lib.fsgs_gs_view_gather(P, W, H, L.ptr(a['depths']), L.ptr(a['rects']), masks(a), L.ptr(a['counters']), L.ptr(regions[0]), None,
                                    L.ptr(lists), lists.numel(), stream), 'gather')
    L.check(lib.fsgs_gs_view_place(P, W, H, L.ptr(a['depths']), L.ptr(a['rects']), masks(a), R, L.ptr(got_ranges), L.ptr(got), L.ptr(lists),
                                   lists.numel(), L.ptr(space), space.numel(), stream), 'place')
    torch.cuda.synchronize()
    assert not a['counters'].any() and torch.equal(*regions)
    assert torch.equal(got_ranges, ranges) and torch.equal(got, want)
    kept = int((ranges[:, 1] - ranges[:, 0]).sum())
    if masked and kind == 'surfel' and thin and P > 1:
        words = a['masks'].cpu().numpy().view(np.uint32)
        r = a['rects'].cpu().numpy().view(np.uint32)[:P].astype(int)
        w, h = 128 - (r >> 8 & 127) - (r & 127), 128 - (r >> 24) - (r >> 16 & 127)
        assert ((w * h > 32) & (words != 0) & (words != 0xffffffff)).sum() > P // 40 and kept < R  # there are windows


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


@pytest.mark.parametrize('gx,gy,P,small', [(40, 51, 900, True), (41, 50, 900, False), (127, 3, 500, True), (128, 3, 500, False),
                                           (41, 25, 46_829, True), (41, 25, 46_830, False), (5, 7, 7000, True), (5, 7, 7001, False)])
@pytest.mark.parametrize('cull', [False, True])
def test_gaussian_views_at_the_limits(gx, gy, P, small, cull, device, monkeypatch):
    import math

    from fast_sp_gs_amd import lib as L, scenes
    from fast_sp_gs_amd._C import get_C_function
    from fast_sp_gs_amd.renderer import gaussian_render as m
    print(f'[small view] Gaussian limits {gx}x{gy} P={P} cull={cull}', flush=True)
    W, H = 16 * gx - 3, 16 * gy - 5
    assert bool(L.load().fsgs_gs_view_gathers(P, W, H)) == small
    s = scenes._surfels(torch.Generator().manual_seed(P), P, 'cube', -3.5 if P < 10_000 else -4.5, 0.7, 0.0, 1.5).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    scales, tan = torch.cat([s.scales, s.scales[:, :1]], 1), (math.tan(math.radians(25.0)), math.tan(math.radians(25.0)) * H / W)
    monkeypatch.setattr(m, 'CULL_LISTS', cull)
    m2, depths, _, radii, touched, _, conic = get_C_function('gs_preprocess_forward')(
        W, H, 3, False, s.means3D, scales, s.rotations, s.opacities, s.shs, None, cam.Tw2v, cam.Tv2c, cam.campos, tan, None, None, None, None)
    masks = get_C_function('gs_cull_masks')(W, H, m2, conic, radii) if cull else None
    want = get_C_function('GS_prepare')(W, H, m2, depths, radii, touched, False, cull=cull, keep_masks=masks)[:2]
    for grad in (False, True):
        b = m.render(cam.Tw2v, cam.Tv2c, (W, H), s.means3D.requires_grad_(grad), s.opacities, scales, s.rotations, campos=cam.campos,
                     FoV=tuple(2 * math.atan(t) for t in tan), sh_degree=3, sh_features=s.shs)['buffer']
        assert torch.equal(b.tile_ranges, want[0])
        kept = int((want[0][:, 1] - want[0][:, 0]).sum())
        assert torch.equal(b.point_list[:kept], want[1][:kept]) and b.R == int(touched.sum())


# no memory for the lists (4 KB a tile): binned as larger views are. No memory for the workspace that is allocated ahead of the count (128
# bytes a point): the count is waited for. P, grid, the sizes above 1 MB that the view allocates besides
@pytest.mark.parametrize('P,gx,gy,refused', [(500, 40, 51, 'lists'), (60_000, 32, 32, 'workspace')])
def test_views_that_memory_does_not_suffice_for(P, gx, gy, refused, device):
    """The allocator is left with free blocks of the sizes that the view needs and none for what is to be refused, which is larger."""
    from fast_sp_gs_amd import lib as L, scenes
    from fast_sp_gs_amd.renderer import gaussian_render as m
    lib = L.load()
    W, H = 16 * gx - 3, 16 * gy - 5
    assert lib.fsgs_gs_view_gathers(P, W, H)
    s = scenes._surfels(torch.Generator().manual_seed(P), P, 'cube', -3.5 if P < 10_000 else -5.5, 0.5, 0.0, 1.5).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    scales = torch.cat([s.scales, s.scales[:, :1]], 1)
    MB = 2 ** 20
    slab, keep, image, space = 12 * (P + 256) + lib.fsgs_gs_view_gather_bytes(W, H), 36 * P, 12 * W * H, 128 * P
    needed = [keep, image, 4 * W * H, 4 * W * H, lib.fsgs_gs_prepare_bins_bytes(P, W, H) + 8 * P if refused == 'lists' else slab]
    needed = [(n + 4096 + 511) // 512 * 512 for n in needed if n > MB - 8192]
    assert max(needed) < (slab if refused == 'lists' else space) < 10 * MB

    def view():
        with torch.no_grad():
            return m.render(cam.Tw2v, cam.Tv2c, (W, H), s.means3D, s.opacities, scales, s.rotations, campos=cam.campos, FoV=(0.8, 0.8),
                            sh_degree=3, sh_features=s.shs)

    def refusals():
        return torch.cuda.memory_stats().get('num_ooms', 0)

    before = refusals()
    out = view()
    want, lists = {k: out[k].clone() for k in ('images', 'opacity', 'radii')}, out['buffer'].point_list.clone()
    kept = int((out['buffer'].tile_ranges[:, 1] - out['buffer'].tile_ranges[:, 0]).sum())
    assert refusals() == before and 8 * out['buffer'].R < MB and kept > 0
    del out
    total = torch.cuda.get_device_properties(device).total_memory
    limit = lambda room: torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room * MB) / total)
    filled, blocks = [], []
    try:
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        limit(0)
        for size in (2 ** 28, 2 ** 26, 2 ** 24, 2 ** 22, MB + 1):  # what other tests have left free between their tensors
            try:
                while True:
                    filled.append(torch.empty(size, dtype=torch.uint8, device=device))
            except torch.OutOfMemoryError:
                pass
        limit(400)
        for n in needed:  # a segment of 20 MB each, what is behind the block in use
            blocks.append(torch.empty(n, dtype=torch.uint8, device=device))
            filled.append(torch.empty(20 * MB - n, dtype=torch.uint8, device=device))
            assert filled[-1].data_ptr() == blocks[-1].data_ptr() + n
        limit(19)  # segments of 2 MB, for what is smaller, and no other
        blocks.clear()
        print(f'[small view] {refused} refused: P={P} {gx}x{gy}', flush=True)
        before = refusals()
        out = view()
        torch.cuda.synchronize()
        assert refusals() == before + 1
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for k, v in want.items():
        assert torch.equal(out[k], v), k
    assert torch.equal(out['buffer'].point_list[:kept], lists[:kept])
