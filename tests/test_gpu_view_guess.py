"""A view's instances are scattered for a guessed count before the count is known (instances_to_guess in
csrc/host/torch_util.hpp: 16 per surfel, 65 536 at least, one per surfel and tile at most). Scenes with more instances than that
are scattered again: the same maps, lists, counts and gradients as by the operators, which wait for the count. Nothing that a
view hands out or keeps is sized by the guess."""
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


# The surfels' and Gaussians' views of the sizes above are gathered tile by tile and need no guess (their lists' workspace is sized
# by one, too, and made anew). Beyond those limits: grids of more than 127 columns, 1280 and 512 tiles, and more than 200 points a tile
@pytest.mark.parametrize('P,W,H,more', [(700, 2048, 160, True), (900, 2048, 64, True), (20_001, 160, 160, True), (1, 2048, 64, False)])
@pytest.mark.parametrize('which', ['surfel', 'gaussian'])
def test_more_instances_than_guessed_beyond_small_views(which, P, W, H, more, device, monkeypatch):
    from fast_sp_gs_amd import lib as L
    assert not L.load().fsgs_gs_view_gathers(P, W, H)
    test_more_instances_than_guessed(which, P, W, H, more, device, monkeypatch)


def _view(s, cam):
    from fast_sp_gs_amd.renderer import GS_2D_render
    with torch.no_grad():
        return GS_2D_render(s.means3D, s.scales, s.rotations, s.opacities, (cam.W, cam.H), cam.Tw2v, cam.Tv2c,
                            campos=cam.campos, sh_degree=3, sh_features=s.shs)


def _time(f):
    """Microseconds a call: the best of five times 10."""
    best = float('inf')
    for _ in range(6):  # the first one warms up
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(10):
            f()
        end.record()
        end.synchronize()
        best = min(best, start.elapsed_time(end) * 1000 / 10)
    return best


@pytest.mark.parametrize('P,W,H,log_scale', [(20_000, 256, 256, -4.6), (900, 480, 288, 0.3), (1, 480, 288, -3.0),
                                             (60_000, 272, 272, -4.6), (900, 2048, 64, 0.3), (1, 2048, 64, -3.0)])  # the last three: not gathered
@pytest.mark.parametrize('train', [False, True])
def test_lists_are_no_longer_than_the_count(P, W, H, log_scale, train, device):
    """Kept, or saved to a file, a list takes the memory of its entries."""
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd.renderer import GS_2D_render
    s = scenes._surfels(torch.Generator().manual_seed(P), P, 'cube', log_scale, 0.3, -1.0, 1.0).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.3, 0.2, 4.0])).to(device)
    out = GS_2D_render(s.means3D.requires_grad_(train), s.scales, s.rotations, s.opacities, (W, H), cam.Tw2v, cam.Tv2c,
                       campos=cam.campos, sh_degree=3, sh_features=s.shs)
    point_list = out['buffer'].point_list
    assert point_list.untyped_storage().nbytes() == point_list.nbytes == 4 * out['buffer'].R


def test_exceeded_guess_costs_an_empty_launch(device):
    """The same 900 large surfels with as many small ones behind the camera as raise the guess above the count: without them the
    counting, and all behind it, ran twice (1.5 times the time). Both views are gathered tile by tile; for grids that are not, see below."""
    s, cam, g = _large_surfels(900, 480, 288, 901)
    more = type(s)(*(torch.cat([t, t[torch.randint(900, (30_000,), generator=g)]])
                     for t in (s.means3D, s.scales, s.rotations, s.opacities, s.shs)), s.sh_degree)
    more.means3D[900:, 2] = 50.0
    s, more, cam = s.to(device), more.to(device), cam.to(device)
    a, b = _view(s, cam), _view(more, cam)
    assert 65_536 < a['buffer'].R <= 16 * 30_900 and a['buffer'].R == b['buffer'].R and torch.equal(a['images'], b['images'])
    assert _time(lambda: _view(s, cam)) < 1.25 * _time(lambda: _view(more, cam))


def test_exceeded_guess_costs_an_empty_launch_beyond_small_views(device):
    """As above on a grid that is not gathered, with opacities that leave each surfel a small part of its rectangle (which is what is counted):
    the time is the binning's, not the blend's."""
    from fast_sp_gs_amd import lib as L
    s, cam, g = _large_surfels(900, 2048, 64, 901)
    s.opacities.fill_(0.0045)
    more = type(s)(*(torch.cat([t, t[torch.randint(900, (30_000,), generator=g)]])
                     for t in (s.means3D, s.scales, s.rotations, s.opacities, s.shs)), s.sh_degree)
    more.means3D[900:, 2] = 50.0
    assert not L.load().fsgs_gs_view_gathers(900, 2048, 64) and not L.load().fsgs_gs_view_gathers(30_900, 2048, 64)
    s, more, cam = s.to(device), more.to(device), cam.to(device)
    a, b = _view(s, cam), _view(more, cam)
    assert 65_536 < a['buffer'].R <= 16 * 30_900 and a['buffer'].R == b['buffer'].R and torch.equal(a['images'], b['images'])
    turns = [(_time(lambda: _view(s, cam)), _time(lambda: _view(more, cam))) for _ in range(3)]
    took, with_room = (min(t) for t in zip(*turns))
    print(f'[exceeded guess] {took:.1f} us, with room {with_room:.1f}', flush=True)
    assert took < 1.35 * with_room  # 90 and 77: an empty launch, and one that the host's answer to the count is waited for


def test_guess_that_memory_does_not_suffice_for(device):
    """A view for whose guess there is no memory waits for its count: it needs no more than that."""
    g = torch.Generator().manual_seed(3)
    from fast_sp_gs_amd import scenes
    s = scenes._surfels(g, 262_144, 'cube', -9.0, 0.1, -1.0, 1.0).to(device)
    cam = scenes.pinhole(256, 256, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    want, total = _view(s, cam)['images'], torch.cuda.get_device_properties(device).total_memory
    busy = torch.ones(2 ** 28, device=device)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    base, tried, filled = torch.cuda.memory_reserved(), False, []
    try:
        torch.cuda.set_per_process_memory_fraction(base / total)
        for size in (2 ** 28, 2 ** 26, 2 ** 24, 2 ** 22, 2 ** 20 + 1):  # what other tests have left free between their tensors
            try:
                while True:
                    filled.append(torch.empty(size, dtype=torch.uint8, device=device))
            except torch.OutOfMemoryError:
                pass
        for room in range(160, 0, -4):  # MB
            torch.cuda.set_per_process_memory_fraction((base + room * 2 ** 20) / total)
            failed = torch.cuda.memory_stats().get('num_ooms', 0)
            for _ in range(30):  # some milliseconds: the count is not there before the guess
                busy.mul_(1.0)
            try:
                got = _view(s, cam)['images']
            except torch.OutOfMemoryError:
                break
            finally:
                torch.cuda.synchronize()
                torch.cuda.empty_cache()
            assert torch.equal(got, want)
            tried |= torch.cuda.memory_stats().get('num_ooms', 0) > failed
            del got
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert tried


# grids whose ranges one block forms, several do, and beyond the tiles that LDS counters serve
@pytest.mark.parametrize('gx,gy,P', [(30, 18, 3000), (64, 64, 3000), (17, 2410, 300)])
def test_scatter_without_room_writes_nothing(gx, gy, P, device):
    """The C entries with a guess that is too small: nothing is written, and the scatter for the count leaves the lists of
    `GS_prepare`."""
    from fast_sp_gs_amd import lib as L, scenes
    from fast_sp_gs_amd._C import get_C_function
    lib, stream = L.load(), L.current_stream()
    W, H = 16 * gx - 3, 16 * gy - 5
    scene, _ = scenes.config0(P=P, size=max(W, H), seed=4)
    scene.scales = scene.scales * 20.0
    s, cam = scene.to(device), scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    print(f'[scatter without room] {gx}x{gy} tiles, P={P}', flush=True)
    m2, _, _, _, depths, radii, touched = get_C_function('gs_2d_preprocess_forward')(
        W, H, 3, False, s.means3D, s.scales, s.rotations, s.opacities, s.shs, None, cam.Tw2v, cam.Tv2c, cam.campos, None, None, None)
    want_ranges, want_list = get_C_function('GS_prepare')(W, H, m2, depths, radii, touched, False)[:2]
    R = int(touched.sum())
    assert R == want_list.numel() > P
    counters = torch.zeros(64, dtype=torch.int64, device=device)
    counters[5], counters[63] = R - 7, 7
    word = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    ranges = torch.full((gx * gy, 2), -1, dtype=torch.int64, device=device)
    bins = torch.full((lib.fsgs_gs_prepare_bins_bytes(P, W, H),), 0xff, dtype=torch.uint8, device=device)
    L.check(lib.fsgs_gs_view_count(P, W, H, L.ptr(m2), None, None, L.ptr(radii), None, L.ptr(counters), None, word.data_ptr(),
                                   L.ptr(ranges), L.ptr(bins), bins.numel(), stream), 'count')
    L.check(lib.fsgs_gs_view_wait(word.data_ptr(), stream), 'wait')
    assert int(word[0]) == R and not counters.any()
    point_list = torch.full((R,), -5, dtype=torch.int32, device=device)
    for room in (1, R // 2, R - 1, R):
        size = lib.fsgs_gs_view_lists_workspace_bytes(room)
        space = torch.full((size + 4096,), 0xab, dtype=torch.uint8, device=device)
        args = (P, W, H, L.ptr(m2), None, L.ptr(depths), None, L.ptr(radii), None)
        L.check(lib.fsgs_gs_view_scatter(*args, room, L.ptr(ranges), L.ptr(bins), bins.numel(), L.ptr(space), size, stream), 'scatter')
        torch.cuda.synchronize()
        assert (room == R and gx * gy <= 40_960) != bool((space == 0xab).all()) and bool((space[size:] == 0xab).all())
        rc = lib.fsgs_gs_view_sort(*args, R, room, L.ptr(ranges), L.ptr(point_list), L.ptr(bins), bins.numel(), L.ptr(space),
                                   size, stream)
        assert (rc == 0) == (room == R)
    torch.cuda.synchronize()
    assert torch.equal(ranges, want_ranges) and torch.equal(point_list, want_list) and bool((space[size:] == 0xab).all())


# around the grids whose ranges one block forms (1024 tiles, 65 536 surfels), the scatter itself, and a kernel of its own (from
# 4097 tiles on); the last tile of a lane's four, and grids that end inside them
@pytest.mark.parametrize('gx,gy,P', [(32, 32, 65_536), (32, 32, 65_537), (25, 41, 900), (61, 67, 2000), (64, 64, 2000), (17, 241, 2000)])
def test_lists_of_a_view_are_the_operators(gx, gy, P, device, monkeypatch):
    from fast_sp_gs_amd import scenes
    from fast_sp_gs_amd._C import get_C_function
    from fast_sp_gs_amd.renderer import gs_2d_render as m
    W, H = 16 * gx - 3, 16 * gy - 5
    s = scenes._surfels(torch.Generator().manual_seed(P), P, 'cube', -3.5 if P < 10_000 else -4.5, 0.7, 0.0, 1.5).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    monkeypatch.setattr(m, 'CULL_LISTS', False)
    m2, _, _, _, depths, radii, touched = get_C_function('gs_2d_preprocess_forward')(
        W, H, 3, False, s.means3D, s.scales, s.rotations, s.opacities, s.shs, None, cam.Tw2v, cam.Tv2c, cam.campos, None, None, None)
    want_ranges, want_list = get_C_function('GS_prepare')(W, H, m2, depths, radii, touched, False)[:2]
    with torch.no_grad():
        for _ in range(2):  # the second view's room is guessed
            b = m.GS_2D_render(s.means3D, s.scales, s.rotations, s.opacities, (W, H), cam.Tw2v, cam.Tv2c, campos=cam.campos,
                               sh_degree=3, near=0.2, far=100.0, sh_features=s.shs)['buffer']
            assert torch.equal(b.tile_ranges, want_ranges) and torch.equal(b.point_list, want_list)


# the same sides of those lines
@pytest.mark.parametrize('gx,gy,P', [(32, 32, 65_536), (32, 32, 65_537), (25, 41, 900), (61, 67, 2000), (64, 64, 2000), (17, 241, 2000)])
def test_operators_end_what_the_count_of_a_view_began(gx, gy, P, device):
    """The C entries: `fsgs_gs_view_count`, then `fsgs_gs_prepare_fill_counted` instead of scatter and sort of a view, twice. The count
    leaves empty ranges where the scatter forms them, which is all there is to do for a view without instances."""
    from fast_sp_gs_amd import lib as L, scenes
    from fast_sp_gs_amd._C import get_C_function
    lib, stream = L.load(), L.current_stream()
    W, H = 16 * gx - 3, 16 * gy - 5
    s = scenes._surfels(torch.Generator().manual_seed(P), P, 'cube', -3.5 if P < 10_000 else -4.5, 0.7, 0.0, 1.5).to(device)
    cam = scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    m2, _, _, _, depths, radii, touched = get_C_function('gs_2d_preprocess_forward')(
        W, H, 3, False, s.means3D, s.scales, s.rotations, s.opacities, s.shs, None, cam.Tw2v, cam.Tv2c, cam.campos, None, None, None)
    want_ranges, want_list = get_C_function('GS_prepare')(W, H, m2, depths, radii, touched, False)[:2]
    bins = torch.full((lib.fsgs_gs_prepare_bins_bytes(P, W, H),), 0xff, dtype=torch.uint8, device=device)
    word = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    for seen in (radii, torch.zeros_like(radii)):
        R = int(touched.sum()) if seen is radii else 0
        counters = torch.zeros(64, dtype=torch.int64, device=device)
        counters[7] = R
        ranges = torch.full((gx * gy, 2), -1, dtype=torch.int64, device=device)
        L.check(lib.fsgs_gs_view_count(P, W, H, L.ptr(m2), None, None, L.ptr(seen), None, L.ptr(counters), None, word.data_ptr(),
                                       L.ptr(ranges), L.ptr(bins), bins.numel(), stream), 'count')
        L.check(lib.fsgs_gs_view_wait(word.data_ptr(), stream), 'wait')
        assert int(word[0]) == R and bool((ranges[:, 0] <= ranges[:, 1]).all())
        space = torch.empty(max(lib.fsgs_gs_prepare_fill_workspace_bytes(R), 1), dtype=torch.uint8, device=device)
        for _ in range(2):
            point_list = torch.full((R,), -5, dtype=torch.int32, device=device)
            L.check(lib.fsgs_gs_prepare_fill_counted(P, W, H, L.ptr(m2), L.ptr(depths), L.ptr(seen), R, L.ptr(ranges), L.ptr(point_list),
                                                     None, L.ptr(bins), bins.numel(), L.ptr(space), space.numel(), stream), 'fill')
            if R:
                assert torch.equal(ranges, want_ranges) and torch.equal(point_list, want_list)
        if not R:
            assert bool((ranges[:, 0] == ranges[:, 1]).all())
