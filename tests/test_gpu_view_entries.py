"""The views' preprocess entry points of the C ABI in their plain forms, which programs outside this package call: the same outputs, bit
for bit, as from the `_derivs` and `_rects` forms that the host layer calls, given null pointers or what they write besides."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# blocks of 256 points that have a region of the record slots each, so that the slots do not depend on which block comes first
SIZES = [(1, 33, 17), (257, 61, 45), (5000, 160, 96)]


def _scene(P, W, H, split, device):
    from fast_sp_gs_amd import scenes
    s, _ = scenes.config0(P=P, size=64, seed=P)
    s.scales = s.scales * 3
    s, cam = s.to(device), scenes.pinhole(W, H, 50.0, torch.tensor([0.0, 0.0, 4.0])).to(device)
    sh = (s.shs[:, :1].clone(memory_format=torch.contiguous_format), s.shs[:, 1:].clone(memory_format=torch.contiguous_format)) if split else (s.shs, None)
    return s, cam, sh, 15 if split else 16


def _run(entry, outputs, call, **more):
    """Calls `entry`; its outputs and what `more` names (allocated here, in the order of the entry's last parameters; None stays null)."""
    from fast_sp_gs_amd import lib as L
    device = 'cuda'
    made = {k: torch.full(shape, 0 if k == 'counters' else 85, dtype=dtype, device=device) for k, (shape, dtype) in outputs.items()}
    extra = {k: None if v is None else torch.zeros(v[0], dtype=v[1], **({'pin_memory': True} if k == 'word' else {'device': device}))
             for k, v in more.items()}
    L.check(call(getattr(L.load(), entry), {k: L.ptr(t) for k, t in made.items()}, [L.ptr(t) for t in extra.values()]), entry)
    torch.cuda.synchronize()
    return made, extra


def _same(a, b):
    for k in a:
        if k != 'counters':
            assert torch.equal(torch.nan_to_num(a[k].float()), torch.nan_to_num(b[k].float())), k


@pytest.mark.parametrize('P,W,H', SIZES)
@pytest.mark.parametrize('split', [False, True])
def test_surfel_view_entries(P, W, H, split, device):
    from fast_sp_gs_amd import lib as L
    lib, p, stream = L.load(), L.ptr, L.current_stream()
    s, cam, (sh, rest), n_sh = _scene(P, W, H, split, device)
    print(f'[view entries] surfels P={P} {W}x{H} split={split}', flush=True)
    f, i = torch.float32, torch.int32
    outputs = dict(means2D=((P, 2), f), colors=((P, 3), f), trans=((P, 9), f), no=((P, 4), f), depths=((P,), f), radii=((P,), i),
                   visible=((P,), torch.uint8), touched=((P,), i), offsets=((P,), i), counters=((65,), torch.int64), records=((P, 20), f),
                   masks=((P,), i))
    front = (P, W, H, 3, n_sh, p(s.means3D), p(s.scales), p(s.rotations), p(s.opacities), p(sh), p(rest), p(cam.Tw2v), p(cam.Tv2c),
             p(cam.campos), None)
    before = lambda o: [o[k] for k in ('means2D', 'colors', 'trans', 'no', 'depths', 'radii', 'visible', 'touched')]
    tail = lambda o: [o[k] for k in ('counters', 'records', 'masks')]
    call = lambda e, o, x: e(*front, *before(o), o['offsets'], *tail(o), *x, stream)
    plain, _ = _run('fsgs_gs_2d_view_preprocess', outputs, call)
    wide, _ = _run('fsgs_gs_2d_view_preprocess_derivs', outputs, call, derivs=None, rects=None, word=None)
    full, extra = _run('fsgs_gs_2d_view_preprocess_derivs', outputs, call, derivs=((P, 9), f), rects=(((P + 255) // 256 * 256,), i),
                       word=((1,), torch.int64))
    _same(plain, wide), _same(plain, full)
    assert torch.equal(plain['counters'], wide['counters']) and int(extra['word'][0]) == int(plain['touched'].sum())
    call = lambda e, o, x: e(*front, *before(o), *tail(o), *x, stream)
    outputs.pop('offsets')
    windows, _ = _run('fsgs_gs_2d_view_preprocess_no_backward', outputs, call)
    wide, _ = _run('fsgs_gs_2d_view_preprocess_no_backward_rects', outputs, call, rects=None, word=None)
    _same(windows, wide)
    # the backward, from records of any values
    R = int(plain['touched'].sum())
    regions = (plain['counters'][:64].cumsum(0) - plain['counters'][:64]).int()
    g = torch.Generator().manual_seed(P)
    records = torch.randn(max(R, 1), 18, generator=g).to(device)
    grads = dict(means2D=((P, 2), f), means3D=((P, 3), f), scales=((P, 2), f), rot=((P, 4), f), opac=((P, 1), f), sh=(tuple(sh.shape), f))
    if split:
        grads['rest'] = (tuple(rest.shape), f)
    call = lambda e, o, x: e(P, W, H, 3, n_sh, p(s.means3D), p(s.scales), p(s.rotations), p(sh), p(rest), p(cam.Tw2v), p(cam.Tv2c),
                             p(cam.campos), p(plain['trans']), p(plain['radii']), p(plain['colors']), p(plain['offsets']), p(regions),
                             p(plain['touched']), None, p(records), *x, *[o[k] for k in ('means2D', 'means3D', 'scales', 'rot', 'opac', 'sh')],
                             o.get('rest'), stream)
    a, _ = _run('fsgs_gs_2d_view_preprocess_backward', grads, call)
    b, _ = _run('fsgs_gs_2d_view_preprocess_backward_derivs', grads, call, derivs=None)
    c, _ = _run('fsgs_gs_2d_view_preprocess_backward_derivs', grads, lambda e, o, x: call(e, o, [p(extra['derivs'])]))
    _same(a, b), _same(a, c)


@pytest.mark.parametrize('P,W,H', SIZES)
@pytest.mark.parametrize('split', [False, True])
def test_fast_surfel_view_entries(P, W, H, split, device):
    from fast_sp_gs_amd import lib as L
    p, stream = L.ptr, L.current_stream()
    s, cam, (sh, rest), n_sh = _scene(P, W, H, split, device)
    print(f'[view entries] fast surfels P={P} {W}x{H} split={split}', flush=True)
    f, i = torch.float32, torch.int32
    outputs = dict(means2D=((P, 2), f), colors=((P, 3), f), trans=((P, 9), f), inverse=((P, 9), f), no=((P, 4), f), depths=((P,), f),
                   radii=((P,), i), visible=((P,), torch.uint8), touched=((P,), i), offsets=((P,), i), counters=((65,), torch.int64),
                   masks=((P,), i))
    call = lambda e, o, x: e(P, W, H, 3, n_sh, p(s.means3D), p(s.scales), p(s.rotations), p(s.opacities), p(sh), p(rest), p(cam.Tw2v),
                             p(cam.Tv2s), p(cam.campos), None, *[o[k] for k in outputs], *x, stream)
    plain, _ = _run('fsgs_gs_2d_fast_view_preprocess', outputs, call)
    wide, _ = _run('fsgs_gs_2d_fast_view_preprocess_derivs', outputs, call, derivs=None)
    full, _ = _run('fsgs_gs_2d_fast_view_preprocess_derivs', outputs, call, derivs=((P, 9), f))
    _same(plain, wide), _same(plain, full)
    assert torch.equal(plain['counters'], wide['counters']) and torch.equal(plain['counters'], full['counters'])


@pytest.mark.parametrize('P,W,H', SIZES)
@pytest.mark.parametrize('split', [False, True])
def test_gaussian_view_entries(P, W, H, split, device):
    from fast_sp_gs_amd import lib as L
    p, stream = L.ptr, L.current_stream()
    s, cam, (sh, rest), n_sh = _scene(P, W, H, split, device)
    print(f'[view entries] Gaussians P={P} {W}x{H} split={split}', flush=True)
    f, i = torch.float32, torch.int32
    scales, tan = torch.cat([s.scales, s.scales[:, :1]], 1), (math.tan(0.4), math.tan(0.4) * H / W)
    outputs = dict(means2D=((P, 2), f), depths=((P,), f), colors=((P, 3), f), radii=((P,), i), visible=((P,), torch.uint8),
                   counters=((65,), torch.int64), cov3D=((P, 6), f), conic=((P, 4), f), masks=((P,), i))
    call = lambda e, o, x: e(P, W, H, 3, n_sh, 0, p(s.means3D), p(scales), p(s.rotations), p(s.opacities), p(sh), p(rest), p(cam.Tw2v),
                             p(cam.Tv2c), p(cam.campos), *tan, None, None, None, 0, *[o[k] for k in outputs], *x, stream)
    plain, _ = _run('fsgs_gs_view_preprocess', outputs, call)
    wide, _ = _run('fsgs_gs_view_preprocess_derivs', outputs, call, derivs=None, rects=None, word=None)
    full, extra = _run('fsgs_gs_view_preprocess_derivs', outputs, call, derivs=((P, 9), f), rects=(((P + 255) // 256 * 256,), i),
                       word=((1,), torch.int64))
    _same(plain, wide), _same(plain, full)
    assert torch.equal(plain['counters'], wide['counters']) and int(extra['word'][0]) == int(plain['counters'].sum())
