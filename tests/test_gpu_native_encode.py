"""The host layer's nodes of the spherical-harmonic operators against the Python operator pairs, which launch the same kernels: the same
values bit for bit, and every call that is not the layer's own (other types, layouts, devices, modes) gets the pair's answer."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(P, F, device, camera=True):
    g = torch.Generator().manual_seed(P + F)
    normal = lambda *s: torch.randn(*s, generator=g).to(device)
    dirs = torch.nn.functional.normalize(normal(P, 3), dim=-1)
    return normal(P, F, 3), normal(P, 3) if camera else dirs, normal(3) * 3 if camera else None, dirs, normal(P, 3)


def _native(out):
    return out.grad_fn is not None and '_KernelNode' not in out.grad_fn.name()


@pytest.mark.parametrize('P', [1, 65, 700])
@pytest.mark.parametrize('degree,F', [(0, 1), (1, 4), (2, 16), (3, 16), (4, 25), (5, 36), (7, 130)])
@pytest.mark.parametrize('camera', [False, True])
def test_same_as_the_pair(P, degree, F, camera, device):
    from fast_sp_gs_amd import ops
    print(f'[native encode] P={P} degree={degree} F={F} camera={camera}', flush=True)
    sh, pos, cam, dirs, up = _inputs(P, F, device, camera)
    for clamp in (True, False):
        for wants in range(1, 8 if camera else 4):
            def run(f):
                p = [sh.clone(), pos.clone(), cam.clone() if camera else None]
                wrt = [t.requires_grad_(True) for k, t in enumerate(p) if t is not None and wants >> k & 1]
                out = f(*p, degree, clamp)
                # the upstream gradient strided, as a transposed loss leaves it
                return out, torch.autograd.grad(out, wrt, up.t().contiguous().t())
            (a, ga), (b, gb) = run(ops.SH_to_RGB), run(ops._rgb_pair)
            assert _native(a) and not _native(b) and torch.equal(a, b)
            for x, y in zip(ga, gb):
                if x.shape == (3,):  # a sum over blocks of 256 points, one atomic each, in any order
                    assert (x - y).abs().max() <= 1e-6 * P ** 0.5 * max(float(y.abs().max()), 1.0)
                else:
                    assert torch.equal(x, y)
    for width in (3, 5):
        d = torch.cat([dirs, dirs], 1)[:, :width].contiguous()
        def run(f):
            x = d.clone().requires_grad_(True)
            out = f(x, degree)
            return out, torch.autograd.grad(out, x, torch.ones(out.shape, device=device) * 0.3)[0]
        (a, ga), (b, gb) = run(ops.sh_encode), run(ops._sh_pair)
        assert _native(a) and torch.equal(a, b) and torch.equal(ga, gb)
    with torch.no_grad():
        assert torch.equal(ops.SH_to_RGB(sh, pos, cam, degree), ops._rgb_pair(sh, pos, cam, degree, True))
        assert torch.equal(ops.sh_encode(dirs, degree), ops._sh_pair(dirs, degree))


def test_calls_of_the_pair(device):
    from fast_sp_gs_amd import ops
    sh, pos, cam, dirs, up = _inputs(130, 16, device)
    ask = lambda t: t.clone().requires_grad_(True)
    # other layouts and types
    strided = ask(sh.permute(2, 1, 0)).permute(2, 1, 0)
    assert torch.equal(ops.SH_to_RGB(strided, pos, cam, 3), ops.SH_to_RGB(sh, pos, cam, 3))
    assert ops.sh_encode(ask(dirs.double()), 3).dtype == torch.float64
    assert ops.sh_encode(ask(dirs).reshape(13, 10, 3), 2).shape == (13, 10, 9)
    with torch.autocast('cuda', dtype=torch.float16):
        assert ops.sh_encode(ask(dirs.half()), 3).dtype == torch.float32 and _native(ops.sh_encode(ask(dirs), 3))
    # refused as before
    for bad in (lambda: ops.SH_to_RGB(sh, pos, cam, 4), lambda: ops.SH_to_RGB(sh[:, :64].repeat(1, 4, 1), pos, cam, 7), lambda: ops.SH_to_RGB(sh, pos[:9], cam, 3),
                lambda: ops.SH_to_RGB(sh, pos, cam[:2], 3), lambda: ops.SH_to_RGB(sh.double(), pos, cam, 3),
                lambda: ops.SH_to_RGB(sh.cpu(), pos, cam, 3), lambda: ops.sh_encode(dirs, 8), lambda: ops.sh_encode(dirs[:0], 3)):
        with pytest.raises(RuntimeError):
            bad()
    for f, x in ((lambda x: ops.sh_encode(x, 3), dirs), (lambda x: ops.SH_to_RGB(sh, x, cam, 3), pos)):
        with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):
            f(torch.autograd.forward_ad.make_dual(ask(x), torch.ones_like(x)))
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda x: f(x).sum())(x)
        x = ask(x)
        first, = torch.autograd.grad((f(x) ** 2).sum(), x, create_graph=True)
        with pytest.raises(RuntimeError, match='differentiate twice'):
            torch.autograd.grad((first ** 2).sum(), x)
        x = ask(x)
        out = f(x)
        with torch.no_grad():
            x.mul_(2.0)  # what the backward reads has been edited
        with pytest.raises(RuntimeError, match='modified by an inplace operation'):
            out.sum().backward()


@pytest.mark.parametrize('strided', [0, 1])
@pytest.mark.parametrize('wanted', [0, 1])
@pytest.mark.parametrize('camera', [False, True])
def test_saved_inputs_handed_back_strided(camera, wanted, strided, device):
    """A hook may hand the saved coefficients or positions back in another layout (kept by columns, say): the pair takes them so where
    their own gradient is not asked for, and the node does what the pair does."""
    from fast_sp_gs_amd import ops
    sh, pos, cam, _, up = _inputs(300, 16, device, camera)
    def run(f):
        inputs = [sh.clone(), pos.clone()]
        inputs[wanted].requires_grad_(True)
        at = inputs[strided].data_ptr()
        back = lambda s: s[0].transpose(0, 1).contiguous().transpose(0, 1) if s[1] else s[0]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (t, t.data_ptr() == at), back):
            out = f(*inputs, cam, 3, True)
        return [out, torch.autograd.grad(out, inputs[wanted], up)[0]]
    if wanted == strided:
        for f in (ops.SH_to_RGB, ops._rgb_pair):
            with pytest.raises(RuntimeError, match='must be contiguous'):
                run(f)
    else:
        for x, y in zip(run(ops.SH_to_RGB), run(ops._rgb_pair)):
            assert torch.equal(x, y)
