"""The deformation branch through the native host layer against the operators and torch: the network with its encoding
formed in the kernel (rows around a block of 32, one head missing its gradient), the K-NN + warp node with a slice of a wider scaling head, the dense Adam."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B', [1, 31, 32, 33, 300])
@pytest.mark.parametrize('local_frame', [False, True])
def test_network_equals_encoded_rows(B, local_frame, device):
    from fast_sp_gs_amd._C import get_C_function
    from fast_sp_gs_amd.deform import DeformNetwork, _DeformMlp
    torch.manual_seed(B)
    net = DeformNetwork(local_frame=local_frame).to(device)
    g = torch.Generator().manual_seed(B)
    x, t = (torch.rand(B, 3, generator=g) * 2 - 1).to(device), torch.rand(1, generator=g).to(device)
    out = [o for o in net(x, t) if o is not None]
    params = net._mlp_parameters()
    rows = sum(h.out_features for h in net._heads())
    ref = _DeformMlp.apply(net.encode(x, t), *net._packed, net._packed_t, net._heads_w, net.D, net.skip, rows, *params)
    assert torch.equal(torch.cat(out, 1), ref)
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(net(x, t), out))
    up = torch.randn(B, rows, generator=g).to(device)
    up[:, 3:7] = 0  # the rotation head gets no gradient below
    parts = [p for p in up.split([h.out_features for h in net._heads()], dim=1)]
    keep = [k for k in range(len(out)) if k != 1]
    got = torch.autograd.grad([out[k] for k in keep], params, [parts[k].contiguous() for k in keep], allow_unused=True)
    want = torch.autograd.grad(ref, params, up)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    hidden = get_C_function('mlp_forward')(net.encode(x, t), *net._packed, net.D, net.skip, rows, True)[1]
    assert hidden.shape == (net.D, B, 256) and bool((hidden.view(torch.bfloat16) >= 0).all())


@pytest.mark.parametrize('N,M,K,warp,columns', [(1, 1, 1, 'LBS', 3), (1000, 40, 3, 'LBS', 2), (1025, 300, 4, 'LBS_c', 2),
                                                (777, 65, 5, None, 1)])
def test_warp_node_equals_operators(N, M, K, warp, columns, device):
    from fast_sp_gs_amd.deform import _fused_deform, _LbsBlend, knn_points
    g = torch.Generator().manual_seed(N)
    mk = lambda *s: torch.randn(*s, generator=g).to(device).requires_grad_(True)
    points, ctrl, sp_t, sp_r, sp_s = mk(N, 3).detach(), mk(M, 3), mk(M, 3), mk(M, 4), mk(M, 3)
    sp_rot = mk(M, 4) if warp else None
    out = _fused_deform(points, ctrl, sp_t, sp_r, sp_s, sp_rot, K, 0.5, warp or 'LBS', 'dist', None, None, columns)
    d2, idx = knn_points(points, ctrl, K)
    ref = _LbsBlend.apply(points, ctrl, sp_t, sp_r, sp_s[:, :columns], sp_rot, d2, idx, None, None, 0.5, warp, 'dist')
    for a, b in zip(out[:4], ref):
        assert torch.equal(a, b)
    assert torch.equal(out[4], idx)
    up = [torch.randn(o.shape, generator=g).to(device) for o in ref[:3]]
    wanted = [ctrl, sp_t, sp_r, sp_s] + ([sp_rot] if warp else [])
    for a, b in zip(torch.autograd.grad(out[:3], wanted, up), torch.autograd.grad(ref[:3], wanted, up)):
        assert (a - b).norm() <= 1e-5 * b.norm() + 1e-7


def test_dense_adam_follows_torch(device):
    from fast_sp_gs_amd.deform import DeformNetwork
    from fast_sp_gs_amd.sparse_gaussian_adam import DenseAdam
    g = torch.Generator().manual_seed(3)
    shapes = [(1,), (1023,), (1024,), (1025,), (256, 340)] * 7  # more tensors than one launch takes
    values = [torch.randn(s, generator=g) for s in shapes]
    mine, theirs = ([v.clone().to(device).requires_grad_(True) for v in values] for _ in range(2))
    a, b = DenseAdam(mine, lr=1e-2), torch.optim.Adam(theirs, lr=1e-2)
    for _ in range(3):
        for p, q in zip(mine, theirs):
            p.grad = torch.randn(p.shape, generator=g).to(device)
            q.grad = p.grad.clone()
        a.step(), b.step()
    for p, q in zip(mine, theirs):
        assert torch.allclose(p, q, rtol=0, atol=1e-6) and float(a.state[p]['step']) == 3
        assert torch.allclose(a.state[p]['exp_avg_sq'], b.state[q]['exp_avg_sq'], rtol=1e-5, atol=1e-9)
    b.load_state_dict(a.state_dict())
    net = DeformNetwork().to(device)
    opt = DenseAdam(net.parameters(), lr=1e-2)
    x, t = torch.rand(64, 3, generator=g).to(device), torch.rand(1, generator=g).to(device)
    first = net(x, t)[0]
    first.sum().backward()
    opt.step()
    net.pack()
    second = net(x, t)[0]
    assert not torch.equal(first, second)  # the step's weights are in use
    assert (second - net.forward_fp32(x, t)[0]).norm() <= 2e-2 * second.norm() + 1e-5


@pytest.mark.parametrize('change', ['torch', 'dense', 'weight_decay'])
def test_dense_adam_state_goes_on_in_torch(change, device):
    """Three plain steps, then two more: in torch's Adam or a new DenseAdam with the saved state, or in the same optimiser
    with a setting that takes torch's step. Step counts and parameters as torch's throughout."""
    import io

    from fast_sp_gs_amd.sparse_gaussian_adam import DenseAdam
    g = torch.Generator().manual_seed(4)
    values = [torch.randn(n, generator=g) for n in (1, 3, 64, 1025)]
    mine, theirs = ([v.clone().to(device).requires_grad_(True) for v in values] for _ in range(2))
    a, b = DenseAdam(mine, lr=1e-2), torch.optim.Adam(theirs, lr=1e-2)

    def step(first, second):
        for p, q in zip(mine, theirs):
            p.grad = torch.randn(p.shape, generator=g).to(device)
            q.grad = p.grad.clone()
        first.step(), second.step()

    for _ in range(3):
        step(a, b)
    if change == 'weight_decay':
        for opt in (a, b):
            opt.param_groups[0]['weight_decay'] = 1e-2
    else:
        file = io.BytesIO()
        torch.save(a.state_dict(), file)
        file.seek(0)
        a = (torch.optim.Adam if change == 'torch' else DenseAdam)(mine, lr=1e-2)
        a.load_state_dict(torch.load(file, weights_only=True))
    for _ in range(2):
        step(a, b)
    for p, q in zip(mine, theirs):
        assert float(a.state[p]['step']) == 5 and torch.allclose(p, q, rtol=0, atol=1e-6)


@pytest.mark.parametrize('M', [1, 40])
@pytest.mark.parametrize('layout', ['broadcast', 'transposed', 'column', 'one_column', 'overlapping', 'slice'])
def test_scale_table_of_any_layout(layout, M, device):
    from fast_sp_gs_amd.deform import superpoint_deform
    g = torch.Generator().manual_seed(M)
    r = lambda *shape: torch.randn(*shape, generator=g).to(device)
    points, controls, sp_t, sp_r, up = r(100, 3), r(M, 3), r(M, 3), r(M, 4), r(100, 2)
    base, view = {'broadcast': (r(1, 2), lambda t: t.expand(M, 2)), 'transposed': (r(2, M), lambda t: t.t()),
                  'column': (r(3, M), lambda t: t.t()[:, :1]), 'one_column': (r(M, 3), lambda t: t[:, 1:2]),
                  'overlapping': (r(M + 1), lambda t: t.as_strided((M, 2), (1, 1))),
                  'slice': (r(M, 5), lambda t: t[:, 2:4])}[layout]
    results = []
    for table in (view, lambda t: view(t).clone(memory_format=torch.contiguous_format)):
        leaf = base.clone().requires_grad_(True)
        out = superpoint_deform(points, controls, sp_t, sp_r, table(leaf), K=min(3, M))[2]
        results.append((out, *torch.autograd.grad((out * up[:, :out.shape[1]]).sum(), [leaf])))
    assert torch.equal(results[0][0], results[1][0])
    assert torch.allclose(results[0][1], results[1][1], rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize('B', [1, 31, 32, 33, 300])
def test_network_entry_points_with_states_as_rows(B, device):
    """fsgs_mlp_forward / _backward, whose callers keep [layer][B][256] states and read dZ in that form, against the
    operators, which keep the batch innermost: the same numbers."""
    from fast_sp_gs_amd import lib as L
    from fast_sp_gs_amd._C import get_C_function
    from fast_sp_gs_amd.deform import DeformNetwork
    torch.manual_seed(B)
    net, lib = DeformNetwork().to(device), L.load()
    net.pack()
    x = net.encode(torch.rand(B, 3, device=device) * 2 - 1, torch.rand(1, device=device)).detach()
    rows, Din = 10, x.shape[1]
    want, states = get_C_function('mlp_forward')(x, *net._packed, net.D, net.skip, rows, True)
    up = torch.randn(B, rows, device=device)
    w_want, b_want, dz_want = get_C_function('mlp_backward')(x, net._packed_t, net._heads_w, states, up, net.D, net.skip, True)
    out = torch.full((B, rows), float('nan'), device=device)
    saved = torch.zeros(net.D, B, 256, dtype=torch.int16, device=device)
    stream = L.current_stream()
    rc = lib.fsgs_mlp_forward(B, Din, 256, net.D, net.skip, rows, L.ptr(x), *map(L.ptr, net._packed), L.ptr(out), L.ptr(saved),
                              stream)
    L.check(rc, 'fsgs_mlp_forward')
    assert torch.equal(out, want) and torch.equal(saved, states)
    g_w, g_b = (torch.full_like(t, float('nan')) for t in (w_want, b_want))
    ws = torch.empty(lib.fsgs_mlp_backward_workspace_bytes(B, net.D), dtype=torch.uint8, device=device)
    args = (B, Din, 256, net.D, net.skip, rows, L.ptr(x), L.ptr(net._packed_t), L.ptr(net._heads_w), L.ptr(saved), L.ptr(up),
            L.ptr(g_w), L.ptr(g_b), L.ptr(ws))
    L.check(lib.fsgs_mlp_backward(*args, ws.numel(), stream), 'fsgs_mlp_backward')
    dz = ws[:net.D * B * 512].view(torch.bfloat16).view(net.D, B, 256)
    assert torch.equal(g_w, w_want) and torch.equal(g_b, b_want) and torch.equal(dz, dz_want)
    assert lib.fsgs_mlp_backward(*args, ws.numel() - 1, stream) != 0


def test_short_control_tables_are_refused(device):
    """On the host: fewer radii or weights than control points, positions with fewer than three coordinates."""
    from fast_sp_gs_amd.deform import superpoint_deform
    g = torch.Generator().manual_seed(5)
    r = lambda *shape: torch.randn(*shape, generator=g).to(device)
    M, points, moves = 40, r(100, 3), (r(40, 3), r(40, 4), r(40, 2))
    kernel = lambda radius, weight: superpoint_deform(points, r(M, 3), *moves, LBS_method='weighted_kernel', sp_radius=radius,
                                                      sp_weight=weight)[0]
    assert torch.isfinite(kernel(r(M), r(M, 1))).all()
    for radius, weight in ((r(M - 1), r(M)), (r(M), r(M - 1))):
        with pytest.raises(RuntimeError, match='a value per control point'):
            kernel(radius, weight)
    with pytest.raises(RuntimeError, match='positions'):
        superpoint_deform(points[:, :2], r(M, 2), *moves)
