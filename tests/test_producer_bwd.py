"""The layer's producers and epilogue under autograd on the GPU: the kernels'
gradients against torch's own autograd of the module's expressions in fp64.

The bars are the repository's parity bars: rel_l2 <= 2e-2 for 16-bit inputs,
1e-5 for fp32.
"""
import pytest
import torch
import torch.nn.functional as F

BARS = {torch.float32: 1e-5, torch.bfloat16: 2e-2, torch.float16: 2e-2}


def _rel(x, ref):
    x, ref = x.double().cpu(), ref.double().cpu()
    return ((x - ref).norm() / ref.norm().clamp_min(1e-30)).item()


def _check(label, got, want, dtype):
    for name, x, ref in zip(label, got, want):
        err = _rel(x, ref)
        print(f'[parity] {name} rel_l2={err:.3e}', flush=True)
        assert err <= BARS[dtype]


def _grads(fn, inputs, cotangent):
    xs = [t.detach().requires_grad_() for t in inputs]
    y = fn(*xs)
    return [y.detach()] + list(torch.autograd.grad(y, xs, cotangent.to(y.dtype)))


# 16 x 8 token runs in one workgroup's rows, channel groups of 32 x 4 (the last one
# partly filled), runs of 8, 16 and 32 tokens with remainders, sequences shorter than
# the window, and the longest kernel (whose window is wider than the tokens of a step)
@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('B,T,D,K,act', [(1, 1, 8, 4, 'silu'), (3, 2, 40, 4, 'silu'), (2, 70, 192, 1, None),
                                         (2, 129, 136, 3, 'silu'), (3, 1001, 512, 4, 'silu'), (1, 300, 64, 8, 'silu'),
                                         (16, 1024, 1024, 4, None)])
def test_short_conv_gradients(dtype, B, T, D, K, act):
    from vagus_amd import ops
    print(f'\n[case] short conv bwd {dtype} B={B} T={T} D={D} K={K} {act}', flush=True)
    g = torch.Generator().manual_seed(T + D + K)
    x, w, dy = (torch.randn(*s, generator=g).to(dtype).cuda() for s in ((B, T, D), (D, 1, K), (B, T, D)))
    got = _grads(lambda x, w: ops.short_conv(x, w, act), (x, w), dy)
    assert type(got[0]) is torch.Tensor
    want = _grads(lambda x, w: ops.short_conv_expression(x, w, act), (x.cpu().double(), w.cpu().double()), dy.cpu())
    _check(('y', 'dx', 'dw'), got, want, dtype)


@pytest.mark.gpu
def test_short_conv_second_derivative():
    """create_graph: the kernel's backward differentiated again equals torch's."""
    from vagus_amd import ops
    g = torch.Generator().manual_seed(3)
    x, w, dy = (torch.randn(*s, generator=g).cuda() for s in ((2, 9, 8), (8, 1, 4), (2, 9, 8)))

    def second(fn, x, w, dy):
        x, w = x.requires_grad_(), w.requires_grad_()
        dx, dw = torch.autograd.grad(fn(x, w, 'silu'), (x, w), dy, create_graph=True)
        return torch.autograd.grad(dx.square().sum() + dw.square().sum(), (x, w))

    got = second(ops.short_conv, x.clone(), w.clone(), dy)
    want = second(ops.short_conv_expression, x.cpu().double(), w.cpu().double(), dy.cpu().double())
    _check(('ddx', 'ddw'), got, want, torch.float32)


# one row, rows that leave a workgroup's last pass partly filled, more rows than the grid takes
# in one pass (1024 workgroups x 256 / lanes rows), the shortest and the longest row
@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('rows,dv', [(1, 128), (37, 8), (1001, 256), (20001, 128), (70001, 64), (513, -64)])
def test_norm_gate_gradients(dtype, rows, dv):
    from vagus_amd import ops
    dv = dv if dv > 0 else -dv * (4 if dtype == torch.float32 else 8)       # 64 lanes: the longest
    print(f'\n[case] epilogue bwd {dtype} rows={rows} dv={dv}', flush=True)
    g = torch.Generator().manual_seed(rows + dv)
    o, gate, dy = (torch.randn(rows, dv, generator=g).to(dtype).cuda() for _ in range(3))
    gamma = (torch.rand(dv, generator=g) + 0.5).to(dtype).cuda()
    got = _grads(lambda *a: ops.norm_gate(*a, 1e-6), (o, gate, gamma), dy)
    want = _grads(lambda *a: ops.norm_gate_expression(*a, 1e-6), [t.cpu().double() for t in (o, gate, gamma)], dy.cpu())
    _check(('y', 'do', 'dgate', 'dgamma'), got, want, dtype)


@pytest.mark.gpu
def test_norm_gate_second_derivative():
    from vagus_amd import ops
    g = torch.Generator().manual_seed(4)
    o, gate, dy = (torch.randn(5, 16, generator=g).cuda() for _ in range(3))
    gamma = torch.rand(16, generator=g).cuda() + 0.5

    def second(fn, o, gate, gamma, dy):
        xs = [t.requires_grad_() for t in (o, gate, gamma)]
        d = torch.autograd.grad(fn(*xs, 1e-6), xs, dy, create_graph=True)
        return torch.autograd.grad(sum(x.square().sum() for x in d), xs)

    got = second(ops.norm_gate, o.clone(), gate.clone(), gamma.clone(), dy)
    want = second(ops.norm_gate_expression, *(t.cpu().double() for t in (o, gate, gamma, dy)))
    _check(('ddo', 'ddgate', 'ddgamma'), got, want, torch.float32)


# one row, a partly filled last workgroup, the shortest and the longest row, a row length
# the kernel does not take (torch's own expression), a strided view
@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('rows,d', [(1, 64), (37, 8), (1001, 128), (513, -64), (65, 100)])
@pytest.mark.parametrize('view', [False, True])
def test_l2norm_gradients(dtype, rows, d, view):
    from vagus_amd import ops
    d = d if d > 0 else -d * (4 if dtype == torch.float32 else 8)
    print(f'\n[case] l2norm {dtype} rows={rows} d={d} view={view}', flush=True)
    g = torch.Generator().manual_seed(rows + d)
    x, dy = (torch.randn(rows, 2 * d if view else d, generator=g).to(dtype).cuda()[:, :d] for _ in range(2))
    got = _grads(lambda x: ops.l2norm_rows(x, 1e-6), (x,), dy)
    want = _grads(lambda x: ops.l2norm_expression(x, 1e-6), (x.cpu().double(),), dy.cpu())
    _check(('y', 'dx'), got, want, dtype)
    assert torch.equal(ops.l2norm_rows(x.detach()), got[0])


# tiles of 256 x 128 with rows and columns left over, several matrices of one input (widths that
# are no multiple of 8 or 16 among them), token counts below one step, with a partial last step,
# with one split and with many
@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('T,dim,widths', [(1, 8, [8]), (31, 40, [4, 264]), (127, 136, [256]), (1003, 1024, [512, 64, 3]),
                                          (3003, 64, [512]), (8200, 520, [300, 16, 1032]), (70000, 64, [24])])
@pytest.mark.parametrize('view', [False, True])
def test_linear_weight_gradients(dtype, T, dim, widths, view):
    """The sum's bound: fp32 accumulation, one rounding of the result."""
    from vagus_amd import ops
    print(f'\n[case] wgrad {dtype} T={T} dim={dim} widths={widths} view={view}', flush=True)
    g = torch.Generator('cuda').manual_seed(T + dim)
    # a view: rows of a wider buffer that start on a 16-byte unit
    mats = [torch.randn(T, d + (16 if view else 0), generator=g, device='cuda').to(dtype)[:, 8 if view else 0:][:, :d]
            for d in [dim] + widths]
    got = ops.linear_wgrads(mats[0], mats[1:])
    for dy, dw in zip(mats[1:], got):
        ref = dy.double().T.contiguous() @ mats[0].double()
        err = _rel(dw, ref)
        print(f'[parity] rel_l2={err:.3e}', flush=True)
        assert dw.shape == ref.shape and err <= (4e-3 if dtype == torch.bfloat16 else 5e-4)


@pytest.mark.gpu
@pytest.mark.parametrize('frozen', [(), ('x',), (1,), (0, 2)])
def test_projections_gradients(frozen):
    from vagus_amd import ops
    print(f'\n[case] projections frozen={frozen}', flush=True)
    g = torch.Generator().manual_seed(6)
    x = torch.randn(2, 65, 128, generator=g).bfloat16().cuda().requires_grad_('x' not in frozen)
    ws = [(0.1 * torch.randn(n, 128, generator=g)).bfloat16().cuda().requires_grad_(i not in frozen)
          for i, n in enumerate((256, 64, 4))]
    dys = [torch.randn(2, 65, n, generator=g).bfloat16().cuda() for n in (256, 64, 4)]
    leaves = [t for t in [x] + ws if t.requires_grad]
    got = torch.autograd.grad(ops.projections(x, *ws), leaves, dys)
    x64, w64 = x.detach().cpu().double(), [w.detach().cpu().double() for w in ws]
    for t, s in zip([x64] + w64, [x] + ws):
        t.requires_grad_(s.requires_grad)
    want = torch.autograd.grad([F.linear(x64, w) for w in w64], [t for t in [x64] + w64 if t.requires_grad],
                               [d.cpu().double() for d in dys])
    _check([f'd{i}' for i in range(len(got))], got, want, torch.bfloat16)
