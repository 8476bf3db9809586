"""The layer's autograd functions under create_graph when one tensor is used
more than once (a layer applied twice, tied weights): first and second
derivatives against the plain torch expressions, in fp64 on the CPU (the
kernels of the forwards replaced by their expressions; a differentiable backward is
torch throughout) and on the GPU with the kernels.

Bars: 1e-12 in fp64; on the GPU the repository's bars, 1e-5 in fp32 and 2e-2 in bf16.
"""
import pytest
import torch
import torch.nn.functional as F

from vagus_amd import ops


def _rel(x, ref):
    x, ref = x.double().cpu(), ref.double().cpu()
    return ((x - ref).norm() / ref.norm().clamp_min(1e-30)).item()


def _linear(apply):
    """x -> W2 (SiLU(W2 SiLU(W1 x) + W1 x)), W1 and W2 each used twice, once together."""
    def fn(x, w1, w2):
        a, b = apply(x, w1, w2)
        c, d = apply(F.silu(a) + b, w1, w2)
        return c * d
    return fn


def _conv(apply):
    return lambda x, w: apply(apply(x, w) + x, w)


def _norm(apply):
    return lambda o, gate, gamma: apply(apply(o, gate, gamma), gate + o, gamma)


def _l2(apply):
    return lambda x: apply(apply(x) * x + x)


def _inputs(kind, dtype, device):
    g = torch.Generator().manual_seed(0)
    shapes = {'linear': [(2, 9, 16), (16, 16), (16, 16)], 'conv': [(2, 9, 8), (8, 1, 4)],
              'norm': [(3, 5, 16), (3, 5, 16), (16,)], 'l2': [(3, 5, 16)]}[kind]
    return [torch.randn(*s, generator=g).to(device, dtype).requires_grad_() for s in shapes]


def _derivatives(fn, xs):
    """The output, the gradients taken with create_graph, and the gradients of their squares' sum."""
    y = fn(*xs)
    dy = torch.linspace(-1, 1, y.numel(), dtype=torch.float64).reshape(y.shape).to(y)
    first = torch.autograd.grad(y, xs, dy, create_graph=True)
    # (create_graph: the forwards' own nodes are part of this pass, and on the CPU theirs have no kernels)
    second = torch.autograd.grad(sum(d.square().sum() for d in first), xs, create_graph=not y.is_cuda)
    return [t.detach() for t in (y, *first, *second)]


KINDS = {
    'linear': (_linear, lambda x, *ws: ops._Projections.apply(x, *ws), lambda x, *ws: [F.linear(x, w) for w in ws]),
    'conv': (_conv, lambda x, w: ops._ShortConvRule.apply(x, w, 'silu'),
             lambda x, w: ops.short_conv_expression(x, w, 'silu')),
    'norm': (_norm, lambda o, gate, gamma: ops._NormGateRule.apply(o, gate, gamma, 1e-6),
             lambda o, gate, gamma: ops.norm_gate_expression(o, gate, gamma, 1e-6)),
    'l2': (_l2, lambda x: ops._L2NormRows.apply(x, 1e-6), lambda x: ops.l2norm_expression(x, 1e-6)),
}


@pytest.mark.parametrize('kind', list(KINDS))
def test_repeated_use(kind, monkeypatch):
    monkeypatch.setattr(ops, 'causal_conv1d', lambda x, w, activation: (ops.short_conv_expression(x, w, activation), None))
    monkeypatch.setattr(ops, '_norm_gate', lambda o, ep: ops.norm_gate_expression(o, ep.gate, ep.gamma, ep.eps))
    monkeypatch.setattr(ops, '_check_device', lambda *ts: None)
    net, rule, expression = KINDS[kind]
    xs = _inputs(kind, torch.float64, 'cpu')
    for a, b in zip(_derivatives(net(rule), xs), _derivatives(net(expression), xs)):
        assert _rel(a, b) < 1e-12


@pytest.mark.parametrize('kind', ['linear', 'conv', 'norm'])
def test_gradient_of_one_input_links_to_the_others(kind, monkeypatch):
    """The gradient with respect to the first input alone, differentiated with respect to all."""
    monkeypatch.setattr(ops, 'causal_conv1d', lambda x, w, activation: (ops.short_conv_expression(x, w, activation), None))
    monkeypatch.setattr(ops, '_norm_gate', lambda o, ep: ops.norm_gate_expression(o, ep.gate, ep.gamma, ep.eps))
    monkeypatch.setattr(ops, '_check_device', lambda *ts: None)
    net, rule, expression = KINDS[kind]
    xs = _inputs(kind, torch.float64, 'cpu')

    def second(fn):
        dx, = torch.autograd.grad(net(fn)(*xs).square().sum(), xs[:1], create_graph=True)
        return [d.detach() for d in torch.autograd.grad(dx.square().sum(), xs, create_graph=True)]

    for a, b in zip(second(rule), second(expression)):
        assert _rel(a, b) < 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize('kind,dtype', [('linear', torch.bfloat16), ('conv', torch.float32), ('norm', torch.float32),
                                        ('l2', torch.float32)])
def test_repeated_use_on_the_gpu(kind, dtype):
    net, rule, expression = KINDS[kind]
    xs = _inputs(kind, dtype, 'cuda')
    if kind == 'linear':
        assert type(ops.projections(*xs)[0].grad_fn).__name__.startswith('_Projections')
    ref = [t.detach().cpu().double().requires_grad_() for t in xs]
    first = _derivatives(net(rule), xs)
    for a, b in zip(first, _derivatives(net(expression), ref)):
        e = _rel(a, b)
        print(f'[parity] {kind} {dtype} rel_l2={e:.3e}', flush=True)
        assert e < (1e-5 if dtype == torch.float32 else 2e-2)
