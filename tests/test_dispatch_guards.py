"""Where a kernel stands for a module's call, it must not when something has to see
the call itself: hooks, subclasses, biases, adapters, parametrisations.  On the CPU:
the guards' decisions.
"""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from vagus_amd import ops
from vagus_amd.layer import GatedDeltaNet, RMSNorm, ShortConv


def _layer(gate='scalar', dtype=torch.float32, device='cpu', **kw):
    torch.manual_seed(0)
    kw = {'dim': 64, 'head_count': 2, 'key_head_dim': 64, 'value_head_dim': 64, 'gate_rank': 16, **kw}
    return GatedDeltaNet(gate=gate, **kw).to(device, dtype)


class Adapter(nn.Module):
    """A low-rank adapter's shape: a module around the projection."""

    def __init__(self, base):
        super().__init__()
        self.base = base
        self.scale = 1.5

    def forward(self, x):
        return self.scale * self.base(x)


class OwnLinear(nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


def _hook(m, name):
    getattr(m, name).register_forward_hook(lambda mod, args, out: out + 3)


def _pre_hook(m, name):
    getattr(m, name).register_forward_pre_hook(lambda mod, args: (2 * args[0],))


def _adapt(m, name):
    setattr(m, name, Adapter(getattr(m, name)))


def _bias(m, name):
    getattr(m, name).bias = nn.Parameter(torch.ones_like(getattr(m, name).weight[:, 0]))


def _subclass(m, name):
    lin = getattr(m, name)
    own = OwnLinear(lin.in_features, lin.out_features, bias=False).to(lin.weight)
    own.weight = lin.weight
    setattr(m, name, own)


def _own_forward(m, name):
    lin = getattr(m, name)
    lin.forward = lambda x: F.linear(x, lin.weight) - 1


def _parametrize(m, name):
    class Half(nn.Module):
        def forward(self, w):
            return 0.5 * w
    nn.utils.parametrize.register_parametrization(getattr(m, name), 'weight', Half())


CHANGES = [_hook, _pre_hook, _adapt, _bias, _subclass, _own_forward, _parametrize]


@pytest.mark.parametrize('change', CHANGES, ids=lambda f: f.__name__)
@pytest.mark.parametrize('gate,name', [('scalar', n) for n in ('wq', 'wk', 'wv', 'wg', 'wa', 'wb')]
                         + [('vector', 'wa1'), ('vector', 'wb'), ('none', 'wb')])
def test_decode_inputs_call_a_module_that_is_not_plain(change, gate, name, monkeypatch):
    """The one-token step's inputs, with the kernel ready to take them: a plain layer takes it, a
    changed one calls its modules."""
    m = _layer(gate)
    x = torch.randn(3, 1, 64, generator=torch.Generator().manual_seed(1))
    took = []
    monkeypatch.setattr(ops, 'project_rows_fits', lambda x, ws: True)

    def project_rows(x, ws, w_b=None):
        took.append(1)
        raise KeyError('the kernel')

    monkeypatch.setattr(ops, 'project_rows', project_rows)
    with pytest.raises(KeyError):
        m._decode_inputs(x)
    assert took
    change(m, name)
    with torch.no_grad():
        qp, kp, vp, og, g, beta, gate_proj = m._decode_inputs(x)
        want_g, want_beta = m._gates(x, raw_gate=gate == 'vector', raw_beta=True)
        assert len(took) == 1 and gate_proj is None
        for y, w in zip((qp, kp, vp, og, beta), (m.wq, m.wk, m.wv, m.wg, m.wb)):
            assert torch.equal(y, w(x))
        assert (g is None) if gate == 'none' else torch.equal(g, want_g)
        assert torch.equal(beta, want_beta)


def _conv_bias(conv):
    conv.bias = nn.Parameter(torch.full((conv.weight.shape[0],), 0.5))


def _conv_padding(conv):
    """A module that pads by itself."""
    conv.padding = (2,)


def _conv_dilation(conv):
    conv.dilation = (2,)


def _conv_stride(conv):
    conv.stride = (2,)


@pytest.mark.parametrize('change', [_conv_bias, _conv_padding, _conv_dilation, _conv_stride], ids=lambda f: f.__name__)
def test_short_conv_calls_a_conv_of_other_settings(change):
    """Under autograd the short conv is the module's own call (opt.py:78-80) unless that is
    the plain causal conv of its weight."""
    conv = ShortConv(8, 4)
    x = torch.randn(2, 9, 8, generator=torch.Generator().manual_seed(1))
    change(conv.conv)
    want = F.silu(conv.conv(F.pad(x.transpose(1, 2), (3, 0))).transpose(1, 2))
    got = conv(x, 'silu')
    assert got.shape == want.shape and torch.equal(got, want)


def test_training_pass_of_a_layer_without_write_strengths(monkeypatch):
    """A subclass that writes by itself and has no W_b: the training pass groups the projections
    that are there."""
    class OwnWrite(GatedDeltaNet):
        def __init__(self, *args, **kw):
            super().__init__(*args, **kw)
            del self.wb

        def _write(self, x, k, g, beta):
            assert beta is None
            return None, 0.5 * k

    torch.manual_seed(0)
    m = OwnWrite(64, 2, 64, 64)
    monkeypatch.setattr(OwnWrite, '_pick_impl', lambda self, q: 'hip')
    scans = []

    def scan(q, k, v, g, beta, S0, *, w, **kw):
        scans.append(w)
        return v + w.sum(-1, keepdim=True) + g.sum(-1, keepdim=True), S0

    monkeypatch.setattr(ops, 'chunk_scan_vec', scan)
    m(torch.randn(2, 5, 64)).sum().backward()
    # the scan in the kernels' place reads no q
    assert len(scans) == 1 and all(p.grad is not None for n, p in m.named_parameters()
                                   if not n.startswith(('wq', 'conv_q')))


# --------------------------------------------------------------------------
# the training pass
# --------------------------------------------------------------------------

def _chained(m, x):
    """The layer's training pass up to the scan, by its pieces, as one scalar."""
    names = m._input_projections()
    if m._plain_projections():
        y = dict(zip(names, ops.projections(x, *(getattr(m, n).weight for n in names))))
        qp, kp, vp, kw = y['wq'], y['wk'], y['wv'], dict(proj=y)
    else:
        qp, kp, vp, kw = m.wq(x), m.wk(x), m.wv(x), {}
    q, k, v = m._heads(qp, kp, vp)
    g, beta = m._gates(x, **kw)
    return m._output(q * k + v * beta[..., None] + g.reshape(*g.shape[:2], m.head_count, -1)[..., :1], x, **kw)


class OwnNorm(RMSNorm):
    def forward(self, x):
        return 2 * super().forward(x)


def _own_norm(m, name):
    own = OwnNorm(m.o_norm.dim).to(m.o_norm.gamma)
    own.gamma = m.o_norm.gamma
    m.o_norm = own


TRAINED = [(change, name) for change in CHANGES for name in ('wq', 'wk', 'wv', 'wg', 'wa', 'wb', 'wo')] + [
    (_hook, 'o_norm'), (_pre_hook, 'o_norm'), (_own_norm, 'o_norm'), (_own_forward, 'wo'),
    (lambda m, name: _hook(m.conv_q, 'conv'), 'conv_q'), (lambda m, name: _hook(m, 'conv_k'), 'conv_k'),
    (lambda m, name: _pre_hook(m.conv_v, 'conv'), 'conv_v')]


@pytest.mark.parametrize('change,name', TRAINED, ids=[f'{getattr(c, "__name__", "hook")}-{n}' for c, n in TRAINED])
def test_training_pass_calls_a_module_that_is_not_plain(change, name):
    """On the CPU: what the changed layer gives, and its gradients, against the modules called one by one."""
    m = _layer('scalar')
    x = torch.randn(2, 7, 64, generator=torch.Generator().manual_seed(1), requires_grad=True)
    change(m, name)
    y = _chained(m, x)
    H, d = 2, 64
    conv = lambda c, t: c(t, 'silu').view(2, 7, H, d)  # noqa: E731
    q, k, v = (conv(c, w(x)) for c, w in ((m.conv_q, m.wq), (m.conv_k, m.wk), (m.conv_v, m.wv)))
    q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    g = -m.A_log.exp() * F.softplus(m.wa(x) + m.dt_bias)
    o = q * k + v * torch.sigmoid(m.wb(x))[..., None] + g[..., None]
    want = m.wo((m.o_norm(o) * F.silu(m.wg(x).view(2, 7, H, d))).reshape(2, 7, -1))
    assert torch.allclose(y, want, atol=1e-5, rtol=1e-5)
    params = [x, *m.parameters()]
    for a, b in zip(torch.autograd.grad(y.square().sum(), params), torch.autograd.grad(want.square().sum(), params)):
        assert torch.allclose(a, b, atol=1e-3 * b.abs().max().item(), rtol=1e-4)


@pytest.mark.gpu
def test_kernel_autograd_steps_aside():
    """_kernel_autograd takes plain GPU tensors of one type, and nothing where the expression has to be seen."""
    decide = ops._kernel_autograd
    x = torch.randn(3, 8, device='cuda')
    assert decide(x) and decide(x, nn.Parameter(x.clone()))
    assert not decide(x.cpu()) and not decide(x[:0]) and not decide(x.double()) and not decide(x, x.half())
    assert not decide(x, x.cpu())

    class Sub(torch.Tensor):
        pass

    assert not decide(x.as_subclass(Sub)) and not decide(x, x.as_subclass(Sub))
    with torch.autocast('cuda', torch.bfloat16):
        assert not decide(x)
    seen = []
    torch.func.vmap(lambda t: seen.append(decide(x)) or t)(x)
    torch.func.jvp(lambda t: seen.append(decide(x)) or t, (x,), (x,))
    torch.func.grad(lambda t: seen.append(decide(x)) or t.sum())(x)
    with torch.autograd.forward_ad.dual_level():
        seen.append(decide(x))
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        seen.append(decide(x))
    torch.jit.trace(lambda t: seen.append(decide(x)) or t + 1, (x,), check_trace=False)
    assert seen and not any(seen)
    assert decide(x)                                           # and back


@pytest.mark.gpu
@pytest.mark.parametrize('gate', ['scalar', 'vector'])
@pytest.mark.parametrize('aside', ['autocast', 'hooks', 'nothing'])
def test_training_pass_of_a_layer(gate, aside, monkeypatch):
    """A layer's training pass under autocast and with hooks on every module is its modules' own calls (the same
    pass with the kernels' rules ruled out, to within what repeating torch's conv gradients gives); otherwise it takes
    the rules."""
    torch.manual_seed(0)
    dtype = torch.float32 if aside == 'autocast' else torch.bfloat16
    m = _layer(gate, dtype, 'cuda', fused='scan')
    x = torch.randn(2, 70, 64, device='cuda').to(dtype).requires_grad_()
    fired = []
    if aside == 'hooks':
        for n in (*m._input_projections(), 'wo', 'o_norm'):
            getattr(m, n).register_forward_hook(lambda mod, args, out: fired.append(mod) or 1.01 * out)
        for c in (m.conv_q, m.conv_k, m.conv_v):
            c.conv.register_forward_hook(lambda mod, args, out: fired.append(mod) or 1.01 * out)
    rules = []
    for cls in (ops._Projections, ops._ShortConvRule, ops._NormGateRule):
        forward = cls.forward
        monkeypatch.setattr(cls, 'forward', staticmethod(lambda ctx, *a, f=forward, c=cls: rules.append(c) or f(ctx, *a)))

    def run():
        with torch.autocast('cuda', torch.bfloat16, enabled=aside == 'autocast'):
            y = m(x)
        return [y, *torch.autograd.grad(y.float().square().sum(), [x, *m.parameters()])]

    got, n = run(), len(fired)
    if aside == 'nothing':
        assert set(rules) == {ops._Projections, ops._ShortConvRule, ops._NormGateRule}
        return
    assert not rules and n == (len(m._input_projections()) + 5 if aside == 'hooks' else 0)
    monkeypatch.setattr(ops, '_kernel_autograd', lambda *ts: False)
    for a, b in zip(got, run()):
        assert a.dtype == b.dtype and ((a.double() - b.double()).norm() / b.double().norm()).item() < 2 ** -8
