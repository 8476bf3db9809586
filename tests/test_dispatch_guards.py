"""Where a kernel stands for a module's call, it must not when something has to see
the call itself: hooks, subclasses, biases, adapters, parametrisations.  On the CPU:
the guards' decisions.
"""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from vagus_amd import ops
from vagus_amd.layer import GatedDeltaNet, ShortConv


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
