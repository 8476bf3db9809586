"""Which calls give a sequence the same bits alone, in a dense batch and in a packed
batch: every call of up to 8,192 tokens a sequence, either gate, and above that every call with
whole_sequences=True, forward and backward; without it a longer call may be
walked in segments and agrees to rounding (2.5 roundings of the element type between
two runs that are each about one from exact).
"""
import pytest
import torch

from vagus_amd import _lib, ops, workloads
from vagus_amd.layer import GatedDeltaNet

LONGEST = 8192                  # that stays whole by default


def _scan(x, rows=slice(None), packed=False, grads=None, w=None, **kw):
    """(o, S) of the chosen sequences, with grads (do, dS) also the gradients."""
    t = [None if a is None else a[rows].cuda().requires_grad_(grads is not None)
         for a in (x.q, x.k, x.v, x.g, x.beta, x.initial_state, w)]
    B, T = t[0].shape[:2]
    q, k, v, g, beta, S0, w = (a.reshape(1, B * T, *a.shape[2:]) if packed and a is not None and i != 5 else a
                               for i, a in enumerate(t))
    cu = torch.arange(0, B * T + 1, T, dtype=torch.int32, device='cuda') if packed else None
    if w is not None:
        o, S = ops.chunk_scan_vec(q, k, v, g, None, S0, scale=0.1, delta=True, w=w, cu_seqlens=cu, **kw)
    else:
        fn = ops.chunk_kda if g.dim() == 4 else ops.chunk_gated_delta_rule
        o, S = fn(q, k, v, g, beta, scale=0.1, initial_state=S0, output_final_state=True, cu_seqlens=cu, **kw)
    out = [o.reshape(B, T, *o.shape[2:]), S]
    if grads is not None:
        wrt = [a for i, a in enumerate(t) if a is not None and not (i == 4 and w is not None)]
        out += torch.autograd.grad(out, wrt, [d[rows].cuda() for d in grads])
    return [a.detach() for a in out]


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize('gate', ['scalar', 'vector'])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('T,kw', [(4033, {}), (4100, {}), (LONGEST, {}), (LONGEST + 1, dict(whole_sequences=True)),
                                  (9000, dict(whole_sequences=True))])
def test_same_bits_alone_in_a_batch_and_packed(gate, dtype, T, kw):
    x = workloads.make_inputs(2, T, 2, 128, 64, gate=gate, dtype=dtype, s0_scale=1.0, seed=T)
    both, packed = _scan(x, **kw), _scan(x, packed=True, **kw)
    for i in range(2):
        alone = _scan(x, slice(i, i + 1), **kw)
        for a, b, c in zip(alone, both, packed):
            assert torch.equal(a[0], b[i]) and torch.equal(a[0], c[i])


@pytest.mark.gpu
@pytest.mark.parametrize('gate,write', [('scalar', False), ('vector', False), ('vector', True)])
@pytest.mark.parametrize('T,kw', [(4100, {}), (8300, dict(whole_sequences=True))])
def test_training_pass_alone_and_in_a_batch(gate, write, T, kw):
    """The training forward's bits; its gradients to rounding (their sums over a tile's columns depend on
    the tile, and that on the batch)."""
    x = workloads.make_inputs(2, T, 2, 128, 64, gate=gate, dtype=torch.bfloat16, s0_scale=1.0, seed=1)
    g = torch.Generator().manual_seed(2)
    grads = torch.randn(x.v.shape, generator=g).bfloat16(), torch.randn(x.initial_state.shape, generator=g)
    w = (x.beta[..., None] * x.k.float()).bfloat16() if write else None
    kw = dict(grads=grads, w=w, **kw)
    both = _scan(x, **kw)
    for i in range(2):
        alone = _scan(x, slice(i, i + 1), **kw)
        assert torch.equal(alone[0][0], both[0][i]) and torch.equal(alone[1][0], both[1][i])
        assert all(_rel(a[0], b[i]) < 2.5 * 2 ** -8 for a, b in zip(alone, both))


@pytest.mark.gpu
@pytest.mark.parametrize('gate', ['scalar', 'vector'])
@pytest.mark.parametrize('dtype,step', [(torch.bfloat16, 2 ** -8), (torch.float16, 2 ** -11)])
def test_longer_calls_agree_to_rounding(gate, dtype, step):
    x = workloads.make_inputs(1, LONGEST + 1, 2, 128, 64, gate=gate, dtype=dtype, s0_scale=1.0, seed=3)
    for a, b in zip(_scan(x), _scan(x, whole_sequences=True)):
        assert not torch.equal(a, b) and _rel(a, b) < 2.5 * step


@pytest.mark.gpu
def test_layer_passes_it_on():
    torch.manual_seed(0)
    m = GatedDeltaNet(64, 2, 64, 64, gate='vector', whole_sequences=True).to('cuda', torch.bfloat16).eval()
    x = torch.randn(2, 8256, 64, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    with torch.no_grad():
        # the projections row by row, so that their library's choice of kernel is the same
        batch, alone = m.forward(torch.cat([x, x])), m.forward(torch.cat([x, x.flip(0)]))
    assert torch.equal(batch[0], alone[0]) and torch.equal(batch[1], alone[1])


def test_workspace_sizes():
    """Sizes on the CPU: the two agree but for the calls that may be split (per channel, in two that keep
    the bits, from 4,033 tokens on)."""
    L = _lib.load()
    for dtype, kind, B, T, H, split in [(1, 1, 1, LONGEST, 2, False), (1, 2, 1, 4032, 2, False), (1, 2, 1, 4033, 2, True),
                                        (1, 1, 1, LONGEST + 1, 2, True), (2, 2, 1, LONGEST + 1, 2, True),
                                        (0, 1, 1, LONGEST + 1, 2, False), (1, 1, 64, 9000, 16, False)]:
        for name, dv in (('', []), ('_bwd', [128])):
            size = [getattr(L, f'vgdr_chunk{name}{whole}_workspace_size')(dtype, kind, B, T, H, 128, *dv, B, 0, 64)
                    for whole in ('', '_whole')]
            assert (size[0] > size[1] > 0) if split else (size[0] == size[1] > 0)
