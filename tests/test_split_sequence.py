"""Dense calls of few (sequence, head) pairs and more than 8,192 tokens, whose
sequences the chunked scan splits into segments walked side by side: against the
fp64 oracle, and against the same tokens as a packed batch, which is never
split.  The decays are weak (a few per cent over a whole sequence), so that
every segment depends on its entry state.

Split and unsplit runs round the same quantities to the element type in the
same places, so their errors are of one size: the split run's may be at most
1.25 times the unsplit run's."""
import pytest
import torch

from oracle import gdr
from vagus_amd import _lib, ops, workloads

pytestmark = pytest.mark.gpu


def rel(x, ref):
    x, ref = x.double().cpu(), ref.double().cpu()
    return ((x - ref).norm() / ref.norm().clamp_min(1e-30)).item()


def inputs(B, T, H, dk, dv, gate, dtype, seed):
    x = workloads.make_inputs(B, T, H, dk, dv, gate='scalar' if gate == 'none' else gate, dtype=dtype, s0_scale=1.0,
                              seed=seed)
    x.g = None if gate == 'none' else 1e-3 * x.g
    return x


def segment_bytes(gate, dtype, B, T, H, dk, dv):
    """What this very call keeps between segments (the backward's workspace size takes dv, and has the plan's own
    bytes); 0 when it is not split."""
    L = _lib.load()
    kind = {'none': _lib.VGDR_GATE_NONE, 'scalar': _lib.VGDR_GATE_SCALAR, 'vector': _lib.VGDR_GATE_VECTOR}[gate]
    call = ops._DTYPES[dtype], kind, B, T, H, dk, dv, B, 0, 64
    return L.vgdr_chunk_bwd_workspace_size(*call) - L.vgdr_chunk_bwd_whole_workspace_size(*call)


def run(x, gate, packed, grads=None):
    """(o, S), or with grads (do, dS) the gradients too; packed: the sequences as one packed batch."""
    B, T = x.q.shape[:2]
    t = [None if a is None else a.cuda().requires_grad_(grads is not None)
         for a in (x.q, x.k, x.v, x.g, x.beta, x.initial_state)]
    flat = [a.reshape(1, B * T, *a.shape[2:]) if packed and a is not None else a for a in t[:5]]
    cu = torch.arange(0, B * T + 1, T, dtype=torch.int32, device='cuda') if packed else None
    fn = ops.chunk_kda if gate == 'vector' else ops.chunk_gated_delta_rule
    o, S = fn(*flat, initial_state=t[5], output_final_state=True, cu_seqlens=cu)
    out = [o.reshape(B, T, *o.shape[2:]), S]
    if grads is not None:
        wrt = [a for a in t if a is not None]
        out += torch.autograd.grad(out, wrt, [g.cuda() for g in grads])
    return [a.detach() for a in out]


# a last chunk of one token; dv past a tile's end and under one; two sequences; two segments (no entry-state chain)
@pytest.mark.parametrize('gate,dtype,B,T,H,dk,dv', [
    ('scalar', torch.bfloat16, 1, 8193, 1, 128, 128),
    ('scalar', torch.bfloat16, 1, 8200, 16, 128, 128),
    ('scalar', torch.float16, 2, 8257, 2, 64, 48),
    ('none', torch.bfloat16, 1, 9000, 3, 64, 16),
    ('none', torch.float16, 1, 10001, 2, 128, 256),
    ('vector', torch.bfloat16, 1, 8193, 3, 128, 128),
    ('vector', torch.bfloat16, 4, 8200, 8, 128, 128),
    ('vector', torch.bfloat16, 4, 4100, 8, 128, 128),
    ('vector', torch.bfloat16, 1, 4033, 3, 128, 128),
    ('vector', torch.float16, 1, 8600, 2, 128, 272),
    ('vector', torch.bfloat16, 2, 8224, 1, 64, 64),
])
def test_split_against_oracle_and_packed(gate, dtype, B, T, H, dk, dv):
    assert segment_bytes(gate, dtype, B, T, H, dk, dv) > 0, 'this call is not split'
    x = inputs(B, T, H, dk, dv, gate, dtype, seed=T)
    up = lambda a: None if a is None else a.double()  # noqa: E731
    ref = gdr.recurrent(up(x.q), up(x.k), up(x.v), up(x.g), up(x.beta), x.initial_state.double(), scale=dk ** -0.5)
    split, whole = run(x, gate, False), run(x, gate, True)
    # two segments have no M and are the unsplit chain in two places at once: the same bits
    two = segment_bytes(gate, dtype, B, T, H, dk, dv) < 2 * 4 * B * H * dk * dv
    assert two == (T <= 8192 or B * H == 32) and torch.equal(split[0], whole[0]) == two
    for name, a, b, r in zip(('o', 'S'), split, whole, ref):
        ea, eb = rel(a, r), rel(b, r)
        print(f'[split] {gate} {dtype} {B}x{T}x{H} {dk}/{dv}: {name} {ea:.2e}, unsplit {eb:.2e}', flush=True)
        assert ea < 2e-2 and ea <= 1.25 * eb


@pytest.mark.parametrize('gate,dtype,H,dk,dv', [
    ('scalar', torch.bfloat16, 2, 128, 128),
    ('scalar', torch.float16, 16, 64, 80),
    ('vector', torch.bfloat16, 2, 128, 64),
])
def test_split_training_pass(gate, dtype, H, dk, dv):
    """The entry states that the forward leaves for the backward: every gradient against the unsplit run's.
    Each run is within about a rounding of the element type (2^-8, 2^-11) of the exact gradients, so
    the two are within 2.5 of them of each other."""
    tol = 2.5 * (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11)
    x = inputs(1, 8300, H, dk, dv, gate, dtype, seed=9)
    assert segment_bytes(gate, dtype, 1, 8300, H, dk, dv) > 0, 'this call is not split'
    g = torch.Generator().manual_seed(10)
    grads = torch.randn(x.v.shape, generator=g).to(dtype), torch.randn(x.initial_state.shape, generator=g)
    for i, (a, b) in enumerate(zip(run(x, gate, False, grads), run(x, gate, True, grads))):
        e = rel(a, b)
        print(f'[split] {gate} {dtype} training output {i}: {e:.2e}', flush=True)
        assert e < tol


def test_workspace_without_room_runs_unsplit():
    """The size a workspace had before sequences were split is still taken: the same result up to rounding,
    and one byte less is refused."""
    T, H, d = 8256, 2, 128
    x = inputs(1, T, H, d, d, 'scalar', torch.bfloat16, seed=3)
    y = {n: getattr(x, n).cuda() for n in ('q', 'k', 'v', 'g', 'beta', 'initial_state')}
    L = _lib.load()
    full = L.vgdr_chunk_workspace_size(1, 1, 1, T, H, d, 1, 0, 64)
    least = L.vgdr_chunk_whole_workspace_size(1, 1, 1, T, H, d, 1, 0, 64)
    assert least == T // 64 * L.vgdr_chunk_workspace_size(1, 1, 1, 64, H, d, 1, 0, 64) < full

    def call(nbytes):
        o, S = torch.empty_like(y['v']), torch.empty_like(y['initial_state'])
        ws = torch.empty(nbytes, dtype=torch.uint8, device='cuda')
        p = lambda n: y[n].data_ptr()  # noqa: E731
        rc = L.vgdr_chunk_fwd(1, 1, 1, p('q'), p('k'), p('v'), p('g'), p('beta'), o.data_ptr(), p('initial_state'),
                              S.data_ptr(), None, ws.data_ptr(), nbytes, 1, T, H, d, d, 1, d ** -0.5, 64,
                              torch.cuda.current_stream().cuda_stream)
        return rc, o, S

    (rc, o, S), (rc1, o1, S1) = call(full), call(least)
    assert rc == 0 and rc1 == 0 and call(least - 1)[0] == _lib.VGDR_ERR_INVALID
    whole = run(x, 'scalar', True)
    assert torch.equal(o1, whole[0]) and torch.equal(S1, whole[1])
    assert rel(o, o1) < 2.5 * 2 ** -8 and rel(S, S1) < 2.5 * 2 ** -8      # two runs, each about 2^-8 from exact
