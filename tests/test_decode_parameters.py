"""The one-token decode step reads its parameters where they lie: a change of
any of them reaches the next step, and the next replay of a recorded graph,
however it was written (p.data.copy_ changes neither a parameter's
storage nor its version), and the projections behind it (ops.project_rows)
against fp64.

Bars: a step after a change is bit-equal to the same step of a layer made from the
changed parameters; projections within half an ulp of the element type
(2^-9 for bf16, 2^-12 for fp16; twice that for a sum's own error), fp32 1e-5, the
repository's fp32 bar, which also holds the gate in fp32.
"""
import copy

import pytest
import torch
import torch.nn.functional as F

from vagus_amd.layer import GatedDeltaNet

SIZES = [(64, 128), (128, 128), (128, 256)]


def _layer(gate, dk, dv, dtype, device, *, delta=True, H=2, dim=256, seed=0, rank=20):
    torch.manual_seed(seed)
    m = GatedDeltaNet(dim=dim, head_count=H, key_head_dim=dk, value_head_dim=dv, gate=gate, delta=delta, gate_rank=rank)
    for lin in (m.wq, m.wk, m.wv, m.wg):
        torch.nn.init.normal_(lin.weight, std=dim ** -0.5)
    return m.to(device=device, dtype=dtype).eval()


def _rewrite(m, seed):
    """Every parameter overwritten through .data."""
    g = torch.Generator().manual_seed(seed)
    for p in m.parameters():
        p.data.copy_(p.data.cpu().float() * (0.5 + torch.rand(p.shape, generator=g)))


# 300: more streams than the projection kernel takes; with a rank of 22 and two heads the stacked rows are whole 16-byte units,
# with 20 they are not
@pytest.mark.parametrize('gate', ['scalar', 'vector', 'none'])
@pytest.mark.parametrize('dk,dv', SIZES)
@pytest.mark.parametrize('streams,rank', [(3, 20), (300, 22), (300, 20)])
def test_projections_follow_data_writes(gate, dk, dv, streams, rank):
    """On the CPU: the decode step's inputs before and after the change."""
    m = _layer(gate, dk, dv, torch.float32, 'cpu', rank=rank)
    x = torch.randn(streams, 1, 256, generator=torch.Generator().manual_seed(1))
    with torch.no_grad():
        m._decode_inputs(x)
        _rewrite(m, 2)
        got = m._decode_inputs(x)
        for y, w in zip(got, (m.wq, m.wk, m.wv, m.wg)):
            assert torch.allclose(y, w(x), atol=1e-5, rtol=1e-5)
        if got[6] is None:                                      # else the decode kernel forms it from the parameters
            assert torch.allclose(got[5].float(), m.wb(x), atol=1e-5, rtol=1e-5)
        else:
            assert gate == 'scalar' and all(a is b for a, b in zip(got[6], (x, m.wa.weight, m.wb.weight, m.A_log, m.dt_bias)))
        if gate == 'vector':
            assert torch.allclose(got[4].flatten(2), m.wa2(m.wa1(x)), atol=1e-5, rtol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('gate,delta', [('scalar', True), ('scalar', False), ('vector', True), ('none', True)])
@pytest.mark.parametrize('dk,dv,streams', [(*s, 3) for s in SIZES] + [(128, 128, 300)])
def test_decode_step_follows_data_writes(dtype, gate, delta, dk, dv, streams):
    m = _layer(gate, dk, dv, dtype, 'cuda', delta=delta, rank=22)
    x = torch.randn(streams, 4, 256, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    m.reset_cache(streams)
    m.decode_step(x[:, :1])
    for t in range(1, 4):
        _rewrite(m, t)
        fresh = copy.deepcopy(m)
        for k in [k for k in fresh.__dict__ if k not in GatedDeltaNet(8, 1, 8, 8).__dict__]:
            del fresh.__dict__[k]                               # nothing that an earlier step left
        assert torch.equal(m.decode_step(x[:, t:t + 1]), fresh.decode_step(x[:, t:t + 1])), t
        assert torch.equal(m.state, fresh.state)


@pytest.mark.gpu
@pytest.mark.parametrize('gate', ['scalar', 'vector', 'none'])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_large_batches_step_as_small_ones(gate, dtype):
    """More streams than the projection kernel takes, against the same streams in two batches."""
    m = _layer(gate, 128, 128, dtype, 'cuda', rank=22)
    x = torch.randn(300, 3, 256, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()

    def steps(x):
        m.reset_cache(x.shape[0])
        y = torch.cat([m.decode_step(x[:, t:t + 1]) for t in range(3)], 1)
        return y, m.state.clone()

    tol = 1e-5 if dtype == torch.float32 else 2e-2
    halves = [steps(h) for h in (x[:150], x[150:])]
    for a, b in zip(steps(x), (torch.cat(t) for t in zip(*halves))):
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() < tol


@pytest.mark.gpu
@pytest.mark.parametrize('gate,dk,dv', [('vector', 128, 256), ('vector', 128, 128), ('scalar', 128, 128),
                                        ('scalar', 64, 128)])
def test_recorded_step_follows_parameter_changes(gate, dk, dv):
    """A graph recorded over the step, replayed after in-place changes of every parameter (through
    load_state_dict and through .data), with eager steps of other layers between the replays."""
    from vagus_amd.serving import DecodeGraph
    m = _layer(gate, dk, dv, torch.bfloat16, 'cuda')
    x = torch.randn(3, 1, 256, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    m.reset_cache(3)
    m.decode_step(x)
    graph = DecodeGraph(lambda: m.decode_step(x))
    for t in range(4):
        if t % 2:
            _rewrite(m, t)
        else:
            m.load_state_dict({n: v * (1 + 0.1 * t) for n, v in m.state_dict().items()})
        fresh = copy.deepcopy(m)
        want = fresh.decode_step(x)
        torch.cuda.synchronize()
        assert torch.equal(graph.replay(), want) and torch.equal(m.state, fresh.state), t
        x.copy_(-0.9 * x + 0.1)


# one row and row; rows that fill and overflow 16, 32 and 64, and a second block of 64; rows shorter than
# a unit of 64 k and with a part of one; widths under, at and over a tile of 16, 32 and 64; grids for each of the
# three tile shapes
@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('rows,dim,widths', [(1, 8, [1]), (4, 1024, [512, 1024, 64]), (16, 72, [16, 17, 3, 40]),
                                             (17, 264, [33, 64]), (33, 2048, [128, 20]), (64, 128, [4096, 4096, 4096]),
                                             (65, 136, [65, 4]), (130, 64, [8192, 8192]), (256, 200, [48])])
@pytest.mark.parametrize('view', [False, True])
def test_project_rows(dtype, rows, dim, widths, view):
    from vagus_amd import ops
    print(f'\n[case] project_rows {dtype} rows={rows} dim={dim} widths={widths} view={view}', flush=True)
    g = torch.Generator('cuda').manual_seed(rows + dim)
    randn = lambda *s: torch.randn(*s, generator=g, device='cuda')  # noqa: E731
    x = randn(rows, dim + (16 if view else 0)).to(dtype)[:, 8 if view else 0:][:, :dim]
    ws = [(dim ** -0.5 * randn(n, dim)).to(dtype) for n in widths]
    w_b = (dim ** -0.5 * randn(5, dim)).to(dtype)
    assert ops.project_rows_fits(x, ws + [w_b])
    y, at, beta = ops.project_rows(x, ws, w_b)
    tol = {torch.float32: 1e-5, torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[dtype]

    def check(got, want, tol):
        e = ((got.double() - want).norm() / want.norm()).item()
        print(f'[parity] rel_l2={e:.3e}', flush=True)
        assert got.shape == want.shape and e <= tol

    lin = lambda w: x.double() @ w.double().T.contiguous()  # noqa: E731
    for w, c in zip(ws, at):
        assert c % 8 == 0
        check(y[:, c:c + w.shape[0]], lin(w), tol)
    check(beta, lin(w_b), tol)
    assert torch.equal(beta, beta.to(dtype).float())


# the gate's parameters in the module's type and in fp32 (the decode kernel reads both), a lower-bounded gate,
# and a head too wide for the kernel's own gate projections (dim 4096 in fp32): the module's values
@pytest.mark.gpu
@pytest.mark.parametrize('gate,dim,kw', [('scalar', 256, {}), ('vector', 256, {}), ('scalar', 4096, {}),
                                         ('vector', 256, {'gate_lower_bound': -5.0})])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('fp32_constants', [False, True])
def test_gate_parameters_in_the_decode_kernel(gate, dim, kw, dtype, fp32_constants):
    from vagus_amd import ops
    torch.manual_seed(3)
    m = GatedDeltaNet(dim=dim, head_count=2, key_head_dim=128, value_head_dim=128, gate=gate, **kw).to('cuda', dtype)
    if fp32_constants:
        m.A_log.data, m.dt_bias.data = m.A_log.data.float(), m.dt_bias.data.float()
    x = torch.randn(3, 1, dim, generator=torch.Generator().manual_seed(4)).to(dtype).cuda()
    with torch.no_grad():
        qp, kp, vp, og, g, beta, gp = m._decode_inputs(x)
        assert (gp is not None) == (gate == 'scalar')
        want_g, want_b = m._gates(x, raw_beta=True)
        s1, s2 = (torch.randn(3, 2, 128, 128, generator=torch.Generator().manual_seed(5)).cuda() for _ in range(2))
        caches = [[torch.zeros(3, 4, 256, dtype=dtype, device='cuda') for _ in range(3)] for _ in range(2)]
        step = dict(scale=0.1, conv_weights=m._conv_weights(), beta_logits=True, out_gate=og,
                    out_norm_weight=m.o_norm.gamma)
        vec = dict(gate_in_kernel=True, A_log=m.A_log, dt_bias=m.dt_bias,
                   lower_bound=m.gate_lower_bound) if gate == 'vector' else {}
        a = ops.hip_decode_step(qp, kp, vp, g, beta, s1, conv_cache=caches[0], gate_proj=gp, **step, **vec)
        b = ops.hip_decode_step(qp, kp, vp, want_g, want_b, s2, conv_cache=caches[1], **step)
    # the projections' sums differ in order: a rounding of the element type in the gate's exponent
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    for got, want in ((a, b), (s1, s2)):
        e = ((got.double() - want.double()).norm() / want.double().norm()).item()
        print(f'[parity] {gate} {dtype} rel_l2={e:.3e}', flush=True)
        assert e <= tol


def test_project_rows_checks_its_arguments():
    """Refused by the host before anything is launched."""
    import ctypes

    from vagus_amd import _lib
    L = _lib.load()

    def call(dtype=1, n=(16, 16), w=(4096, 8192), x=256, ldx=64, y=512, ldy=32, beta_mat=-1, beta=None, rows=1, dim=64):
        c = len(n)
        return L.vgdr_project_rows(dtype, c, (ctypes.c_void_p * max(c, 1))(*w[:c]), (ctypes.c_int64 * max(c, 1))(*n), x, ldx,
                                   y, ldy, beta_mat, beta, rows, dim, None)

    bad = _lib.VGDR_ERR_INVALID
    assert call(rows=0) == _lib.VGDR_OK
    assert call(dtype=7) == bad and call(n=(), w=()) == bad and call(n=(1,) * 9, w=(16,) * 9) == bad
    assert call(dim=60) == _lib.VGDR_ERR_UNSUPPORTED and call(dim=0) == _lib.VGDR_ERR_UNSUPPORTED
    assert call(ldx=56) == bad and call(ldx=68) == bad and call(x=264) == bad and call(x=None) == bad
    assert call(ldy=24) == bad and call(y=None) == bad and call(y=520) == bad
    assert call(w=(4096, 8200)) == bad and call(w=(4096, None)) == bad and call(w=(4096, 512)) == bad
    assert call(beta_mat=2, beta=64) == bad and call(beta_mat=1) == bad              # no such matrix; nowhere to put it


def test_decode_step_params_checks_its_arguments():
    import ctypes

    from vagus_amd import _lib
    L = _lib.load()
    sc = _lib.ShortConv(weight_q=16, weight_k=16, weight_v=16, cache_q=16, cache_k=16, cache_v=16, kernel_size=4,
                        weight_dtype=1)

    def call(gate=1, fusion=None, ld=256, h0=16, **kw):
        pm = _lib.GateParams(**{**dict(x=16, w_a=16, w_b=16, A_log=16, dt_bias=16, dim=64, param_dtype=1), **kw})
        return L.vgdr_decode_step_params(1, gate, 1, 16, 16, 16, 16, 16, 16, h0, h0, 0, 2, 128, 128, ld, 256, 1.0,
                                         None if fusion is None else ctypes.byref(fusion), ctypes.byref(sc), None,
                                         ctypes.byref(pm), None)

    bad = _lib.VGDR_ERR_INVALID
    assert call() == _lib.VGDR_OK                                                    # no tokens: nothing to launch
    assert call(A_log=None) == bad and call(dt_bias=None) == bad and call(param_dtype=3) == bad
    assert call(x=None) == bad and call(w_a=8) == bad and call(w_b=None) == bad and call(ld=128) == bad
    assert call(dim=60) == _lib.VGDR_ERR_UNSUPPORTED and call(h0=None) == _lib.VGDR_ERR_UNSUPPORTED
    assert call(gate=0) == _lib.VGDR_ERR_UNSUPPORTED and call(gate=2) == _lib.VGDR_ERR_UNSUPPORTED
    fz = _lib.Fusion(0, 0, 1, 1, None, None, 0, 0.0)
    assert call(gate=2, fusion=fz) == _lib.VGDR_OK
