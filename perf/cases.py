"""The framework's timed cases: what its users have it do, through its public
entry points.

    scan         the chunked scans of prefill (ops.chunk_gated_delta_rule,
                 ops.chunk_kda), dense or packed
    scan_train   the same scans with their gradients, through autograd
    layer_train  a GatedDeltaNet layer's training pass: output, input gradient
                 and every weight's gradient
    layer_decode one token through a layer's streaming decode_step, eagerly
    lm_decode    one token for every stream through a language model, replayed
                 from a recorded graph as a serving loop does
    lm_prefill   ragged prompts, packed, through a language model

``exact`` computes the same in 64 bits in plain torch on the same inputs.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from vagus_amd import ops
from vagus_amd.layer import GatedDeltaNet
from vagus_amd.model import GDNLM
from vagus_amd.serving import DecodeGraph

DT = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
SIZE = {'bf16': 2, 'fp16': 2, 'fp32': 4}


def listed():
    return [
        # a small fp32 batch: the size of a unit check or of a toy model's layer
        dict(name='gdn_small_fp32', kind='scan', gate='scalar', dtype='fp32', B=2, T=256, H=4, dk=64, dv=64,
             fused=False, h0=False, packed=0),
        # one short prompt of an odd length through a 340M layer's KDA heads, producers in the kernel
        dict(name='kda_one_prompt', kind='scan', gate='vector', dtype='bf16', B=1, T=1000, H=4, dk=128, dv=256,
             fused=True, h0=False, packed=0),
        # a 340M layer's prefill of a batch, continuing from states
        dict(name='gdn_340m', kind='scan', gate='scalar', dtype='bf16', B=8, T=4096, H=8, dk=128, dv=128,
             fused=False, h0=True, packed=0),
        # the per-channel gate over longer sequences
        dict(name='kda_prefill', kind='scan', gate='vector', dtype='bf16', B=4, T=8192, H=8, dk=128, dv=128,
             fused=False, h0=False, packed=0),
        # ragged prompts packed into one stream, a 1.3B layer's heads
        dict(name='gdn_varlen', kind='scan', gate='scalar', dtype='bf16', B=1, T=8192, H=16, dk=128, dv=128,
             fused=False, h0=False, packed=32, shortest=128, mix=3),
        # one long document through a 1.3B layer's heads
        dict(name='gdn_long_prompt', kind='scan', gate='scalar', dtype='bf16', B=1, T=32768, H=16, dk=128, dv=128,
             fused=False, h0=False, packed=0),
        # the scan's share of a 340M layer's training pass
        dict(name='gdn_340m_train', kind='scan_train', gate='scalar', dtype='bf16', B=8, T=4096, H=8, dk=128, dv=128,
             fused=False, h0=True, packed=0),
        # a KDA layer's training pass: dim 1024, 4 heads of 128 / 256, 16 x 2048 tokens
        dict(name='kda_layer_train', kind='layer_train', gate='vector', dtype='bf16', B=16, T=2048, dim=1024, H=4,
             dk=128, dv=256, fused=True),
        # a GDN layer's training pass on a small batch of an odd length
        dict(name='gdn_layer_train_odd', kind='layer_train', gate='scalar', dtype='bf16', B=3, T=1001, dim=1024, H=8,
             dk=128, dv=128, fused=True),
        # a few streams' next token through one KDA layer, called eagerly: latency
        dict(name='kda_layer_decode', kind='layer_decode', gate='vector', dtype='bf16', B=4, dim=1024, H=4, dk=128,
             dv=256),
        # 64 streams' next token through layers of the 1.3B model's shape
        dict(name='lm_decode_b64', kind='lm_decode', gate='scalar', dtype='bf16', B=64, layers=4, dim=2048, H=16,
             dk=128, dv=128, vocab=32000),
        # 32 ragged prompts through layers of the 1.3B model's shape
        dict(name='lm_prefill_ragged', kind='lm_prefill', gate='scalar', dtype='bf16', packed=32, shortest=64, T=2048,
             mix=4, layers=2, dim=2048, H=16, dk=128, dv=128, vocab=32000),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['scan', 'scan', 'scan', 'scan_train', 'scan_train', 'layer_train', 'layer_train',
                       'layer_decode', 'lm_decode', 'lm_prefill'])
    gate = rng.choice(['scalar', 'scalar', 'vector'])
    dk, dv = rng.choice([(64, 64), (128, 128), (128, 128), (128, 256)])
    if kind in ('scan', 'scan_train'):
        dtype = rng.choice(['bf16', 'bf16', 'bf16', 'bf16', 'fp16', 'fp32' if gate == 'scalar' else 'bf16'])
        H = rng.choice([2, 4, 5, 8, 16])
        most = 32768 if dtype == 'fp32' else 262144 if (kind == 'scan_train' or gate == 'vector') else 524288
        packed = rng.choice([0, 0, rng.randint(2, 32)])
        T = min(_log(rng, 64, 32768), most // H)
        B = 1 if packed else _log(rng, 1, max(1, min(16, most // (T * H))))
        c = dict(kind=kind, gate=gate, dtype=dtype, B=B, T=T, H=H, dk=dk, dv=dv,
                 fused=dtype != 'fp32' and rng.random() < 0.5, h0=rng.random() < 0.5, packed=packed)
        if packed:
            c['T'] = min(T, 8192, 2 * most // (H * packed))
            c.update(shortest=rng.randint(1, c['T']), mix=rng.randint(0, 10 ** 6))
        return c
    dim = rng.choice([512, 1024, 2048] if kind != 'layer_train' else [512, 768, 1024])
    H = max(2, dim // dv)
    if kind == 'layer_train':
        T = _log(rng, 100, 8192)
        return dict(kind=kind, gate=gate, dtype='bf16', B=_log(rng, 1, max(1, min(16, 32768 // T))), T=T, dim=dim, H=H,
                    dk=dk, dv=dv, fused=rng.random() < 0.7)
    if kind == 'layer_decode':
        return dict(kind=kind, gate=gate, dtype='bf16', B=_log(rng, 1, 128), dim=dim, H=H, dk=dk, dv=dv)
    if kind == 'lm_decode':
        return dict(kind=kind, gate=gate, dtype='bf16', B=_log(rng, 1, 64), layers=rng.randint(2, 4), dim=dim, H=H,
                    dk=dk, dv=dv, vocab=32000)
    T = _log(rng, 64, 2048)
    return dict(kind=kind, gate=gate, dtype='bf16', packed=rng.randint(1, 32), shortest=rng.randint(8, T), T=T,
                mix=rng.randint(0, 10 ** 6), layers=rng.randint(1, 2), dim=dim, H=H, dk=dk, dv=dv, vocab=32000)


# --- inputs ------------------------------------------------------------------


def _lengths(c):
    gen = torch.Generator('cpu').manual_seed(c['mix'])
    return torch.randint(c['shortest'], c['T'] + 1, (c['packed'],), generator=gen).tolist()


def _cu(lens):
    return torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device='cuda')


def _scan_inputs(c, seed):
    """q, k unit vectors per head, v ~ N(0, 1), write strengths sigmoid(N), decays
    logsigmoid(N + 4); with `fused` what the layer's projections give instead: q, k
    not normalised, beta logits and (per channel) the gate's pre-activation with
    the layer's A_log and dt_bias."""
    gen = torch.Generator('cuda').manual_seed(seed)
    dt = DT[c['dtype']]

    def randn(*s):
        return torch.randn(*s, generator=gen, device='cuda')

    lens = _lengths(c) if c['packed'] else None
    B, T, N = (1, sum(lens), len(lens)) if lens else (c['B'], c['T'], c['B'])
    H, dk, dv = c['H'], c['dk'], c['dv']
    x = dict(q=randn(B, T, H, dk), k=randn(B, T, H, dk), v=randn(B, T, H, dv).to(dt), beta=randn(B, T, H),
             initial_state=0.1 * randn(N, H, dk, dv) if c['h0'] else None, cu_seqlens=_cu(lens) if lens else None)
    g = randn(B, T, H, dk) if c['gate'] == 'vector' else randn(B, T, H)
    flags = {}
    if c['fused']:
        x['q'], x['k'], x['beta'] = x['q'].to(dt), x['k'].to(dt), x['beta'].to(dt)
        flags = dict(use_qk_l2norm_in_kernel=True, use_beta_sigmoid_in_kernel=True)
    else:
        x['q'], x['k'] = (F.normalize(x[n], dim=-1).to(dt) for n in 'qk')
        x['beta'] = torch.sigmoid(x['beta'])
    if c['fused'] and c['gate'] == 'vector':
        u = torch.rand(H + H * dk, generator=gen, device='cuda')
        step = torch.exp(u[H:] * math.log(100.0) + math.log(1e-3))
        x.update(g=g.to(dt), A_log=(1 + 15 * u[:H]).log(), dt_bias=step + torch.log(-torch.expm1(-step)))
        flags['use_gate_in_kernel'] = True
    else:
        x['g'] = F.logsigmoid(g + 4)
    return x, flags, gen


def _layer(c, seed):
    torch.manual_seed(seed)
    with torch.device('cuda'):
        m = GatedDeltaNet(c['dim'], c['H'], c['dk'], c['dv'], gate=c['gate'], fused=c.get('fused', True))
    return m.to(DT[c['dtype']])


def _lm(c, seed):
    torch.manual_seed(seed)
    with torch.device('cuda'):
        m = GDNLM(vocab_size=c['vocab'], dim=c['dim'], layer_count=c['layers'], head_count=c['H'],
                  key_head_dim=c['dk'], value_head_dim=c['dv'], gate=c['gate'], la_fused=True)
    return m.to(DT[c['dtype']]).eval()


def _fill_caches(m, B, gen):
    """A stream's state and conv tails some way into its text."""
    for att in ([m] if isinstance(m, GatedDeltaNet) else [b.att for b in m.blocks]):
        att.state.copy_(0.1 * torch.randn(att.state.shape, generator=gen, device='cuda'))
        for t in (att.qp_cache, att.kp_cache, att.vp_cache):
            t.copy_(torch.randn(t.shape, generator=gen, device='cuda'))


def prepare(case, seed):
    c = case
    s = dict(case=c)
    if c['kind'] in ('scan', 'scan_train'):
        x, flags, gen = _scan_inputs(c, seed)
        s.update(x=x, flags=flags)
        if c['kind'] == 'scan_train':
            s['wrt'] = [n for n in ('q', 'k', 'v', 'g', 'beta', 'initial_state', 'A_log', 'dt_bias')
                        if x.get(n) is not None]
            for n in s['wrt']:
                x[n].requires_grad_()
            s['do'] = torch.randn(x['v'].shape, generator=gen, device='cuda').to(x['v'].dtype)
        return s
    gen = torch.Generator('cuda').manual_seed(seed)
    if c['kind'] == 'layer_train':
        s['m'] = _layer(c, seed)
        x = torch.randn(c['B'], c['T'], c['dim'], generator=gen, device='cuda').to(DT[c['dtype']])
        s['do'] = torch.randn(x.shape, generator=gen, device='cuda').to(x.dtype)
        s['x'] = x.requires_grad_()
        return s
    if c['kind'] == 'layer_decode':
        m = s['m'] = _layer(c, seed).eval()
        m.reset_cache(c['B'])
        _fill_caches(m, c['B'], gen)
        s['x'] = torch.randn(c['B'], 1, c['dim'], generator=gen, device='cuda').to(DT[c['dtype']])
        return s
    m = s['m'] = _lm(c, seed)
    if c['kind'] == 'lm_decode':
        m.reset_cache(c['B'])
        s['tokens'] = torch.randint(0, c['vocab'], (c['B'], 1), generator=gen, device='cuda')
        m.decode_step(s['tokens'])
        s['graph'] = DecodeGraph(lambda: m.decode_step(s['tokens']))
        _fill_caches(m, c['B'], gen)
        return s
    lens = _lengths(c)
    s['tokens'] = torch.randint(0, c['vocab'], (1, sum(lens)), generator=gen, device='cuda')
    s['cu'] = _cu(lens)
    m.reset_cache(len(lens))
    return s


def run(state):
    s = state
    c = s['case']
    if c['kind'] in ('scan', 'scan_train'):
        x = s['x']
        scan = ops.chunk_kda if c['gate'] == 'vector' else ops.chunk_gated_delta_rule
        o, S = scan(**x, **s['flags'], output_final_state=True)
        if c['kind'] == 'scan':
            return dict(o=o, S=S)
        grads = torch.autograd.grad(o, [x[n] for n in s['wrt']], s['do'])
        return dict(o=o.detach(), S=S.detach(), **{'d_' + n: d for n, d in zip(s['wrt'], grads)})
    m = s['m']
    if c['kind'] == 'layer_train':
        y = m(s['x'])
        names, params = zip(*m.named_parameters())
        grads = torch.autograd.grad(y, [s['x'], *params], s['do'])
        return dict(y=y.detach(), d_x=grads[0], **{'d_' + n: d for n, d in zip(names, grads[1:])})
    if c['kind'] == 'layer_decode':
        return dict(y=m.decode_step(s['x']), S=m.state)
    if c['kind'] == 'lm_decode':
        return dict(logits=s['graph'].replay(), states=[b.att.state for b in m.blocks])
    m.reset_cache(c['packed'])
    return dict(logits=m.prefill_packed(s['tokens'], s['cu']), states=[b.att.state for b in m.blocks])


# --- what a pass cannot do without ----------------------------------------------


def _tokens(c):
    return sum(_lengths(c)) if c.get('packed') else c['B'] * c.get('T', 1)


def _scan_work(c, tokens, seqs, train):
    """Operations of the chunked form in 64-token chunks; q, k, v, o, the gate, beta
    and the states once each (training: and their gradients)."""
    H, dk, dv, e = c['H'], c['dk'], c['dv'], SIZE[c['dtype']]
    flops = tokens * H * (6 * dk * dv + 2 * 64 * (3 * dk + 2 * dv))
    gate = (dk * (e if c.get('fused') else 4)) if c['gate'] == 'vector' else 4
    rows = tokens * H * (e * (2 * dk + dv) + gate + 4)
    states = 4 * seqs * H * dk * dv
    out = tokens * H * e * dv
    if train:
        return 3 * flops, 2 * rows + 2 * out + states * (3 if c.get('h0') else 1)
    return flops, rows + out + states * (2 if c.get('h0') else 1)


def _layer_weights(c):
    d, H, dk, dv = c['dim'], c['H'], c['dk'], c['dv']
    gates = d * H + (64 * (d + H * dk) if c['gate'] == 'vector' else d * H)
    return d * H * (2 * dk + 3 * dv) + gates


def work(case):
    c = case
    n = _tokens(c)
    e = SIZE[c['dtype']]
    if c['kind'] in ('scan', 'scan_train'):
        flops, nbytes = _scan_work(c, n, c['packed'] or c['B'], c['kind'] == 'scan_train')
        return dict(bytes=nbytes, flops=flops)
    H, dk, dv, w = c['H'], c['dk'], c['dv'], _layer_weights(c)
    scan = n * H * (6 * dk * dv + 2 * 64 * (3 * dk + 2 * dv))
    if c['kind'] == 'layer_train':
        return dict(bytes=e * (4 * n * c['dim'] + 2 * w), flops=3 * (2 * n * w + scan))
    states = 8 * c.get('B', c.get('packed', 0)) * H * dk * dv
    if c['kind'] == 'layer_decode':
        return dict(bytes=e * (2 * n * c['dim'] + w) + states, flops=n * (2 * w + 6 * H * dk * dv))
    hidden = math.ceil(int(8 * c['dim'] / 3) / 256) * 256
    w = c['layers'] * (w + 3 * c['dim'] * hidden)
    head = c['dim'] * c['vocab']
    out = n if c['kind'] == 'lm_decode' else c['packed']
    flops = 2 * n * w + 2 * out * head + c['layers'] * (n * 6 * H * dk * dv if c['kind'] == 'lm_decode' else scan)
    return dict(bytes=e * (w + head + out * c['vocab']) + c['layers'] * states, flops=flops)


def tolerance(case):
    # about four times the distance from `exact` that was measured: 2e-7 (fp32 scans), 3e-3 to 5e-3 (16-bit
    # scans, a layer's decode step), 1e-2 (a layer's weight gradients), 1e-2 to 2e-2 (two to four layers of a model)
    if case['dtype'] == 'fp32':
        return {'rel': 1e-5}
    if case['kind'] in ('lm_prefill', 'lm_decode', 'layer_train'):
        return {'rel': 3e-2}
    return {'rel': 1.6e-2}


# --- the same in 64 bits ----------------------------------------------------------


def _scan64(q, k, v, g, beta, S, scale):
    """The gated delta rule S_t = (I - beta k k^T) diag(a) S_{t-1} + beta k v^T,
    o_t = scale q_t S_t, over chunks, in q's 64-bit type.  q, k (B, T, H, dk), v (B, T, H,
    dv), g (B, T, H) or (B, T, H, dk), beta (B, T, H), S (B, H, dk, dv)."""
    B, T, H, dk = q.shape
    vec = g.dim() == 4
    C = 16 if vec else 64
    n = -(-T // C)

    def chunks(x):
        x = x if x.dim() == 4 else x[..., None]
        x = F.pad(x, (0, 0, 0, 0, 0, n * C - T))
        return x.view(B, n, C, H, x.shape[-1]).permute(1, 0, 3, 2, 4).contiguous()   # (n, B, H, C, d)

    q, k, v, beta = chunks(q * scale), chunks(k), chunks(v), chunks(beta)
    y = chunks(g).cumsum(3)                                                       # decay from the chunk's start
    low = torch.ones(C, C, dtype=torch.bool, device=q.device).tril()
    if vec:
        A, M = [], []
        for i in range(n):                                                         # exact pairwise decays
            E = torch.exp((y[i][..., :, None, :] - y[i][..., None, :, :]).masked_fill(~low[:, :, None], -1e30))
            E = E * k[i][..., None, :, :]
            A.append((E * q[i][..., :, None, :]).sum(-1))
            M.append((E * k[i][..., :, None, :]).sum(-1))
        A, M = torch.stack(A), torch.stack(M)
    else:
        D = torch.exp((y - y.transpose(-1, -2)).masked_fill(~low, -1e30))
        kt = k.transpose(-1, -2).contiguous()
        A, M = q @ kt * D, k @ kt * D
    A = A.tril()
    N = -(beta * M).tril(-1)
    inv = torch.eye(C, dtype=q.dtype, device=q.device).expand_as(N)
    for _ in range(int(math.log2(C))):                                             # (I - N)^-1, N nilpotent
        inv = inv + N @ inv
        N = N @ N
    decay = y.exp()
    kin, qin = k * decay, q * decay
    kout = (k * torch.exp(y[..., -1:, :] - y)).transpose(-1, -2).contiguous()
    end = decay[..., -1, :, None]                                                  # (n, B, H, dk or 1, 1)
    outs = []
    for i in range(n):
        u = inv[i] @ (beta[i] * (v[i] - kin[i] @ S))
        outs.append(qin[i] @ S + A[i] @ u)
        S = end[i] * S + kout[i] @ u
    o = torch.stack(outs, 1).permute(0, 1, 3, 2, 4).reshape(B, n * C, H, -1)[:, :T]
    return o, S


def _unpack(x, lens):
    """(1, sum, ...) -> (N, longest, ...), zeros after each sequence."""
    return torch.nn.utils.rnn.pad_sequence(x[0].split(lens), batch_first=True)


def _pack(x, lens):
    return torch.cat([x[i, :n] for i, n in enumerate(lens)])[None]


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _gate64(f, A_log, dt_bias):
    H = A_log.numel()
    if f.dim() == 4:
        return -A_log.exp()[:, None] * F.softplus(f + dt_bias.view(H, -1))
    return -A_log.exp() * F.softplus(f + dt_bias)


def _conv64(x, w, tail=None):
    """SiLU of the causal depthwise conv; tail (B, K, D): the inputs before x."""
    K = w.shape[-1]
    T = x.shape[1]
    x = F.pad(x, (0, 0, K - 1, 0)) if tail is None else torch.cat([tail[:, 1:], x], 1)
    return F.silu(sum(x[:, j:j + T] * w[:, 0, j] for j in range(K)))


def _layer64(p, x, c, S=None, tails=(None, None, None), lens=None):
    """GatedDeltaNet in 64 bits: x (B, T, dim), parameters p by name.  lens: only the
    first lens[i] tokens of row i are real (the others leave the state alone)."""
    B, T, H, dk, dv = x.shape[0], x.shape[1], c['H'], c['dk'], c['dv']
    q, k, v = (_conv64(x @ p[f'w{n}.weight'].T, p[f'conv_{n}.conv.weight'], t) for n, t in zip('qkv', tails))
    q, k, v = _unit(q.view(B, T, H, dk)), _unit(k.view(B, T, H, dk)), v.view(B, T, H, dv)
    if c['gate'] == 'vector':
        f = (x @ p['wa1.weight'].T @ p['wa2.weight'].T).view(B, T, H, dk)
    else:
        f = x @ p['wa.weight'].T
    g, beta = _gate64(f, p['A_log'], p['dt_bias']), torch.sigmoid(x @ p['wb.weight'].T)
    if lens is not None:
        pad = torch.arange(T, device=x.device) >= torch.tensor(lens, device=x.device)[:, None]
        beta = beta.masked_fill(pad[..., None], 0)
        g = g.masked_fill(pad.view(B, T, *[1] * (g.dim() - 2)), 0)
    S = x.new_zeros(B, H, dk, dv) if S is None else S
    o, S = _scan64(q, k, v, g, beta, S, dk ** -0.5)
    o = _rms64(o, p['o_norm.gamma']) * F.silu((x @ p['wg.weight'].T).view(B, T, H, dv))
    return o.reshape(B, T, H * dv) @ p['wo.weight'].T, S


def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w


def exact(case, seed):
    c = case
    s = prepare(case, seed)
    up = lambda t: None if t is None else t.detach().double()  # noqa: E731
    if c['kind'] in ('scan', 'scan_train'):
        train = c['kind'] == 'scan_train'
        x = {n: up(s['x'].get(n)) for n in ('q', 'k', 'v', 'g', 'beta', 'initial_state', 'A_log', 'dt_bias')}
        if train:
            for n in s['wrt']:
                x[n].requires_grad_()
        q, k, g, beta = x['q'], x['k'], x['g'], x['beta']
        if c['fused']:
            q, k, beta = _unit(q), _unit(k), torch.sigmoid(beta)
            g = _gate64(g, x['A_log'], x['dt_bias']) if c['gate'] == 'vector' else g
        a = [q, k, x['v'], g, beta]
        lens = _lengths(c) if c['packed'] else None
        if lens:
            a = [_unpack(t, lens) for t in a]
        S0 = x['initial_state']
        S0 = a[0].new_zeros(a[0].shape[0], c['H'], c['dk'], c['dv']) if S0 is None else S0
        o, S = _scan64(*a, S0, c['dk'] ** -0.5)
        o = _pack(o, lens) if lens else o
        if not train:
            return dict(o=o, S=S)
        grads = torch.autograd.grad(o, [x[n] for n in s['wrt']], up(s['do']))
        return dict(o=o.detach(), S=S.detach(), **{'d_' + n: d for n, d in zip(s['wrt'], grads)})
    m = s['m']
    p = {n: up(t) for n, t in m.named_parameters()}
    if c['kind'] == 'layer_train':
        x = up(s['x']).requires_grad_()
        for t in p.values():
            t.requires_grad_()
        y, _ = _layer64(p, x, c)
        grads = torch.autograd.grad(y, [x, *p.values()], up(s['do']))
        return dict(y=y.detach(), d_x=grads[0], **{'d_' + n: d for n, d in zip(p, grads[1:])})
    if c['kind'] == 'layer_decode':
        y, S = _layer64(p, up(s['x']), c, up(m.state), [up(t) for t in (m.qp_cache, m.kp_cache, m.vp_cache)])
        return dict(y=y, S=S)
    decode = c['kind'] == 'lm_decode'
    lens = None if decode else _lengths(c)
    table = p['embedding.weight']
    x = table[s['tokens'] if decode else _unpack(s['tokens'], lens)]
    states = []
    with torch.no_grad():
        for i, b in enumerate(m.blocks):
            w = {n.removeprefix(f'blocks.{i}.att.'): t for n, t in p.items() if n.startswith(f'blocks.{i}.att.')}
            old = [up(t) for t in (b.att.state, b.att.qp_cache, b.att.kp_cache, b.att.vp_cache)] if decode else None
            y, S = _layer64(w, _rms64(x, p[f'blocks.{i}.rmsnorm1.gamma']), c, old[0] if decode else None,
                            old[1:] if decode else (None,) * 3, lens)
            states.append(S)
            x = x + y
            a, gate = (_rms64(x, p[f'blocks.{i}.rmsnorm2.gamma']) @ p[f'blocks.{i}.ffn.l1.weight'].T).chunk(2, -1)
            x = x + (F.silu(a) * gate) @ p[f'blocks.{i}.ffn.l2.weight'].T
        if not decode:
            x = x[torch.arange(len(lens), device=x.device), torch.tensor(lens, device=x.device) - 1]
        return dict(logits=_rms64(x, p['rms_head.gamma']) @ table.T, states=states)
