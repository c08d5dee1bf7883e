"""Performance cases of the block-sparse operators.

A case is one pass that a user's program makes through the public operators: a sparse linear
layer in inference and in a training step, a feed-forward block whose masks change every step,
sparse attention in inference and in a training step, attention over sequence lengths, and a
mixture-of-experts layer.  `listed()` names the sizes that are always looked at, `draw()` gives
others of the same ranges.

The kinds and their fields:

  linear       SparseLinear(weight_mask) forward.         M rows, K -> N, blocks bn x bk of the [N, K] weight
  linear_step  the same layer, forward + backward         (gradients of input, weight and bias)
  ffn          two dynamic layers K -> N -> K with a relu between them; both masks change before every pass
  attention    SparseAttention forward                    heads (batch x heads), Nt queries, Ns keys, head dim E
  attention_step   forward + backward                     (gradients of query, key and value)
  seqlen       SeqlenDynamicSparseAttention               batch, heads, N positions, E
  moe          DynamicSparseMoE                           tokens, K -> N, experts

Masks keep an exact number of blocks at random places, so that the work of a case does not depend
on the seed.
"""
import math

import numpy as np
import torch

import sparta_amd as sparta

_DTYPES = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16}
_BYTES = {'f32': 4, 'f16': 2, 'bf16': 2}


# ---- the cases --------------------------------------------------------------------------------
def listed():
    return [
        # one sequence of a few tokens through a pruned projection of a BERT-base layer: a launch
        # and its host path, nothing else
        _linear('linear_few_rows', 16, 768, 3072, 32, 32, 0.90, 'f16', bias=True),
        # the example of the README: fp32, 8x8-granular mask at 90 % (35 % of the 16x16 tiles are live)
        _linear('linear_readme', 1024, 1024, 1024, 16, 16, 0.65, 'f32', bias=True),
        # the headline workload: 4096^3, 32x32 blocks, 95 % sparse
        _linear('linear_4096', 4096, 4096, 4096, 32, 32, 0.95, 'f16'),
        # fine-tuning of a pruned projection; the token count of a packed batch is no round number
        _linear('linear_step_bf16', 2992, 768, 3072, 32, 64, 0.90, 'bf16', bias=True, kind='linear_step'),
        # the notebook example of the linear operator as a training step: fp32, 80 % sparse
        _linear('linear_step_f32', 4096, 3072, 768, 32, 32, 0.80, 'f32', bias=True, kind='linear_step'),
        # dynamic-mask feed-forward block of BERT-base, both indexes rebuilt in every pass
        dict(name='ffn_dynamic', kind='ffn', M=8192, K=768, N=3072, bn=32, bk=64, sparsity=0.90, dtype='f16'),
        # a short causal window: 12 heads of one sequence of 512 tokens, element-level causal mask
        _attention('attention_short', 12, 512, 512, 64, 64, 2, 0.0, True, 'bf16'),
        # local window of 256 tokens + 2 % random blocks, 8 x 12 heads x 4096 tokens
        _attention('attention_long', 96, 4096, 4096, 64, 64, 5, 0.02, False, 'f16'),
        # the same problem as a training step
        _attention('attention_step_f16', 96, 4096, 4096, 64, 64, 5, 0.02, False, 'f16', kind='attention_step'),
        # the notebook example of the attention operator: fp32, one head of 768, 80 % sparse
        _attention('attention_step_f32', 1, 4096, 3072, 768, 32, 0, 0.20, False, 'f32', kind='attention_step'),
        # a batch of sequences of every length up to 1024
        dict(name='seqlen_f16', kind='seqlen', batch=32, heads=12, N=1024, E=64, dtype='f16'),
        # top-1 routed experts, Zipf(1.2) skew
        dict(name='moe_zipf', kind='moe', tokens=16384, K=1024, N=4096, experts=8, dtype='f16'),
    ]


def _linear(name, M, K, N, bn, bk, sparsity, dtype, bias=False, relu=False, kind='linear'):
    case = dict(kind=kind, M=M, K=K, N=N, bn=bn, bk=bk, sparsity=sparsity, dtype=dtype, bias=bias, relu=relu)
    return case if name is None else dict(case, name=name)


def _attention(name, heads, Nt, Ns, E, block, window, extra, causal, dtype, kind='attention'):
    """`window`: blocks of the causal band (0: none); `extra`: share of all blocks added at random;
    `causal`: the blocks on the diagonal are cut to their lower triangle, element by element."""
    case = dict(kind=kind, heads=heads, Nt=Nt, Ns=Ns, E=E, block=block, window=window, extra=extra,
                causal=causal, dtype=dtype)
    return case if name is None else dict(case, name=name)


_MAX_FLOPS = 1.38e11   # the largest listed cases: attention_step_f16 and moe_zipf
_MAX_BYTES = 5.0e8


def _log_int(rng, low, high, step=1):
    """A multiple of `step` between low and high, spread evenly over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))) / step)) * step))


def draw(rng):
    kinds = ['linear', 'linear', 'linear_step', 'linear_step', 'ffn', 'attention', 'attention_step', 'seqlen', 'moe']
    while True:
        case = _draw_kind(rng, rng.choice(kinds))
        w = work(case)
        if w['flops'] <= _MAX_FLOPS and w['bytes'] <= _MAX_BYTES:
            return case


def _draw_kind(rng, kind):
    half = rng.choice(['f16', 'bf16'])
    if kind in ('linear', 'linear_step'):
        dtype = rng.choice([half, half, 'f32'])
        bn, bk = rng.choice([(32, 32), (32, 64), (64, 64), (16, 16)] if dtype == 'f32' else [(32, 32), (32, 64), (64, 64)])
        # a training batch is a multiple of 16 tokens (the weight gradient sums over them in tiles)
        M = _log_int(rng, 1, 16384) if kind == 'linear' else _log_int(rng, 64, 8192, 16)
        K, N = (_log_int(rng, 512, 4096, 64) for _ in range(2))
        return _linear(None, M, K, N, bn, bk, round(rng.uniform(0.6, 0.98), 3), dtype,
                       bias=rng.random() < 0.6, relu=kind == 'linear' and rng.random() < 0.3, kind=kind)
    if kind == 'ffn':
        K = _log_int(rng, 512, 1024, 64)
        return dict(kind=kind, M=_log_int(rng, 128, 8192), K=K, N=rng.choice([2, 3, 4]) * K, bn=32,
                    bk=rng.choice([32, 64]), sparsity=round(rng.uniform(0.75, 0.95), 3), dtype=half)
    if kind in ('attention', 'attention_step'):
        dtype = rng.choice([half, half, half, 'f32'])
        block = rng.choice([32, 64])
        if dtype == 'f32':   # the three-operator pipeline: few heads
            heads, Nt, E = rng.randint(1, 4), _log_int(rng, 512, 4096, 64), rng.choice([64, 128, 256, 768])
            Ns = _log_int(rng, 512, 4096, 64)
            return _attention(None, heads, Nt, Ns, E, block, 0, round(rng.uniform(0.05, 0.25), 3), False, dtype, kind)
        heads, N, E = 12 * rng.choice([1, 1, 2, 4, 8]), _log_int(rng, 256, 4096, 64), rng.choice([64, 64, 128])
        return _attention(None, heads, N, N, E, block, rng.randint(2, 6), rng.choice([0.0, 0.02, 0.05]),
                          rng.random() < 0.5, dtype, kind)
    if kind == 'seqlen':
        return dict(kind=kind, batch=_log_int(rng, 1, 32), heads=rng.choice([8, 12, 16]), N=_log_int(rng, 128, 2048, 32),
                    E=rng.choice([64, 64, 128]), dtype=half)
    return dict(kind='moe', tokens=_log_int(rng, 32, 16384), K=rng.choice([768, 1024, 2048]),
                N=rng.choice([768, 2048, 3072, 4096]), experts=rng.choice([4, 8, 16, 32]), dtype=half)


# ---- masks --------------------------------------------------------------------------------------
def _live_count(blocks, share):
    return max(1, int(round(blocks * share)))


def _random_grid(rows, cols, live, gen, device, among=None):
    """uint8 [rows, cols] with exactly `live` ones at random places (of `among`, if given)."""
    score = torch.rand(rows * cols, generator=gen, device=device)
    if among is not None:
        score = torch.where(among.flatten(), score, torch.full_like(score, -1.0))
    grid = torch.zeros(rows * cols, dtype=torch.uint8, device=device)
    grid[score.topk(live).indices] = 1
    return grid.view(rows, cols)


def _expand(grid, bh, bw):
    return grid.repeat_interleave(bh, 0).repeat_interleave(bw, 1).contiguous()


def _weight_mask(N, K, bn, bk, sparsity, gen, device):
    live = _live_count((N // bn) * (K // bk), 1 - sparsity)
    return _expand(_random_grid(N // bn, K // bk, live, gen, device), bn, bk)


def _attention_blocks(case):
    """(blocks of the causal band, random extra blocks)."""
    rows, cols = case['Nt'] // case['block'], case['Ns'] // case['block']
    band = sum(min(i + 1, case['window']) for i in range(rows)) if case['window'] else 0
    extra = int(round(case['extra'] * rows * cols))
    free = rows * cols - band
    if case['causal']:
        free = rows * (rows + 1) // 2 - band   # random blocks lie in the past as well
    return band, min(extra, free)


def _attention_mask(case, gen, device):
    rows, cols, blk = case['Nt'] // case['block'], case['Ns'] // case['block'], case['block']
    i = torch.arange(rows, device=device)[:, None]
    j = torch.arange(cols, device=device)[None, :]
    band = ((i - j >= 0) & (i - j < case['window'])) if case['window'] else torch.zeros((rows, cols), dtype=torch.bool, device=device)
    extra = _attention_blocks(case)[1]
    grid = band.to(torch.uint8)
    if extra:
        free = ~band & (j <= i) if case['causal'] else ~band
        grid = grid | _random_grid(rows, cols, extra, gen, device, among=free)
    mask = _expand(grid, blk, blk)
    return torch.tril(mask).contiguous() if case['causal'] else mask


# ---- operators ------------------------------------------------------------------------------------
def _mm(m, k, n):
    return {'_impl': 'sparta', 'BLOCK_SIZE_M_VALUE': m, 'BLOCK_SIZE_K_VALUE': k, 'BLOCK_SIZE_N_VALUE': n}


def _linear_config(bn, bk, backward):
    config = {'forward:C': _mm(32, bk, bn)}
    if backward:
        config['backward:A'] = _mm(32, bn, bk)
        config['backward:B'] = _mm(bn, 32, bk)
    return config


def _attention_config(blk):
    sm = {'_impl': 'sparta', 'BLOCK_SIZE_H_VALUE': blk, 'BLOCK_SIZE_W_VALUE': blk, 'ROW_TILE_VALUE': 4}
    return {'qk/forward:C': _mm(blk, 32, blk), 'qk/backward:A': _mm(blk, blk, 32), 'qk/backward:B': _mm(blk, blk, 32),
            'sm/forward:y': dict(sm), 'sm/backward:x': dict(sm),
            'out/forward:C': _mm(blk, blk, 32), 'out/backward:A': _mm(blk, 32, blk), 'out/backward:B': _mm(blk, blk, 32)}


def _dense_linear(K, N, bias, dtype, gen, device):
    lin = torch.nn.Linear(K, N, bias=bias, device=device, dtype=dtype)
    with torch.no_grad():
        lin.weight.copy_(torch.randn((N, K), generator=gen, device=device) / math.sqrt(K))
        if bias:
            lin.bias.copy_(0.1 * torch.randn((N,), generator=gen, device=device))
    return lin


def _randn(shape, dtype, gen, device):
    return torch.randn(shape, generator=gen, device=device).to(dtype)


def prepare(case, seed):
    device = torch.device('cuda:0')
    gen = torch.Generator(device=device).manual_seed(int(seed) % (1 << 31))
    return _PREPARE[case['kind']](case, gen, device)


def _prepare_linear(case, gen, device):
    M, K, N, bn, bk = (case[k] for k in ('M', 'K', 'N', 'bn', 'bk'))
    dtype, step = _DTYPES[case['dtype']], case['kind'] == 'linear_step'
    mask = _weight_mask(N, K, bn, bk, case['sparsity'], gen, device)
    lin = _dense_linear(K, N, case['bias'], dtype, gen, device)
    x = _randn((M, K), dtype, gen, device)
    op = sparta.nn.SparseLinear(lin, weight_mask=mask, activation='relu' if case['relu'] else None)
    op.build(_linear_config(bn, bk, step), sample_inputs=[x])
    if not step:
        return dict(run=_run_forward, op=op, inputs=[x])
    return dict(run=_run_step, op=op, inputs=[x.requires_grad_(True)], grad=_randn((M, N), dtype, gen, device),
                leaves=[x] + list(op.parameters()))


def _prepare_ffn(case, gen, device):
    M, K, N, bn, bk = (case[k] for k in ('M', 'K', 'N', 'bn', 'bk'))
    dtype = _DTYPES[case['dtype']]
    masks = [[_weight_mask(n, k, bn, bk, case['sparsity'], gen, device) for _ in range(2)] for n, k in ((N, K), (K, N))]
    x = _randn((M, K), dtype, gen, device)
    up = sparta.nn.SparseLinear(_dense_linear(K, N, False, dtype, gen, device), weight_mask=masks[0][0], dynamic=True, activation='relu')
    down = sparta.nn.SparseLinear(_dense_linear(N, K, False, dtype, gen, device), weight_mask=masks[1][0], dynamic=True)
    up.build(_linear_config(bn, bk, False), sample_inputs=[x])
    with torch.no_grad():
        down.build(_linear_config(bn, bk, False), sample_inputs=[up(x)])
    return dict(run=_run_ffn, up=up, down=down, up_mask=masks[0][1], down_mask=masks[1][1], x=x)


def _prepare_attention(case, gen, device):
    heads, Nt, Ns, E = (case[k] for k in ('heads', 'Nt', 'Ns', 'E'))
    dtype = _DTYPES[case['dtype']]
    mask = _attention_mask(case, gen, device)
    q, k, v = (_randn((heads, n, E), dtype, gen, device) for n in (Nt, Ns, Ns))
    op = sparta.nn.SparseAttention(mask=mask)
    config = _attention_config(case['block'])
    step = case['kind'] == 'attention_step'
    if not step:
        config = {name: cfg for name, cfg in config.items() if '/forward' in name}
    op.build(config, sample_inputs=[q, k, v])
    if not step:
        return dict(run=_run_forward, op=op, inputs=[q, k, v])
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    return dict(run=_run_step, op=op, inputs=leaves, grad=_randn((heads, Nt, E), dtype, gen, device), leaves=leaves)


def _lengths(case):
    """Lengths spread evenly over 1 .. N."""
    B = case['batch']
    return [max(1, int((i + 0.5) / B * case['N'])) for i in range(B)]


def _prepare_seqlen(case, gen, device):
    B, H, N, E = (case[k] for k in ('batch', 'heads', 'N', 'E'))
    dtype = _DTYPES[case['dtype']]
    lens = torch.tensor(_lengths(case), dtype=torch.int32, device=device)[torch.randperm(B, generator=gen, device=device)]
    # the operator applies no temperature: the query comes scaled
    q = (torch.randn((B, H, N, E), generator=gen, device=device) / math.sqrt(E)).to(dtype)
    k, v = (_randn((B, H, N, E), dtype, gen, device) for _ in range(2))
    return dict(run=_run_forward, op=sparta.nn.SeqlenDynamicSparseAttention(global_mode=False), inputs=[q, k, v, lens])


def _prepare_moe(case, gen, device):
    T, K, N, E = (case[k] for k in ('tokens', 'K', 'N', 'experts'))
    dtype = _DTYPES[case['dtype']]
    op = sparta.nn.DynamicSparseMoE([_dense_linear(K, N, False, dtype, gen, device) for _ in range(E)])
    share = torch.from_numpy(np.arange(1, E + 1, dtype=np.float64) ** -1.2).to(device)
    ids = torch.multinomial(share, T, replacement=True, generator=gen).to(torch.int32)
    return dict(run=_run_forward, op=op, inputs=[_randn((T, K), dtype, gen, device), ids])


_PREPARE = {'linear': _prepare_linear, 'linear_step': _prepare_linear, 'ffn': _prepare_ffn, 'attention': _prepare_attention,
            'attention_step': _prepare_attention, 'seqlen': _prepare_seqlen, 'moe': _prepare_moe}


# ---- one pass ---------------------------------------------------------------------------------------
def run(state):
    return state['run'](state)


def _run_forward(state):
    with torch.no_grad():
        return state['op'](*state['inputs'])


def _run_step(state):
    for t in state['leaves']:
        t.grad = None
    out = state['op'](*state['inputs'])
    out.backward(state['grad'])
    return [out.detach()] + [t.grad for t in state['leaves']]


def _run_ffn(state):
    up, down = state['up'], state['down']
    with torch.no_grad():
        sparta.nn.update_masks([(up, {'weight_mask': state['up_mask']}), (down, {'weight_mask': state['down_mask']})])
        return down(up(state['x']))


# ---- what a pass cannot do without ----------------------------------------------------------------------
def work(case):
    kind, es = case['kind'], _BYTES[case['dtype']]
    if kind in ('linear', 'linear_step', 'ffn'):
        M, K, N, bn, bk = (case[k] for k in ('M', 'K', 'N', 'bn', 'bk'))
        live = _live_count((N // bn) * (K // bk), 1 - case['sparsity']) * bn * bk
        if kind == 'ffn':   # two layers; the hidden tensor leaves the chip once, both masks are read
            return {'bytes': es * (2 * M * K + 2 * M * N + 2 * live) + 2 * N * K, 'flops': 4.0 * M * live}
        if kind == 'linear':
            return {'bytes': es * (M * K + M * N + live + (N if case['bias'] else 0)), 'flops': 2.0 * M * live}
        return {'bytes': es * (2 * M * K + 2 * M * N + 2 * live + (2 * N if case['bias'] else 0)), 'flops': 6.0 * M * live}
    if kind in ('attention', 'attention_step'):
        heads, Nt, Ns, E = (case[k] for k in ('heads', 'Nt', 'Ns', 'E'))
        entries = heads * sum(_attention_blocks(case)) * case['block'] ** 2
        io = es * heads * E * (2 * Nt + 2 * Ns)   # query, key, value, output
        if kind == 'attention':
            return {'bytes': io, 'flops': 4.0 * entries * E}
        return {'bytes': 2 * io, 'flops': 12.0 * entries * E}   # every tensor and its gradient; six products
    if kind == 'seqlen':
        H, E, lens = case['heads'], case['E'], _lengths(case)
        return {'bytes': es * H * E * (3 * sum(lens) + case['batch'] * case['N']), 'flops': 4.0 * H * E * sum(n * n for n in lens)}
    T, K, N, E = (case[k] for k in ('tokens', 'K', 'N', 'experts'))
    return {'bytes': es * (T * K + T * N + min(E, T) * K * N) + 4 * T, 'flops': 2.0 * T * K * N}


def tolerance(case):
    # fp32: sums of fp32 products in another order (the training step of attention subtracts
    # nearly equal ones); 16-bit types: results, and the probabilities and hidden values on the
    # way to them, are rounded to 11 or 8 significant bits
    if case['dtype'] == 'f32':
        return {'rel': 2e-5 if case['kind'] == 'attention_step' else 1e-5}
    return {'rel': 2e-3 if case['dtype'] == 'f16' else 1e-2}
