"""The work that users of this package have it do, as cases that can be timed: the attention modules and the chain behind
them, the separate sdd / softmax / dsd operators, block-sparse linear layers and plain block-sparse products, from calls of
a few microseconds of GPU work to the largest shapes of the benchmark, in training (forward and backward) and in inference.

listed() gives the named cases, draw(rng) one more of the same ranges; prepare() makes the inputs and operator objects that a
program holds before the call, run() is one pass through the public entry points, work() what the pass cannot do without,
tolerance() how far another correct implementation at the same precision may differ."""
import math
import os
import sys

import torch

_PKG = os.path.abspath('torch-blocksparse_amd')
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import torch_blocksparse as tb                                            # noqa: E402
from torch_blocksparse.attention_core import attention_chain               # noqa: E402

_DTYPES = {'fp16': torch.float16, 'bf16': torch.bfloat16, 'fp32': torch.float32}
_SIZE = {'fp16': 2, 'bf16': 2, 'fp32': 4}


def _attention(api, layout, block, Z, H, L, d, dtype, train, kpm=False, pair_masks=False, **options):
    return dict(family='attention', api=api, layout=layout, block=block, Z=Z, H=H, L=L, d=d, dtype=dtype, train=train,
                kpm=kpm, pair_masks=pair_masks, **options)


def listed():
    cases = []

    def case(name, **c):
        cases.append(dict(c, name=name))

    # The README's first example: a transposed fp32 sdd in blocks of 16 followed by the softmax; a few launches of a few
    # microseconds each, so the calls themselves count.
    case('readme_sdd_softmax_fp32', family='readme', Z=4, H=2, M=256, N=512, K=384, block=16, density=0.5, dtype='fp32')
    # One short sequence through the self-attention module in its default configuration, as a server answers a request.
    case('module_infer_512', **_attention('module', 'fixed', 16, 1, 8, 512, 64, 'fp16', False, stride=64, bidirectional=False))
    # A pruned feed-forward layer at inference, with a number of tokens that divides by nothing.
    case('linear32_infer_999', family='linear', tokens=999, fin=1024, fout=4096, block=32, density=0.25, dtype='bf16', train=False)
    # Training in single precision, the type that modules are created in: bidirectional layout, padded sequences.
    case('module_train_fp32', **_attention('module', 'fixed', 32, 2, 8, 2048, 64, 'fp32', True, kpm=True, stride=128, bidirectional=True))
    # The self-attention module in its default configuration (block 16, stride 64) at the headline's size.
    case('module_train_default', **_attention('module', 'fixed', 16, 8, 16, 4096, 64, 'fp16', True, stride=64, bidirectional=False))
    # Dense attention through the module (SparsityConfig(mode='dense')) with the wide head: every block of every row, bf16.
    case('module_train_dense_d128', **_attention('module', 'dense', 64, 4, 8, 2048, 128, 'bf16', True))
    # The headline workload, fixed Sparse-Transformer layout with padded keys, as the modules run it ...
    case('chain_train_headline', **_attention('chain', 'transformer', 64, 8, 16, 4096, 64, 'fp16', True, kpm=True))
    # ... and as a program that calls the three operators itself runs it.
    case('ops_train_headline', **_attention('ops', 'transformer', 64, 8, 16, 4096, 64, 'fp16', True, kpm=True))
    # Long context: BigBird-style layout at 16384 positions with a relative position embedding and a causal mask.
    case('chain_train_bigbird', **_attention('chain', 'bigbird', 64, 2, 12, 16384, 64, 'fp16', True, pair_masks=True))
    # Block-sparse linear layer in training: 8192 tokens, 4096 x 4096, a tenth of the blocks of 128; y, dx and dw.
    case('linear128_train_8192', family='linear', tokens=8192, fin=4096, fout=4096, block=128, density=0.1, dtype='fp16', train=True)
    # The reference's matmul benchmark: sdd in blocks of 16 over a hidden size of 512, every head of a 'fixed' layout.
    case('sdd16_hidden512', family='matmul', mode='sdd', Z=1, H=12, M=4096, N=4096, K=512, block=16, density=0., trans_a=False,
         trans_b=False, dtype='fp16', train=False)
    # Large products in blocks of 32 with a quarter of the blocks, forward and both gradients.
    case('dsd32_train_2048', family='matmul', mode='dsd', Z=8, H=16, M=2048, N=2048, K=2048, block=32, density=0.25, trans_a=False,
         trans_b=False, dtype='fp16', train=True)
    return cases


def _spread(rng, lo, hi):
    """a whole number between lo and hi, spread over its logarithm"""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_attention(rng):
    api = rng.choice(('module', 'module', 'chain', 'chain', 'ops'))
    block = rng.choice((16, 32, 64))
    c = _attention(api, 'fixed', block, rng.randint(1, 8), rng.choice((2, 3, 5, 8, 12, 16)), 0, rng.choice((64, 64, 64, 128, 32)),
                   rng.choice(('fp16', 'fp16', 'bf16', 'fp32')), rng.random() < 0.7, kpm=rng.random() < 0.4)
    if api == 'module':
        if rng.random() < 0.2:
            c.update(layout='dense', L=64 * _spread(rng, 2, 32))
        else:
            stride = block * rng.choice((2, 4, 8))
            c.update(stride=stride, bidirectional=rng.random() < 0.4, L=stride * max(1, _spread(rng, 128, 4096) // stride))
    elif rng.random() < 0.5:
        c.update(layout='transformer', L=4 * block * max(1, _spread(rng, 256, 8192) // (4 * block)))
        c['kpm'] = c['kpm'] and c['L'] >= 24 * block                      # (shorter ones would hold rows without any unmasked key)
    else:
        c.update(layout='bigbird', L=64 * _spread(rng, 8, 128), pair_masks=rng.random() < 0.4)
    return c


def _draw_linear(rng):
    block = rng.choice((32, 64, 128))
    return dict(family='linear', tokens=_spread(rng, 16, 8192), fin=block * _spread(rng, 4, 4096 // block), fout=block * _spread(rng, 4, 4096 // block),
                block=block, density=rng.choice((0.1, 0.25, 0.5)), dtype=rng.choice(('fp16', 'bf16', 'fp32')), train=rng.random() < 0.5)


def _draw_matmul(rng):
    block = rng.choice((16, 32, 64, 128))
    mode = rng.choice(('sdd', 'dsd', 'dds'))
    m, n, k = [block * _spread(rng, 2, 2048 // block) for _ in range(3)]
    return dict(family='matmul', mode=mode, Z=rng.randint(1, 4), H=rng.choice((1, 2, 3, 8)), M=m, N=n, K=k, block=block,
                density=rng.choice((0.1, 0.25, 0.5)), trans_a=rng.random() < 0.5, trans_b=rng.random() < 0.5,
                dtype=rng.choice(('fp16', 'bf16', 'fp32')), train=rng.random() < 0.5)


def _draw_readme(rng):
    block = rng.choice((16, 32, 64))
    m, n = [block * _spread(rng, 2, 1024 // block) for _ in range(2)]
    return dict(family='readme', Z=rng.randint(1, 4), H=rng.randint(1, 4), M=m, N=n, K=16 * _spread(rng, 4, 32), block=block,
                density=0.5, dtype=rng.choice(('fp16', 'fp32', 'fp32')))


def draw(rng):
    """One more case of the same ranges: more often attention, which most users come for.  Shapes whose work would exceed a
    quarter of the largest listed case's are drawn again (a product in fp32 counts for what it costs on its matrix pipe)."""
    while True:
        c = rng.choice((_draw_attention, _draw_attention, _draw_linear, _draw_matmul, _draw_readme))(rng)
        w = work(c)
        if w['flops'] * (16 if c['dtype'] == 'fp32' else 1) < 4e11 and w['bytes'] < 2.5e9:
            return c


def _random_layout(H, R, C, density, seed):
    """Bernoulli blocks, every row and every column of blocks holding at least one"""
    g = torch.Generator().manual_seed(seed)
    lay = (torch.rand((H, R, C), generator=g) < density).long()
    r, c = torch.arange(R), torch.arange(C)
    lay[:, r, r % C] |= (lay.sum(2) == 0).long()
    lay[:, c % R, c] |= (lay.sum(1) == 0).long()
    return lay


def _layout(c):
    """the block layout of a case: part of the program, the same for every seed of its inputs"""
    block = c['block']
    if c['family'] == 'attention':
        H, nb = c['H'], c['L'] // block
        if c['layout'] == 'dense':
            return torch.ones((H, nb, nb), dtype=torch.int64)
        if c['layout'] == 'fixed':
            return tb.fixed_layout(H, nb, 'fixed', c['stride'] // block, 'bidirectional' if c['bidirectional'] else 'unidirectional', 1, 1)
        if c['layout'] == 'transformer':
            return tb.sparse_transformer_layout(H, nb, 4, 16, True)
        return tb.bigbird_layout(H, nb, 3, 2, 3, seed=0, causal=True)
    if c['family'] == 'linear':
        return _random_layout(1, c['fin'] // block, c['fout'] // block, c['density'], 1)
    if c['family'] == 'readme':
        return _random_layout(c['H'], c['M'] // block, c['N'] // block, c['density'], 2)
    rows, cols = {'sdd': ('M', 'N'), 'dsd': ('M', 'K'), 'dds': ('K', 'N')}[c['mode']]
    if (c['mode'] == 'dsd' and c['trans_a']) or (c['mode'] == 'dds' and c['trans_b']):
        rows, cols = cols, rows                                           # the layout describes the sparse operand as stored
    if c['density'] == 0.:
        return tb.make_layout(c['H'], c[rows] // block, 'fixed', 4, False, 1, 1)
    return _random_layout(c['H'], c[rows] // block, c[cols] // block, c['density'], 3)


def prepare(c, seed):
    dtype, dev, block = _DTYPES[c['dtype']], 'cuda', c['block']
    g = torch.Generator(device=dev).manual_seed(seed)
    lay = _layout(c)
    s = dict(case=c)

    def normal(*shape, std=1., grad=False):
        t = torch.randn(shape, generator=g, device=dev, dtype=dtype)
        t = t.mul_(std) if std != 1. else t
        return t.requires_grad_(grad)

    if c['family'] == 'readme':
        Z, H, M, N, K = c['Z'], c['H'], c['M'], c['N'], c['K']
        s['a'] = torch.rand((Z, H, K, M), generator=g, device=dev, dtype=dtype)
        s['b'] = torch.rand((Z, H, K, N), generator=g, device=dev, dtype=dtype)
        s['dot'] = tb.MatMul(lay, block, 'sdd', trans_a=True, trans_b=False)
        s['softmax'] = tb.Softmax(lay, block)
        return s

    if c['family'] == 'linear':
        lin = tb.Linear(c['fin'], c['fout'], block, lay).to(device=dev, dtype=dtype)
        with torch.no_grad():
            lin.weight.copy_(normal(*lin.weight.shape, std=0.02))
        s['linear'] = lin
        s['x'] = normal(c['tokens'], c['fin'], grad=c['train'])
        s['dy'] = normal(c['tokens'], c['fout']) if c['train'] else None
        return s

    if c['family'] == 'matmul':
        Z, H, M, N, K, mode = [c[n] for n in ('Z', 'H', 'M', 'N', 'K', 'mode')]
        nnz, std = int(lay.sum()), K ** -0.5
        a = (Z, H, K, M) if c['trans_a'] else (Z, H, M, K)
        b = (Z, H, N, K) if c['trans_b'] else (Z, H, K, N)
        a, b, y = [(Z, nnz, block, block) if sparse == 's' else t for sparse, t in zip(mode[1:] + mode[0], (a, b, (Z, H, M, N)))]
        s['a'], s['b'] = normal(*a, std=std, grad=c['train']), normal(*b, std=std, grad=c['train'])
        s['dy'] = normal(*y) if c['train'] else None
        s['dot'] = tb.MatMul(lay, block, mode, trans_a=c['trans_a'], trans_b=c['trans_b'])
        return s

    Z, H, L, d = c['Z'], c['H'], c['L'], c['d']
    s['q'], s['k'], s['v'] = [normal(Z, H, L, d, grad=c['train']) for _ in range(3)]
    s['do'] = normal(Z, H, L, d) if c['train'] else None
    masks = {}
    if c['kpm']:                                                          # the last 0 - 25 % of the keys of a sequence are padding
        kept = (L * (1 - 0.25 * torch.rand((Z,), generator=g, device=dev))).long()
        kpm = torch.zeros((Z, L), device=dev, dtype=dtype)
        masks['key_padding_mask'] = kpm.masked_fill_(torch.arange(L, device=dev)[None] >= kept[:, None], float('-inf'))
    if c['pair_masks']:
        masks['rpe'] = normal(L, L, std=0.1)
        masks['attn_mask'] = torch.tril(torch.ones((L, L), device=dev, dtype=dtype))
    if c['api'] == 'module':
        config = (tb.SparsityConfig(mode='dense', block=block) if c['layout'] == 'dense' else
                  tb.SparsityConfig(mode='fixed', block=block, stride=c['stride'], attention='bidirectional' if c['bidirectional'] else 'unidirectional'))
        s['module'] = tb.SparseSelfAttention(config)
    else:
        s['sdd'] = tb.MatMul(lay, block, 'sdd', trans_a=False, trans_b=True)
        s['softmax'] = tb.Softmax(lay, block)
        s['dsd'] = tb.MatMul(lay, block, 'dsd')
        masks['scale'] = float(d) ** -0.5
        if c['pair_masks']:
            masks['attn_mask_mode'] = 'mul'
    s['masks'] = masks
    return s


def _forward(s):
    c = s['case']
    if c['family'] == 'readme':
        return s['softmax'](s['dot'](s['a'], s['b']), scale=float(c['K']) ** -0.5)
    if c['family'] == 'linear':
        return s['linear'](s['x'])
    if c['family'] == 'matmul':
        return s['dot'](s['a'], s['b'])
    q, k, v = s['q'], s['k'], s['v']
    if c['api'] == 'module':
        return s['module'](q, k, v, **s['masks'])
    if c['api'] == 'chain':
        return attention_chain(s['sdd'], s['softmax'], s['dsd'], q, k, v, **s['masks'])
    return s['dsd'](s['softmax'](s['sdd'](q, k), **s['masks']), v)


def run(s):
    c = s['case']
    if not c.get('train', False):
        with torch.no_grad():
            return _forward(s)
    y = _forward(s)
    if c['family'] == 'linear':
        inputs, dy = (s['x'], s['linear'].weight), s['dy']
    elif c['family'] == 'matmul':
        inputs, dy = (s['a'], s['b']), s['dy']
    else:
        inputs, dy = (s['q'], s['k'], s['v']), s['do']
    return (y.detach(),) + torch.autograd.grad(y, inputs, dy)


def work(c):
    """Bytes and operations of one pass.  Products count 2 operations per nonzero element and element of the free dimension;
    every input of an entry point is read once and every output written once.  The three operators are entry points of
    their own, so there the sparse tensor between them counts: in training it is written or read eleven times."""
    size, block = _SIZE[c['dtype']], c['block']
    lay = _layout(c)
    elems = float(int(lay.sum()) * block * block)
    if c['family'] == 'readme':
        Z, H, M, N, K = c['Z'], c['H'], c['M'], c['N'], c['K']
        return {'bytes': size * Z * (H * K * (M + N) + 3 * elems), 'flops': 2. * Z * K * elems}
    if c['family'] == 'linear':
        io = float(c['tokens']) * (c['fin'] + c['fout'])
        return {'bytes': size * ((2 * io + 2 * elems) if c['train'] else (io + elems)),
                'flops': (6. if c['train'] else 2.) * c['tokens'] * elems}
    if c['family'] == 'matmul':
        Z, H = c['Z'], c['H']
        free = {'sdd': c['K'], 'dsd': c['N'], 'dds': c['M']}[c['mode']]
        dense = {'sdd': c['K'] * (c['M'] + c['N']), 'dsd': c['N'] * (c['M'] + c['K']), 'dds': c['M'] * (c['K'] + c['N'])}[c['mode']]
        once = Z * (float(H) * dense + elems)
        return {'bytes': size * (2 if c['train'] else 1) * once, 'flops': (6. if c['train'] else 2.) * Z * free * elems}
    Z, H, L, d = c['Z'], c['H'], c['L'], c['d']
    dense = float(Z) * H * L * d
    masks = (Z * L if c['kpm'] else 0) + (2. * int((lay.sum(0) > 0).sum()) * block * block if c['pair_masks'] else 0)
    if c['api'] == 'ops':
        total = (12 * dense + 11 * Z * elems) if c['train'] else (4 * dense + 4 * Z * elems)
    else:
        total = (8 if c['train'] else 4) * dense
    return {'bytes': size * (total + masks), 'flops': (12. if c['train'] else 4.) * Z * d * elems}


def tolerance(c):
    """About four times the relative error measured against the same chain of dense operations in 64 bits: fp32 up to 1.5e-6
    (the README's softmax over products of positive terms); single products in fp16 2.1e-4 and in bf16 1.7e-3, which is the
    rounding of the result; attention in fp16 up to 6.4e-4 and in bf16 5.0e-3, where the scores and the softmax are rounded
    between the products as well; an fp16 softmax of rounded products 9e-4."""
    if c['dtype'] == 'fp32':
        return {'rel': 6e-6}
    if c['family'] == 'attention':
        return {'rel': 2.5e-3 if c['dtype'] == 'fp16' else 2e-2}
    if c['family'] == 'readme':
        return {'rel': 3.6e-3}
    return {'rel': 8e-4 if c['dtype'] == 'fp16' else 6.6e-3}
