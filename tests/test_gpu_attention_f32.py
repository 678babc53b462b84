"""GPU: the attention chain in fp32 on the bfloat16 matrix units (bsp_attention_f32_fwd / _bwd behind attention_chain) against dense 64-bit
arithmetic and against the three operators, which compute on the fp32 units.

Tolerance: a product keeps what counts in 24 bits and is rounded less often than on the fp32 units, and the softmax is formed as the
operator forms it.  So over a tensor the error to 64 bits is no more than the operators', give or take a unit of 2^-23 (relative 2-norm); single rows
may be further off than theirs as they may be closer, which is where a factor stands beside the bound."""
import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import attention_core as ac

pytestmark = pytest.mark.gpu
DEV = 'cuda'


@pytest.fixture(autouse=True)
def _kernels_for_every_layout(request, monkeypatch):
    if 'layouts_of_both_routes' not in request.node.name:
        monkeypatch.setattr(ac._QuadTables, 'pays_f32', lambda *args: True)


def _ops(lay, block):
    return tb.MatMul(lay, block, 'sdd', trans_b=True), tb.Softmax(lay, block), tb.MatMul(lay, block, 'dsd')


def _run(ops, q, k, v, do, fused, **kw):
    xs = [t.detach().clone().requires_grad_() for t in (q, k, v)]
    before, was = ac.fused_f32_calls, ac.FUSED
    ac.FUSED = fused
    try:
        o = ac.attention_chain(*ops, *xs, **kw)
        grads = torch.autograd.grad(o, xs, do)
    finally:
        ac.FUSED = was
    assert ac.fused_f32_calls - before == int(fused)
    return (o.detach(),) + grads


def _dense(q, k, v, do, lay, block, scale, kpm=None):
    xs = [t.detach().double().requires_grad_() for t in (q, k, v)]
    m = lay.to(DEV).repeat_interleave(block, 1).repeat_interleave(block, 2).bool()
    s = xs[0] @ xs[1].transpose(-1, -2) * scale
    if kpm is not None:
        s = s + kpm.double()[:, None, None, :]
    s = s.masked_fill(~m, float('-inf'))
    p = torch.where(m.any(-1, keepdim=True), torch.softmax(s, -1), torch.zeros((), dtype=torch.float64, device=DEV))
    o = p @ xs[2]
    return (o.detach(),) + torch.autograd.grad(o, xs, do.double())


def _layout(H, R, C, kind):
    g = torch.Generator().manual_seed(R * 131 + C)
    if kind == 'dense':
        return torch.ones(H, R, C, dtype=torch.int64)
    lay = (torch.rand((H, R, C), generator=g) < 0.3).long()
    lay[:, :, 0] = 1                                                      # a long column (in parts where it is long enough), no row without keys
    if kind == 'holes':                                                   # rows without any block beside one that has some
        lay[:, 4:8] = 0
        lay[:, 5, min(3, C - 1)] = 1
    return lay


# one tile; a tile of remainders; lines and columns of one to many tiles; parts of long columns (6 and 128 of them, in halves; 192,
# whole); from 32 heads on another order of the workgroups
@pytest.mark.parametrize('Z,H,R,C,block,D,kind,padded', [
    (1, 1, 1, 1, 64, 64, 'dense', False),
    (2, 1, 4, 4, 16, 128, 'random', True),
    (1, 2, 2, 10, 32, 64, 'random', True),
    (2, 2, 16, 24, 32, 64, 'holes', True),
    (1, 2, 12, 8, 16, 64, 'holes', False),
    (1, 3, 40, 6, 64, 64, 'random', False),
    (11, 6, 80, 8, 32, 64, 'random', False),
    (2, 32, 40, 4, 64, 128, 'random', True),
    (64, 8, 40, 2, 64, 64, 'random', False),
    (3, 32, 40, 4, 64, 64, 'random', False),
    (1, 2, 32, 32, 64, 128, 'dense', False),
])
def test_against_64_bits(Z, H, R, C, block, D, kind, padded):
    torch.manual_seed(R + C + D)
    lay = _layout(H, R, C, kind)
    q, do = [torch.randn(Z, H, R * block, D, device=DEV) for _ in range(2)]
    k, v = [torch.randn(Z, H, C * block, D, device=DEV) for _ in range(2)]
    kw = dict(scale=D ** -0.5)
    if padded:
        kpm = torch.zeros(Z, C * block, device=DEV)
        kpm[0, block:block + 9] = float('-inf')
        kpm[-1, block + 5:] = -2.
        kw['key_padding_mask'] = kpm
    ref = _dense(q, k, v, do, lay, block, D ** -0.5, kw.get('key_padding_mask'))
    ops = _ops(lay, block)
    got, other = [_run(ops, q, k, v, do, fused, **kw) for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        assert bool(torch.isfinite(g).all()), name
        err, bound = [float((x.double() - r).norm() / r.norm()) for x in (g, c)]
        assert err <= bound + 2 ** -23, (name, err, bound)
    again = _run(ops, q, k, v, do, True, **kw)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


# Values that have no bfloat16 parts, or whose products fp32 does not hold, in one row of one head: what is and what is not finite comes out
# as it does on the fp32 units, also for rows whose tiles hold the value in a block that they do not have.
@pytest.mark.parametrize('where,value', [('q', float('inf')), ('k', float('-inf')), ('v', float('inf')), ('v', float('nan')), ('do', float('-inf')), ('k', 1e20), ('k', 3.4e38), ('q', 1e10)])
@pytest.mark.parametrize('block,D', [(32, 64), (16, 128)])
def test_values_without_parts(where, value, block, D):
    torch.manual_seed(block)
    n = 256 // block
    lay = _layout(2, n, n, 'random')
    x = {t: torch.randn(2, 2, 256, D, device=DEV) for t in ('q', 'k', 'v', 'do')}
    x[where][0, 1, 37, 5] = value
    ops = _ops(lay, block)
    got, other = [_run(ops, x['q'], x['k'], x['v'], x['do'], fused, scale=D ** -0.5) for fused in (True, False)]
    for name, g, c in zip(('o', 'dq', 'dk', 'dv'), got, other):
        assert bool((torch.isfinite(g) == torch.isfinite(c)).all()), name
        assert bool((torch.isnan(g) == torch.isnan(c)).all()), name
    # the other batch and head are as if nothing had been there (a few 2^-24 of two correct results)
    for g, c in zip(got, other):
        assert float((g[1, 0] - c[1, 0]).norm() / c[1, 0].norm()) < 2e-6


# Scores so large that one unit of theirs in the last place counts in the softmax, and one value elsewhere in the head that sends products to
# the fp32 units: the backward kernels must have the forward pass's scores, bit for bit, for every other row.  Bound: four times the
# operators' error, relative 2-norm over the rows and keys that have nothing to do with the value (both errors are the rounding of the
# scores in the few rows with two shares of the same size; scores of two kinds make it eight times and more).
@pytest.mark.parametrize('where', ['q', 'do'])
@pytest.mark.parametrize('block,D', [(64, 64), (32, 128)])
@pytest.mark.parametrize('large', [100., 1000.])
def test_all_passes_have_the_same_scores(where, block, D, large):
    torch.manual_seed(block + D)
    n = 512 // block
    lay = _layout(2, n, n, 'random')
    lay[:, 0, n // 2:] = 0                                                # (keys that the value's row does not see)
    x = {t: torch.randn(1, 2, 512, D, device=DEV) for t in ('q', 'k', 'v', 'do')}
    x['q'] *= large
    x[where][0, 1, 7, 5] = 2. ** 31
    ops = _ops(lay, block)
    got, other = [_run(ops, x['q'], x['k'], x['v'], x['do'], fused, scale=D ** -0.5) for fused in (True, False)]
    ref = _dense(x['q'], x['k'], x['v'], x['do'], lay, block, D ** -0.5)
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        part = (0, 1, slice(64, None)) if name in ('o', 'dq') else (0, 1, slice(256, None))
        err, bound = [float((t[part].double() - r[part]).norm() / r[part].norm()) for t in (g, c)]
        assert err <= 4 * bound + 2 ** -23, (name, err, bound)


# A mask value that makes NaN of the rows that see its key: no other row takes notice, also where the key's tile is theirs
@pytest.mark.parametrize('value', [float('nan'), float('inf')])
@pytest.mark.parametrize('block,D', [(16, 64), (32, 64), (16, 128), (32, 128)])
def test_mask_values_of_keys_that_a_row_does_not_see(value, block, D):
    torch.manual_seed(block + D)
    n = 256 // block
    lay = _layout(2, n, n, 'random')
    ops = _ops(lay, block)
    q, k, v, do = [torch.randn(2, 2, 256, D, device=DEV) for _ in range(4)]
    kpm = torch.zeros(2, 256, device=DEV)
    kpm[0, 101] = value
    got, other = [_run(ops, q, k, v, do, fused, scale=D ** -0.5, key_padding_mask=kpm) for fused in (True, False)]
    for name, g, c in zip(('o', 'dq', 'dk', 'dv'), got, other):
        finite = torch.isfinite(c)
        assert bool((torch.isfinite(g) == finite).all()) and bool((torch.isnan(g) == torch.isnan(c)).all()), name
        assert float((g[finite] - c[finite]).norm() / c[finite].norm()) < 2e-6, name
    assert bool(torch.isfinite(got[0][0]).any()) and bool(torch.isnan(got[0][0]).any())


def test_padding_values_that_leave_no_score():
    """The lowest finite value (and -1e9) on every key of a sequence: fp32 rounds the scores away beside it and every key gets the same
    share, as from the operators; -inf on every key gives NaN for that sequence alone."""
    torch.manual_seed(3)
    lay = _layout(2, 4, 4, 'random')
    ops = _ops(lay, 64)
    q, k, v, do = [torch.randn(2, 2, 256, 64, device=DEV) for _ in range(4)]
    for value in (-1e9, torch.finfo(torch.float32).min, float('-inf')):
        kpm = torch.zeros(2, 256, device=DEV)
        kpm[0] = value
        got, other = [_run(ops, q, k, v, do, fused, scale=0.125, key_padding_mask=kpm) for fused in (True, False)]
        for g, c in zip(got, other):
            assert bool((torch.isnan(g) == torch.isnan(c)).all())
            assert float((g[1] - c[1]).norm() / c[1].norm()) < 2e-6
        if value != float('-inf'):
            assert float((got[0][0] - other[0][0]).norm() / other[0][0].norm()) < 2e-6


# Finite padding on every key of a sequence: the logits are rounded where they lie beside it, which is most of the error, and no more than
# the softmax operator rounds them.  Against 64 bits; a tenth for what rounding by other scores' last bits may do to it.
@pytest.mark.parametrize('value', [-100., -300., -1000., -10000., -65504., 1000.])
@pytest.mark.parametrize('block,D', [(32, 64), (64, 128)])
def test_padded_sequences_against_64_bits(value, block, D):
    torch.manual_seed(block)
    n = 256 // block
    lay = _layout(2, n, n, 'random')
    ops = _ops(lay, block)
    q, k, v, do = [torch.randn(2, 2, 256, D, device=DEV) for _ in range(4)]
    kpm = torch.zeros(2, 256, device=DEV)
    kpm[0] = value
    ref = _dense(q, k, v, do, lay, block, D ** -0.5, kpm)
    got, other = [_run(ops, q, k, v, do, fused, scale=D ** -0.5, key_padding_mask=kpm) for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        err, bound = [float((x.double() - r).norm() / r.norm()) for x in (g, c)]
        assert err <= 1.1 * bound + 2 ** -23, (name, err, bound)


# Rows whose share is one key's: their gradient of the scores is zero, and what is left of dp minus delta must not come back through a row of q
# or k of any size.  Against 64 bits; four times the operators' error (rows with two shares decide it where there are any).
@pytest.mark.parametrize('where', ['q', 'k'])
@pytest.mark.parametrize('size', [1e3, 1e5, 1e8, 1e15])
@pytest.mark.parametrize('block,D', [(64, 64), (32, 64), (16, 128)])
def test_saturated_rows(where, size, block, D):
    torch.manual_seed(block)
    n = 256 // block
    lay = _layout(2, n, n, 'random')
    x = {t: torch.randn(2, 2, 256, D, device=DEV) for t in ('q', 'k', 'v', 'do')}
    x[where][0, 1, 37] *= size
    ops = _ops(lay, block)
    ref = _dense(x['q'], x['k'], x['v'], x['do'], lay, block, D ** -0.5)
    got, other = [_run(ops, x['q'], x['k'], x['v'], x['do'], fused, scale=D ** -0.5) for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        err, bound = [float((t.double() - r).norm() / r.norm()) for t in (g, c)]
        assert err <= 4 * bound + 2 ** -23, (name, err, bound)


def _rows_error(x, r):
    """relative error of a row (2-norm), root mean square over the rows that are not zero"""
    e, n = (x.double() - r).norm(dim=-1), r.norm(dim=-1)
    return float(((e[n > 0] / n[n > 0]) ** 2).mean().sqrt())


# One value that sends a head's products to the fp32 units.  Against 64 bits row by row, since it dwarfs what has to do with it (and without its
# column where it only reaches that); twice the operators' error, which is of the same units in another order.
@pytest.mark.parametrize('where', ['q', 'k', 'v', 'do'])
@pytest.mark.parametrize('Z,H,R,C,block,D,kind,padded', [
    (2, 2, 16, 24, 32, 64, 'holes', True),
    (1, 2, 12, 8, 16, 64, 'holes', False),
    (1, 3, 40, 6, 64, 64, 'random', False),
    (1, 2, 40, 6, 64, 128, 'random', True),
    (1, 2, 8, 8, 16, 128, 'random', True),
])
def test_whole_values_against_64_bits(where, Z, H, R, C, block, D, kind, padded):
    torch.manual_seed(R + C + D)
    lay = _layout(H, R, C, kind)
    x = {t: torch.randn(Z, H, (R if t in ('q', 'do') else C) * block, D, device=DEV) for t in ('q', 'k', 'v', 'do')}
    x[where][0, 1, 37, 5] = 2. ** 31
    kw = dict(scale=D ** -0.5)
    if padded:
        kpm = torch.zeros(Z, C * block, device=DEV)
        kpm[0, block:block + 9] = float('-inf')
        kpm[-1, block + 5:] = -2.
        kw['key_padding_mask'] = kpm
    ops = _ops(lay, block)
    ref = _dense(x['q'], x['k'], x['v'], x['do'], lay, block, D ** -0.5, kw.get('key_padding_mask'))
    got, other = [_run(ops, x['q'], x['k'], x['v'], x['do'], fused, **kw) for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        if (where, name) in (('v', 'o'), ('do', 'dv'), ('k', 'dq'), ('q', 'dk')):
            g, c, r = [torch.cat((t[..., :5], t[..., 6:]), -1) for t in (g, c, r)]
        err, bound = _rows_error(g, r), _rows_error(c, r)
        assert err <= 2 * bound + 2 ** -22, (name, err, bound)


def test_sums_that_fp32_holds():
    """Values near the largest of fp32: shares times them add up to less than it, numerators would not."""
    torch.manual_seed(6)
    lay = _layout(2, 8, 8, 'random')
    ops = _ops(lay, 32)
    q, k, v, do = [torch.randn(2, 2, 256, 64, device=DEV) for _ in range(4)]
    huge = v.clone()
    huge[0, 1, ::3] = 3e38
    do *= 3e36
    for x, names in (((q, k, huge, do * 1e-38), ('o',)), ((q, k, v, do), ('o', 'dq', 'dk', 'dv'))):
        ref = _dense(*x, lay, 32, 0.125)
        got, other = [_run(ops, *x, fused, scale=0.125) for fused in (True, False)]
        for name, g, c, r in zip(names, got, other, ref):
            assert bool(torch.isfinite(c).all()) and bool(torch.isfinite(g).all()), name
            assert _rows_error(g, r) <= 2 * _rows_error(c, r) + 2 ** -22, name


# Operands and gradients of the scores far below one: they keep their 24 bits.  Against 64 bits, bound as in test_against_64_bits.
@pytest.mark.parametrize('sizes,scale', [(dict(do=-115), 0), (dict(v=-115), 0), (dict(v=-60, do=-60), 0), (dict(q=-118), 118), (dict(q=-60, k=-60), 120), (dict(k=-20, v=19, do=-100), 20)])
@pytest.mark.parametrize('block,D', [(32, 64), (64, 128)])
def test_small_operands(sizes, scale, block, D):
    torch.manual_seed(block)
    n = 256 // block
    lay = _layout(2, n, n, 'random')
    x = {t: torch.randn(2, 2, 256, D, device=DEV) for t in ('q', 'k', 'v', 'do')}
    for t, power in sizes.items():
        x[t].clamp_(-8, 8).mul_(2. ** (power if power < 0 else power - 3))
    scale = D ** -0.5 * 2. ** scale
    ops = _ops(lay, block)
    ref = _dense(x['q'], x['k'], x['v'], x['do'], lay, block, scale)
    got, other = [_run(ops, x['q'], x['k'], x['v'], x['do'], fused, scale=scale) for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        err, bound = [float((t.double() - r).norm() / r.norm()) for t in (g, c)]
        assert err <= bound + 2 ** -23, (name, err, bound)


def test_operands_that_are_copied_and_inference():
    """Odd strides, an expanded gradient, gradients of some operands only, and a forward pass alone (which keeps no parts of q)."""
    torch.manual_seed(4)
    lay = _layout(2, 8, 8, 'random')
    ops = _ops(lay, 32)
    q, k, v = [torch.randn(2, 2, 256, 64, device=DEV) for _ in range(3)]
    want = _run(ops, q, k, v, torch.ones(2, 2, 256, 64, device=DEV), True, scale=0.125)
    odd = torch.empty(2, 2, 256, 66, device=DEV)[..., 1:65].copy_(k)
    got = _run(ops, q.transpose(1, 2).contiguous().transpose(1, 2), odd, v, torch.ones(1, 1, 1, 1, device=DEV).expand(2, 2, 256, 64), True, scale=0.125)
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    for i in range(3):
        xs = [t.clone().requires_grad_(i == j) for j, t in enumerate((q, k, v))]
        (grad,) = torch.autograd.grad(ac.attention_chain(*ops, *xs, scale=0.125).sum(), xs[i])
        assert torch.equal(grad, want[1 + i])
    with torch.no_grad():
        assert torch.equal(ac.attention_chain(*ops, q, k, v, scale=0.125), want[0])


def test_result_may_change_before_the_backward_pass():
    """The operators keep neither the result nor anything that shares its memory: a program may change it in place."""
    torch.manual_seed(5)
    lay = _layout(2, 8, 8, 'random')
    ops = _ops(lay, 32)
    q, k, v, do = [torch.randn(2, 2, 256, 64, device=DEV) for _ in range(4)]
    want = _run(ops, q, k, v, do, True, scale=0.125)
    xs = [t.clone().requires_grad_() for t in (q, k, v)]
    o = ac.attention_chain(*ops, *xs, scale=0.125)
    o += 7.
    o.mul_(0.)
    grads = torch.autograd.grad(o, xs, do)
    assert all(float(g.abs().max()) == 0. for g in grads)
    o = ac.attention_chain(*ops, *xs, scale=0.125)
    o += 7.
    assert all(torch.equal(g, w) for g, w in zip(torch.autograd.grad(o, xs, do), want[1:]))


def test_calls_for_the_operators_make_no_tables():
    """A head dimension, or shapes, that the kernels do not take: the operators run (or raise), and no table of tiles is made for them."""
    lay = _layout(2, 8, 8, 'random')
    ops = _ops(lay, 32)
    q, k, v = [torch.randn(2, 2, 256, 32, device=DEV) for _ in range(3)]
    before = ac.fused_f32_calls
    ac.attention_chain(*ops, q, k, v)
    with pytest.raises(ValueError):
        ac.attention_chain(*ops, *[torch.randn(2, 3, 256, 64, device=DEV) for _ in range(3)])
    assert ac.fused_f32_calls == before and not ac._core_for(*ops)._tables
    ac.attention_chain(*ops, *[torch.randn(2, 2, 256, 64, device=DEV) for _ in range(3)])
    assert ac.fused_f32_calls == before + 1 and ac._core_for(*ops)._tables


# (random layouts of few blocks: tiles that are mostly holes, lines of a tile or two)
@pytest.mark.parametrize('Z,H,n,block,D,density,fused', [(2, 8, 128, 16, 64, 0.05, False), (4, 16, 64, 64, 64, 0.005, False), (2, 8, 32, 64, 64, 1., True),
                                                         (2, 8, 64, 32, 128, 0.05, False), (2, 8, 32, 64, 128, 1., True)])
def test_layouts_of_both_routes(Z, H, n, block, D, density, fused):
    """fp32 calls take the kernels where they are faster, the operators elsewhere"""
    g = torch.Generator().manual_seed(7)
    lay = (torch.rand((H, n, n), generator=g) < density).long()
    lay[:, range(n), range(n)] = 1
    q, k, v = [torch.randn(Z, H, n * block, D, device=DEV, requires_grad=True) for _ in range(3)]
    before = ac.fused_f32_calls
    ac.attention_chain(*_ops(lay, block), q, k, v, scale=D ** -0.5).sum().backward()
    assert ac.fused_f32_calls - before == int(fused)


@pytest.mark.parametrize('rows_of_mask', [1, 2])
@pytest.mark.parametrize('block,D', [(16, 64), (64, 128)])
def test_multiplied_masks_and_one_mask_for_all_batches(rows_of_mask, block, D):
    """mode 'mul': zeros are padding, every other value is none; a mask of one row serves all batches"""
    torch.manual_seed(8)
    n = 256 // block
    lay = _layout(2, n, n, 'random')
    q, k, v, do = [torch.randn(2, 2, 256, D, device=DEV) for _ in range(4)]
    keep = (torch.rand(rows_of_mask, 256, device=DEV) < 0.7).float() * 3.
    keep[:, 0] = 1.                                                       # (every row sees its key)
    add = torch.where(keep == 0, float('-inf'), 0.)
    ref = _dense(q, k, v, do, lay, block, 0.125, add.expand(2, 256))
    ops = _ops(lay, block)
    got, other = [_run(ops, q, k, v, do, fused, scale=0.125, key_padding_mask=keep, key_padding_mask_mode='mul') for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        err, bound = [float((x.double() - r).norm() / r.norm()) for x in (g, c)]
        assert err <= bound + 2 ** -23, (name, err, bound)
    assert all(torch.equal(a, b) for a, b in zip(got, _run(ops, q, k, v, do, True, scale=0.125, key_padding_mask=add)))


# Logits up to some hundreds: most rows have one or two shares.  Bound as in test_against_64_bits.
@pytest.mark.parametrize('times', [4., 16., 64.])
@pytest.mark.parametrize('block,D', [(32, 64), (64, 64), (16, 128)])
def test_large_logits(times, block, D):
    torch.manual_seed(block)
    n = 512 // block
    lay = _layout(2, n, n, 'random')
    q, k, v, do = [torch.randn(2, 2, 512, D, device=DEV) for _ in range(4)]
    ref = _dense(q, k, v, do, lay, block, times * D ** -0.5)
    ops = _ops(lay, block)
    got, other = [_run(ops, q, k, v, do, fused, scale=times * D ** -0.5) for fused in (True, False)]
    for name, g, c, r in zip(('o', 'dq', 'dk', 'dv'), got, other, ref):
        err, bound = [float((x.double() - r).norm() / r.norm()) for x in (g, c)]
        assert err <= 1.1 * bound + 2 ** -23, (name, err, bound)


@pytest.mark.parametrize('Z,R,block,D', [(2, 8, 32, 64), (1, 40, 64, 128)])
def test_capture_and_another_stream(Z, R, block, D):
    """A training step captured in a graph, replayed on new inputs with eager work between; and on a stream of its own."""
    torch.manual_seed(9)
    lay = _layout(3, R, 8, 'random')
    ops = _ops(lay, block)
    q, do = [torch.randn(Z, 3, R * block, D, device=DEV) for _ in range(2)]
    k, v = [torch.randn(Z, 3, 8 * block, D, device=DEV) for _ in range(2)]
    kpm = torch.zeros(Z, 8 * block, device=DEV)
    kpm[:, 3:9] = float('-inf')
    xs = [t.clone().requires_grad_() for t in (q, k, v)]

    def step():
        o = ac.attention_chain(*ops, *xs, scale=0.125, key_padding_mask=kpm)
        return (o.detach(),) + torch.autograd.grad(o, xs, do)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        on_side = step()
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(on_side, step()))
    graph = torch.cuda.CUDAGraph()
    before = ac.fused_f32_calls
    with torch.cuda.graph(graph):
        out = step()
    assert ac.fused_f32_calls == before + 1
    for i in range(3):
        for x in xs:
            x.data.normal_()
        do.normal_()
        graph.replay()
        replayed = [t.clone() for t in out]
        assert all(torch.equal(a, b) for a, b in zip(replayed, step())), i


def test_gradients_through_stored_softmax_gradients(monkeypatch):
    """FUSED_KV = False: fp32 has no kernels for it, the operators run."""
    monkeypatch.setattr(ac, 'FUSED_KV', False)
    torch.manual_seed(10)
    lay = _layout(2, 8, 8, 'random')
    ops = _ops(lay, 32)
    xs = [torch.randn(2, 2, 256, 64, device=DEV, requires_grad=True) for _ in range(3)]
    before = ac.fused_f32_calls
    o = ac.attention_chain(*ops, *xs, scale=0.125)
    assert ac.fused_f32_calls == before
    assert torch.equal(o, ops[2](ops[1](ops[0](xs[0], xs[1]), scale=0.125), xs[2]))
