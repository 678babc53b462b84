"""GPU: the native host side of the launches (csrc/launch.cpp) against the general one in Python: the same bits for the forms that
it takes, nothing for those that it leaves (copies, padding, shapes that do not fit), the same errors, and operators that are copied
after use."""
import copy
import pickle
import types

import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib, attention_core as ac
from helpers import random_layout

pytestmark = pytest.mark.gpu
DEV = 'cuda'
NOTHING = ('xsd', 'sdd', 'softmax_fwd', 'softmax_bwd')


def _general(monkeypatch, calls=None):
    """only the general host side (calls: count the native one's refusals and acceptances instead)"""
    real = _lib.native()
    if calls is None:
        fake = types.SimpleNamespace(**{n: (lambda *a: None) if n in NOTHING else getattr(real, n) for n in dir(real) if not n.startswith('_')})
    else:
        def counted(name):
            def call(*a):
                r = getattr(real, name)(*a)
                calls.append((name, r is not None))
                return r
            return call
        fake = types.SimpleNamespace(**{n: counted(n) for n in dir(real) if not n.startswith('_')})
    monkeypatch.setattr(_lib, 'native', lambda: fake)


def _forms(mode, ta, tb_, block, dtype, lay, Z, N):
    """operands as they lie in memory: packed, cut out of something larger, expanded over the batch, transposed in memory"""
    H, R, C = lay.shape
    nnz = int(lay.sum())
    torch.manual_seed(N)
    if mode == 'sdd':
        dense = [(N, R * block) if ta else (R * block, N), (C * block, N) if tb_ else (N, C * block)]
    else:
        red = (R if (ta if mode == 'dsd' else not tb_) else C) * block
        dense = [(N, red) if (tb_ if mode == 'dsd' else not ta) else (red, N)]
    base = [torch.randn((Z, H) + s, device=DEV).to(dtype) for s in dense]
    sparse = torch.randn(Z, nnz, block, block, device=DEV).to(dtype)
    wide = [torch.randn(Z, H, s[0] + 3, s[1] + 16, device=DEV).to(dtype)[:, :, 1:s[0] + 1, 8:8 + s[1]] for s in dense]
    odd = [torch.randn(Z, H, s[0], s[1] + 3, device=DEV).to(dtype)[..., :s[1]] for s in dense]
    turned = [torch.randn(Z, H, s[1], s[0], device=DEV).to(dtype).transpose(2, 3) for s in dense]
    heads = [torch.randn(Z, s[0], H, s[1], device=DEV).to(dtype).transpose(1, 2) for s in dense]
    for ds in (base, wide, odd, turned, heads):
        if mode == 'sdd':
            yield ds[0], ds[1]
        else:
            for sp in (sparse, sparse[:1], sparse[0], sparse.transpose(2, 3)):
                yield (sp, ds[0]) if mode == 'dsd' else (ds[0], sp)


@pytest.mark.parametrize('mode', ['sdd', 'dsd', 'dds'])
@pytest.mark.parametrize('block,dtype', [(16, torch.float32), (16, torch.float16), (32, torch.bfloat16), (32, torch.float16), (64, torch.float16), (64, torch.float32), (128, torch.bfloat16)])
def test_products_in_every_form(mode, block, dtype, monkeypatch):
    lay = random_layout((2, 4, 6), 0.4, block)
    sizes = (16, 64, 272, 512) if mode == 'sdd' else (1, 17, 64, 264)
    calls = []
    for ta, tb_, N, Z in ((False, False, sizes[0], 1), (True, False, sizes[1], 2), (False, True, sizes[2], 2), (True, True, sizes[3], 1)):
        for a, b in _forms(mode, ta, tb_, block, dtype, lay, Z, N):
            results = []
            for general in (False, True):
                with monkeypatch.context() as m:
                    _general(m, None if general else calls)
                    op = tb.MatMul(lay, block, mode, trans_a=ta, trans_b=tb_)
                    for rep in range(2):                  # (what the first call builds on demand is there in the second)
                        x, y = a.detach(), b.detach()
                        # (the gradient of the sparse operand reduces over the free dimension: a multiple of 16)
                        wrt = [t.requires_grad_() for t, sparse in ((x, mode == 'dsd'), (y, mode == 'dds')) if not sparse or N % 16 == 0]
                        c = op(x, y)
                        g = torch.autograd.grad(c, wrt, torch.ones_like(c))
                    results.append((c.detach(),) + g)
            for one, two in zip(*results):
                assert one.shape == two.shape and torch.equal(one, two), (ta, tb_, N, tuple(a.stride()), tuple(b.stride()))
    kept = [n for n, taken in calls if n in ('sdd', 'xsd') and taken]
    left = [n for n, taken in calls if n in ('sdd', 'xsd') and not taken]
    assert 'sdd' in kept and 'xsd' in kept and left


@pytest.mark.parametrize('dtype', [torch.float16, torch.float32])
def test_softmax_in_every_form(dtype, monkeypatch):
    H, R, block, Z = 2, 4, 32, 2
    lay = random_layout((H, R, R), 0.5, 4, at_least_one_per_row=True)
    L, nnz = R * block, int(lay.sum())
    torch.manual_seed(1)
    rpe, mask = torch.randn(L, L, device=DEV).to(dtype), (torch.rand(L, L, device=DEV) < 0.8).to(dtype)
    kpm = torch.zeros(Z, L, device=DEV).to(dtype)
    kpm[1, :5] = -2.
    for kw in (dict(), dict(rpe=rpe), dict(rpe=torch.randn(H, L, L, device=DEV).to(dtype)), dict(rpe=torch.randn(1, H, L, L + 8, device=DEV).to(dtype)),
               dict(rpe=torch.randn(Z, 1, L, L, device=DEV).to(dtype)), dict(rpe=rpe.t()), dict(key_padding_mask=kpm, attn_mask=mask, attn_mask_mode='mul'),
               dict(key_padding_mask=kpm[:1]), dict(key_padding_mask=torch.zeros(Z, L + 1, device=DEV).to(dtype)[:, 1:]), dict(attn_mask=mask.t(), attn_mask_mode='mul')):
        results = []
        for general in (False, True):
            with monkeypatch.context() as m:
                if general:
                    _general(m)
                torch.manual_seed(2)
                x = torch.randn(Z, nnz, block, block, device=DEV).to(dtype).requires_grad_()
                y = tb.Softmax(lay, block)(x * 1., scale=0.5, **kw)
                results.append((y.detach(),) + torch.autograd.grad(y, x, torch.randn_like(y)))
        for one, two in zip(*results):
            assert torch.equal(torch.nan_to_num(one), torch.nan_to_num(two)), list(kw)


def test_errors_are_those_of_the_general_path():
    lay = random_layout((2, 4, 6), 0.4, 1)
    nnz = int(lay.sum())
    a, b = torch.randn(1, 2, 128, 64, device=DEV), torch.randn(1, 2, 64, 192, device=DEV)
    sdd = tb.MatMul(lay, 32, 'sdd')
    sdd(a, b)
    for x, y in ((a[:, :1], b), (a, b[:, :, :, :160]), (a, b.half()), (a[..., :56], b[:, :, :56])):
        with pytest.raises(ValueError):
            sdd(x, y)
    with pytest.raises(_lib.BlocksparseLibraryError):
        sdd(a, b.cpu())
    dsd, s = tb.MatMul(lay, 32, 'dsd'), torch.randn(1, nnz, 32, 32, device=DEV)
    for x, y in ((s[:, :-1], torch.randn(1, 2, 192, 64, device=DEV)), (s, torch.randn(1, 2, 160, 64, device=DEV)), (torch.randn(3, nnz, 32, 32, device=DEV), torch.randn(2, 2, 192, 64, device=DEV))):
        with pytest.raises(ValueError):
            dsd(x, y)
    sm = tb.Softmax(lay, 32)
    for x, kw in ((s[:, :-1].contiguous(), {}), (s.transpose(2, 3), {}), (s.clone(), dict(attn_mask=torch.ones(64, 64, device=DEV))), (s.clone(), dict(rpe=torch.ones(3, 128, 192, device=DEV)))):
        with pytest.raises(ValueError):
            sm(x, **kw)


def test_operators_can_be_copied_after_use():
    lay = random_layout((2, 4, 4), 0.5, 2, at_least_one_per_row=True)
    lin = tb.Linear(128, 128, 32, lay[:1]).to(DEV)
    x = torch.randn(7, 128, device=DEV)
    q = torch.randn(1, 2, 256, 64, device=DEV).half()
    sdd, sm = tb.MatMul(lay, 64, 'sdd', trans_b=True), tb.Softmax(lay, 64)
    ops = (sdd, sm, tb.MatMul(lay, 64, 'dsd'))
    y, o = lin(x), ac.attention_chain(*ops, q, q, q, scale=0.1)
    p = sm(sdd(q, q))
    assert torch.equal(copy.deepcopy(lin)(x), y) and torch.equal(ac.attention_chain(*copy.deepcopy(ops), q, q, q, scale=0.1), o)
    two = copy.deepcopy((sdd, sm))
    assert torch.equal(two[1](two[0](q, q)), p)
    assert torch.equal(pickle.loads(pickle.dumps(tb.MatMul(lay, 64, 'sdd', trans_b=True)))(q, q), sdd(q, q))
