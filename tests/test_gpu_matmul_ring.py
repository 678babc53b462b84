"""GPU: the wide dsd / dds kernels at the edges of their three-stage ring and of the 64-entry windows in which they hold the
table: lines of 1, 2, 3, 4, 63, 64, 65 and 66 blocks."""
import pytest
import torch

import torch_blocksparse as tb

pytestmark = pytest.mark.gpu


def _lines():
    """[16 lines, 66 reduction blocks]: neighbouring lines with nested blocks, so that a group of four has as many entries as its longest"""
    lines = torch.zeros(16, 66, dtype=torch.int64)
    for i, n in enumerate((1, 1, 1, 1, 2, 1, 2, 2, 3, 66, 4, 65, 64, 63, 62, 64)):
        lines[i, 66 - n:] = 1
    return lines


@pytest.mark.parametrize('block,Z', [(32, 12), (64, 5)])      # launches large enough for the wide kernels in every orientation
@pytest.mark.parametrize('mode', ['dsd', 'dds'])
@pytest.mark.parametrize('trans_a', [False, True])
@pytest.mark.parametrize('trans_b', [False, True])
def test_ring_and_table_windows(mode, block, Z, trans_a, trans_b):
    dtype = torch.float16 if trans_a == trans_b else torch.bfloat16
    lines, free = _lines(), 2048 - 24                          # (the last tile of the free dimension is not full)
    K = 66 * block
    # the sparse operand as stored: dsd op(A) is [lines, reduction], dds op(B) is [reduction, lines]
    stored = lines if (mode == 'dsd') != (trans_a if mode == 'dsd' else trans_b) else lines.t()
    lay = stored.contiguous()[None]
    g = torch.Generator(device='cuda').manual_seed(3)
    sp = torch.randn((Z, int(lay.sum()), block, block), generator=g, device='cuda').mul_(K ** -0.5).to(dtype)
    dense_trans = trans_b if mode == 'dsd' else trans_a
    shape = (Z, 1, K, free) if (mode == 'dsd') != dense_trans else (Z, 1, free, K)
    dn = torch.randn(shape, generator=g, device='cuda').to(dtype)
    dot = tb.MatMul(lay, block, mode, trans_a=trans_a, trans_b=trans_b)
    got = (dot(sp, dn) if mode == 'dsd' else dot(dn, sp)).float()
    full = torch.zeros((Z, 1, lay.size(1), lay.size(2), block, block), device='cuda')
    h, r, c = lay.nonzero().unbind(1)
    full[:, h, r, c] = sp.float()
    full = full.transpose(3, 4).reshape(Z, 1, lay.size(1) * block, lay.size(2) * block)
    a, b = (full, dn.float()) if mode == 'dsd' else (dn.float(), full)
    a, b = (a.transpose(2, 3) if trans_a else a).contiguous(), (b.transpose(2, 3) if trans_b else b).contiguous()
    ref, terms = torch.matmul(a, b), torch.matmul(a.abs(), b.abs())
    # half a unit of the 16-bit result, and two fp32 sums of up to K terms in different orders
    unit = 2. ** -11 if dtype == torch.float16 else 2. ** -8
    bound = unit * ref.abs() + 2 * K * 2. ** -24 * terms + 2. ** -24
    assert got.shape == ref.shape and bool(((got - ref).abs() <= bound).all()), (got - ref).abs().max().item()
