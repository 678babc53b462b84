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


def test_first_wide_launch_under_capture():
    """operators warmed up with a batch too small for the wide kernel, then captured with one that takes it: the plan of the
    wide kernel cannot be built then, and the ordinary one (with its chains of long lines) serves"""
    lay = torch.eye(64, dtype=torch.int64)[None]
    lay[0, 7, :] = 1
    lay[0, :, 9] = 1
    dot = tb.MatMul(lay, 32, 'dsd')
    torch.manual_seed(5)
    sp = torch.randn(6, int(lay.sum()), 32, 32, device='cuda').half() * 0.1
    dn = torch.randn(6, 1, 2048, 1024, device='cuda').half()
    parts = torch.cat([dot(sp[i:i + 1], dn[i:i + 1]) for i in range(6)])      # 64 workgroups of the wide kernel a call
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        whole = dot(sp, dn)                                                  # 384
    for _ in range(3):
        whole.zero_()
        graph.replay()
        torch.cuda.synchronize()
        # the same products in another order of their fp32 sums: one unit of the 16-bit result
        assert bool(((whole.float() - parts.float()).abs() <= 2. ** -10 * parts.float().abs() + 2. ** -12).all())
    torch.testing.assert_close(dot(sp, dn), whole, rtol=2. ** -10, atol=2. ** -12)
