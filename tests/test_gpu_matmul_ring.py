"""GPU: the wide dsd / dds kernels at the edges of their three-stage ring and of the 64-entry windows in which they hold the
table: lines of 1, 2, 3, 4, 63, 64, 65 and 66 blocks; blocks of 32 also on the kernel that works from lists."""
import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib
from torch_blocksparse.matmul import GroupPlan

pytestmark = pytest.mark.gpu


def _lines():
    """[16 lines, 66 reduction blocks]: neighbouring lines with nested blocks, so that a group of four has as many entries as its longest"""
    lines = torch.zeros(16, 66, dtype=torch.int64)
    for i, n in enumerate((1, 1, 1, 1, 2, 1, 2, 2, 3, 66, 4, 65, 64, 63, 62, 64)):
        lines[i, 66 - n:] = 1
    return lines


# launches large enough for the wide kernels in every orientation; blocks of 32: the kernel on lists of blocks, which this layout takes, and
# the one on groups of four lines, whose ring and windows these are
@pytest.mark.parametrize('block,Z,lists', [(32, 12, True), (32, 12, False), (64, 5, None)])
@pytest.mark.parametrize('mode', ['dsd', 'dds'])
@pytest.mark.parametrize('trans_a', [False, True])
@pytest.mark.parametrize('trans_b', [False, True])
def test_ring_and_table_windows(mode, block, Z, lists, trans_a, trans_b, monkeypatch):
    dtype = torch.float16 if trans_a == trans_b else torch.bfloat16
    lines, free = _lines(), 2048 - 24                          # (the last tile of the free dimension is not full)
    K = 66 * block
    tiles = -(-free // 256) * Z                                # the sizes from which the library takes the wide kernels
    assert 16 // 4 * tiles >= 384 if block == 32 else 16 * tiles > 512
    # the sparse operand as stored: dsd op(A) is [lines, reduction], dds op(B) is [reduction, lines]
    stored = lines if (mode == 'dsd') != (trans_a if mode == 'dsd' else trans_b) else lines.t()
    lay = stored.contiguous()[None]
    g = torch.Generator(device='cuda').manual_seed(3)
    sp = torch.randn((Z, int(lay.sum()), block, block), generator=g, device='cuda').mul_(K ** -0.5).to(dtype)
    dense_trans = trans_b if mode == 'dsd' else trans_a
    shape = (Z, 1, K, free) if (mode == 'dsd') != dense_trans else (Z, 1, free, K)
    dn = torch.randn(shape, generator=g, device='cuda').to(dtype)
    if lists is False:
        monkeypatch.setattr(GroupPlan, 'build_xsd_chunks', staticmethod(lambda *args, **kw: None))
    dot = tb.MatMul(lay, block, mode, trans_a=trans_a, trans_b=trans_b)
    got = (dot(sp, dn) if mode == 'dsd' else dot(dn, sp)).float()
    if block == 32:
        assert dot.make_lut(dtype, sp.device)[0].gplan_wide.flags == (_lib.FLAG_PLAN_TILES if lists else 0)
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
    assert 64 // 4 * (1024 // 256) * 6 == 384 and dot.make_lut(sp.dtype, sp.device)[0].gplan_wide is None
    for _ in range(3):
        whole.zero_()
        graph.replay()
        torch.cuda.synchronize()
        # the same products in another order of their fp32 sums: one unit of the 16-bit result
        assert bool(((whole.float() - parts.float()).abs() <= 2. ** -10 * parts.float().abs() + 2. ** -12).all())
    torch.testing.assert_close(dot(sp, dn), whole, rtol=2. ** -10, atol=2. ** -12)
    assert dot.make_lut(sp.dtype, sp.device)[0].gplan_wide is not None


@pytest.mark.parametrize('mode,block,trans_a,trans_b', [
    ('dsd', 64, False, False), ('dsd', 128, False, True), ('dsd', 64, True, False), ('dds', 64, False, False), ('dds', 128, True, False),
    ('sdd', 32, False, True), ('sdd', 32, True, False), ('sdd', 16, False, True)])
def test_operands_beyond_the_reach_of_the_wide_kernels(mode, block, trans_a, trans_b):
    """Dense rows so far apart that a tile's byte offsets leave 32 bits: the general kernels take the launch."""
    torch.manual_seed(block)
    M, N, K = (256, 256, 256)
    ld = 2 ** 31 // (128 if mode == 'sdd' else 256) + 64
    shape = (M if mode == 'sdd' else K, K if mode == 'sdd' else N)
    lay = (torch.rand(1, shape[0] // block if mode == 'sdd' else M // block, (N if mode == 'sdd' else K) // block) < 0.6).long()
    lay[0, :, 0] = lay[0, 0, :] = 1
    far = torch.empty(256 * ld, device='cuda', dtype=torch.float16).as_strided((1, 1, 256, 256), (8, 8, ld, 1))
    far.copy_(torch.randn(256, 256, device='cuda').half())
    sp = torch.randn(1, int(lay.sum()), block, block, device='cuda').half()
    dn = torch.randn(1, 1, 256, 256, device='cuda').half()
    a, b = {'sdd': (far, dn), 'dsd': (sp, far), 'dds': (far, sp)}[mode]
    got = tb.MatMul(lay, block, mode, trans_a=trans_a, trans_b=trans_b)(a, b).float()
    h, r, c = lay.nonzero().unbind(1)

    def full(t):
        if t is not sp:
            return t.float().contiguous()
        x = torch.zeros(1, 1, 256 // block, 256 // block, block, block, device='cuda')
        x[:, h, r, c] = sp.float()
        return x.transpose(3, 4).reshape(1, 1, 256, 256)
    x, y = full(a), full(b)
    x, y = (x.transpose(2, 3) if trans_a else x).contiguous(), (y.transpose(2, 3) if trans_b else y).contiguous()
    ref, terms = torch.matmul(x, y), torch.matmul(x.abs(), y.abs())
    if mode == 'sdd':
        blocks = lambda t: t.reshape(1, 1, 256 // block, block, 256 // block, block).transpose(3, 4)[:, h, r, c]
        ref, terms = blocks(ref), blocks(terms)
    bound = 2. ** -11 * ref.abs() + 2 * K * 2. ** -24 * terms + 2. ** -24      # as above
    assert got.shape == ref.shape and bool(((got - ref).abs() <= bound).all()), (got - ref).abs().max().item()
