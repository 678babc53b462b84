"""GPU: the sdd kernel for long reductions that works from tiles with lists of blocks (block 32, fp16 / bf16): against the general kernel
in every orientation, block-rows that do not fill a tile, tiles of one block and of 64, both ends of the reduction; and the rule that
brings it into a product."""
import ctypes

import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib, matmul
from torch_blocksparse.matmul import GroupPlan, _sparse_matmul
from helpers import assert_close, guard_allocations, random_layout

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _layout(kind):
    if kind == 'one block':
        lay = torch.zeros(1, 3, 2, dtype=torch.int64)
        lay[0, 2, 1] = 1
        return lay
    if kind == 'full':                                    # four columns fill a tile
        return torch.ones(2, 16, 9, dtype=torch.int64)
    if kind == 'ragged':                                  # 21 block-rows: a tile of five; a head without blocks in its second sixteen
        lay = random_layout((2, 21, 37), 0.3, 5)
        lay[1, 16:] = 0
        return lay
    return random_layout((2, 32, 64), 0.08, 7)            # sixteen columns before 64 blocks


@pytest.mark.parametrize('kind', ['one block', 'full', 'ragged', 'thin'])
@pytest.mark.parametrize('dtype,K', [(torch.float16, 256), (torch.bfloat16, 288), (torch.float16, 544)])
def test_tiles_against_the_general_kernel(kind, dtype, K):
    lay = _layout(kind)
    H, R, C = lay.shape
    dev, Z, nnz = torch.device(DEV), 2, int(lay.sum())
    tiles = GroupPlan.build_sdd_tiles(lay, dev)
    t = tiles.table.view(-1, 148).cpu()
    assert int(t[:, 3].sum()) == nnz and int(t[:, 3].max()) <= 64 and int(t[:, 2].max()) <= 16
    ids = torch.cat([row[20:20 + row[3]] for row in t])
    assert ids.sort().values.tolist() == list(range(nnz))
    luts, _, widths, packs = _sparse_matmul.make_sdd_lut(lay, 32, dtype, dev)
    lib, st = _lib.load(), _lib.stream_ptr(dev)
    torch.manual_seed(K)
    for ta, tb_ in ((0, 0), (1, 0), (0, 1), (1, 1)):
        a = torch.randn((Z, H) + ((K, R * 32) if ta else (R * 32, K)), device=DEV).to(dtype) * K ** -0.5
        b = torch.randn((Z, H) + ((C * 32, K) if tb_ else (K, C * 32)), device=DEV).to(dtype)
        ref, got = [torch.full((Z, nnz, 32, 32), float('nan'), device=DEV, dtype=dtype) for _ in range(2)]

        def args(c):
            return (_lib.DTYPES[dtype], _lib.ptr(a), _lib.ptr(b), _lib.ptr(c), ta, tb_, Z, K, a.stride(0), a.stride(1), a.stride(2), b.stride(0), b.stride(1), b.stride(2), c.stride(0), 32)

        for lut, w, p in zip(luts, widths, packs):
            v = getattr(lut, 'valid', None)
            assert lib.bsp_sdd_matmul(*args(ref), p, _lib.ptr(lut), _lib.ptr(v), w, None, 0, 0, _lib.FLAG_GENERAL_ONLY, st) == _lib.OK
        assert lib.bsp_sdd_matmul(*args(got), 0, None, None, C, _lib.ptr(tiles.table), tiles.n_groups, R, _lib.FLAG_PLAN_TILES, st) == _lib.OK_WHOLE_LAYOUT
        torch.cuda.synchronize()
        assert_close(got, ref, dtype, 'tiles %s ta=%d tb=%d' % (kind, ta, tb_))
    # what the kernel does not serve: fp32, a short reduction, one that is no multiple of 32, blocks of 16
    call = lambda dtype=_lib.F16, K=K, block=32: lib.bsp_sdd_matmul(dtype, _lib.ptr(a), _lib.ptr(b), _lib.ptr(got), 1, 1, 1, K, 0, 0, a.stride(2), 0, 0, b.stride(2), 0, block, 0, None, None, C,
                                                                    _lib.ptr(tiles.table), tiles.n_groups, R, _lib.FLAG_PLAN_TILES, st)
    assert call(dtype=_lib.F32) == _lib.NEEDS_TABLE and call(K=224) == _lib.NEEDS_TABLE and call(K=272) == _lib.NEEDS_TABLE and call(block=16) == _lib.NEEDS_TABLE


def test_a_product_takes_them_where_there_are_enough(monkeypatch):
    lay = random_layout((8, 32, 32), 0.5, 3)              # 8 x 2 groups of sixteen rows, four or five tiles each
    torch.manual_seed(2)
    a, b = torch.randn(4, 8, 1024, 256, device=DEV).half(), torch.randn(4, 8, 1024, 256, device=DEV).half()
    op = tb.MatMul(lay, 32, 'sdd', trans_b=True)
    with guard_allocations('sdd tiles'):
        got = op(a, b)
        again = op(a, b)
    luts = op.make_lut(torch.float16, a.device)[0]
    assert luts.tiles is not None and luts.tiles_for(4) is luts.tiles and torch.equal(got, again)
    assert luts.tiles_for(1) is None                      # too few workgroups
    monkeypatch.setattr(matmul, 'KERNEL_FLAGS', _lib.FLAG_GENERAL_ONLY)
    assert_close(got, op(a, b), torch.float16, 'sdd')
    thin = tb.MatMul(random_layout((8, 64, 64), 0.05, 3), 32, 'sdd', trans_b=True).make_lut(torch.float16, a.device)[0]
    assert thin.tiles_for(64) is None                     # tiles of sixteen columns hold 18 blocks each
    dense = tb.MatMul(random_layout((8, 32, 32), 0.9, 3), 32, 'sdd', trans_b=True).make_lut(torch.float16, a.device)[0]
    assert dense.tiles_for(64) is None and dense.tiles is None
