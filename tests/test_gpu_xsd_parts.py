"""GPU: dsd / dds products in fp32 whose long segments run in parts, and the tiles of the free dimension (64, 128, 256 wide): every
orientation, segments around the length of a part, empty ones, free dimensions around the tile widths; the same bits every time."""
import ctypes

import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib
from torch_blocksparse.matmul import _sparse_matmul
from helpers import run_matmul_case

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _outliers(block, by_rows):
    """one line of 96 blocks of 32 (of other sizes: as many elements), one of a part's length, one a block longer, an empty one, the others of 1 - 3"""
    n = 96 * 32 // block
    lay = torch.zeros(2, 8, n, dtype=torch.int64)
    lay[:, :, 0] = 1
    lay[0, 1] = 1
    lay[0, 2, :n // 6] = 1
    lay[0, 3, :n // 6 + 1] = 1
    lay[0, 4] = 0
    lay[1, 5, 3:5] = 1
    return lay if by_rows else lay.transpose(1, 2).contiguous()


@pytest.mark.parametrize('block', [16, 32, 64])
@pytest.mark.parametrize('mode,trans_a,trans_b', [('dsd', False, False), ('dsd', True, False), ('dsd', True, True), ('dds', False, False), ('dds', True, True), ('dds', False, True)])
@pytest.mark.parametrize('free', [20, 64, 132])
def test_long_segments_against_the_oracle(block, mode, trans_a, trans_b, free):
    trans = trans_a if mode == 'dsd' else trans_b
    lay = _outliers(block, by_rows=(not trans) if mode == 'dsd' else trans)
    R, C = lay.shape[1] * block, lay.shape[2] * block
    if mode == 'dsd':
        M, K = (C, R) if trans else (R, C)
        sizes = dict(M=M, K=K, N=free)
    else:
        K, N = (C, R) if trans else (R, C)
        sizes = dict(M=free, K=K, N=N)
    dev = torch.device(DEV)
    lut, _, width, _ = _sparse_matmul.make_dxx_lut(lay, block, 8, trans if mode == 'dds' else not trans, dev)
    part_blocks = ctypes.c_int(0)
    parts = _lib.load().bsp_xsd_parts(_lib.F32, block, width, lut.longest, lut.nnz, free, 1, 0, ctypes.byref(part_blocks))
    assert lut.longest == 96 * 32 // block and parts > 1 and (parts - 1) * part_blocks.value < lut.longest <= parts * part_blocks.value
    run_matmul_case(mode, trans_a, trans_b, block, torch.float32, Z=1, H=2, layout=lay, dist='randn', scale=sizes['K'] ** -0.5, seed=free, backward=False, **sizes)


@pytest.mark.parametrize('block,dtype', [(32, torch.float32), (32, torch.float16), (128, torch.float32), (128, torch.bfloat16), (64, torch.float32)])
@pytest.mark.parametrize('free', [64, 68, 128, 132, 260])
def test_tiles_of_the_free_dimension(block, dtype, free):
    free = free if dtype == torch.float32 else (free + 7) // 8 * 8
    for mode, ta, tb_ in (('dsd', False, True), ('dsd', True, False), ('dds', False, False), ('dds', True, True)):
        sizes = dict(M=3 * block, K=4 * block, N=free) if mode == 'dsd' else dict(M=free, K=4 * block, N=3 * block)
        run_matmul_case(mode, ta, tb_, block, dtype, Z=2, H=1, density=0.6, dist='randn', scale=0.1, seed=free, backward=False, **sizes)


def test_parts_are_added_in_order_and_the_workspace_is_checked():
    lay = _outliers(32, True)
    op = tb.MatMul(lay, 32, 'dsd')
    torch.manual_seed(1)
    sp, dn = torch.randn(1, int(lay.sum()), 32, 32, device=DEV), torch.randn(1, 2, 96 * 32, 64, device=DEV)
    first = op(sp, dn)
    for _ in range(3):
        assert torch.equal(op(sp, dn), first)
    lut, _, width, _ = op.make_lut(torch.float32, dn.device)[:4]
    lib, c = _lib.load(), torch.empty_like(first)

    def call(parts, per, short=0):
        need = lib.bsp_xsd_parts_workspace_bytes(32, width, 64, 1, parts)
        ws = torch.full((max(need, 16),), 255, dtype=torch.uint8, device=DEV)             # (not a number, read as floats)
        rc = lib.bsp_xsd_matmul_parts(0, _lib.F32, _lib.ptr(sp), _lib.ptr(dn), _lib.ptr(c), 0, 0, 0, 1, 64, 0, dn.stride(0), dn.stride(1), 64, c.stride(0), c.stride(1), 64, 32,
                                      _lib.ptr(lut), _lib.ptr(lut.planbuf), width, parts, per, _lib.ptr(ws), need - short, _lib.stream_ptr(dn.device))
        torch.cuda.synchronize()
        return rc

    for per in (1, 7, 95):
        assert call(-(-96 // per), per) == _lib.OK
        assert float((c - first).abs().max()) <= 1e-5 * float(96 * 32 * sp.abs().max() * dn.abs().max())
    assert call(4, 24, 16) == _lib.ERR_CAPACITY and call(1, 96) < 0 and call(2, 0) < 0
