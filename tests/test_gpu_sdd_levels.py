"""GPU: the sdd kernel that takes every pack level of the table in one launch (blocks of 16 and 32): levels of every size, a
last level whose super-blocks do not fill its workgroups, reductions around the depth of the register ring, every
orientation; and the C entry point against one call per level, bit for bit."""
import ctypes

import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib
from torch_blocksparse.matmul import _sparse_matmul
from helpers import run_matmul_case

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _layout(block, kind):
    """per head: block-rows and -columns of whole squares, pairs and single blocks"""
    n = 256 // block
    lay = torch.zeros(2, n, n, dtype=torch.int64)
    if kind != 'single':
        lay[0, :4, :8] = 1
        lay[1, 4:6, 2:4] = 1
    if kind != 'square':
        lay[0, 5, 1::2] = 1
        lay[1, n - 1, n - 1] = 1
        lay[1, 0, 0] = 1
    return lay


@pytest.mark.parametrize('block', [16, 32])
@pytest.mark.parametrize('kind', ['all', 'single', 'square'])
@pytest.mark.parametrize('dtype,K', [(torch.float32, 16), (torch.float32, 80), (torch.float32, 144), (torch.float16, 48), (torch.bfloat16, 240)])
def test_levels_against_the_oracle(block, kind, dtype, K):
    lay = _layout(block, kind)
    for trans_a, trans_b, Z in ((False, False, 1), (True, False, 3), (False, True, 2), (True, True, 1)):
        run_matmul_case('sdd', trans_a, trans_b, block, dtype, Z=Z, H=2, M=256, N=256, K=K, layout=lay, dist='randn', scale=K ** -0.5, seed=K, backward=False)


@pytest.mark.parametrize('block', [16, 32])
def test_one_call_for_all_levels_gives_the_bits_of_a_call_per_level(block):
    torch.manual_seed(block)
    lay = _layout(block, 'all')
    luts, _, widths, packs = _sparse_matmul.make_sdd_lut(lay, block, torch.float32, torch.device(DEV))
    assert len(packs) == (3 if block == 16 else 2) and sum((w * p * p for w, p in zip(widths, packs))) >= int(lay.sum())
    a, b = torch.randn(2, 2, 256, 96, device=DEV), torch.randn(2, 2, 256, 96, device=DEV)
    lib = _lib.load()

    def args(c):
        return (_lib.F32, _lib.ptr(a), _lib.ptr(b), _lib.ptr(c), 0, 1, 2, 96, a.stride(0), a.stride(1), 96, b.stride(0), b.stride(1), 96, c.stride(0), block)

    one, many = [torch.full((2, int(lay.sum()), block, block), float('nan'), device=DEV) for _ in range(2)]
    null, st = ctypes.c_void_p(0), _lib.stream_ptr(torch.device(DEV))
    valid = [getattr(t, 'valid', None) for t in luts]
    for lut, v, w, p in zip(luts, valid, widths, packs):
        assert lib.bsp_sdd_matmul(*args(many), p, _lib.ptr(lut), _lib.ptr(v), w, null, 0, 0, 0, st) == _lib.OK
    n = len(luts)
    arrays = ((ctypes.c_int * n)(*packs), (ctypes.c_void_p * n)(*[t.data_ptr() for t in luts]),
              (ctypes.c_void_p * n)(*[None if v is None else v.data_ptr() for v in valid]), (ctypes.c_int64 * n)(*widths))
    assert lib.bsp_sdd_matmul_levels(*args(one), n, *arrays, null, 0, 0, 0, st) == _lib.OK
    torch.cuda.synchronize()
    assert not bool(torch.isnan(one).any()) and torch.equal(one, many)
    # the same level twice, a level that the block size does not have, no level
    twice = (ctypes.c_int * n)(*([packs[0]] * n))
    assert lib.bsp_sdd_matmul_levels(*args(one), n, twice, *arrays[1:], null, 0, 0, 0, st) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_sdd_matmul_levels(*args(one), 1, (ctypes.c_int * 1)(8), *arrays[1:], null, 0, 0, 0, st) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_sdd_matmul_levels(*args(one), 0, *arrays, null, 0, 0, 0, st) < 0
