"""GPU: the sdd kernel that takes every pack level of the table in one launch (blocks of 16 and 32): levels of every size, a
last level whose super-blocks do not fill its workgroups, reductions around the depth of the register ring, every
orientation; and the C entry point against one call per level, bit for bit."""
import ctypes
import threading

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
    tail = (null, 0, 0, 1, 0, null, 0, 0, st)
    assert lib.bsp_sdd_matmul_levels(*args(one), n, *arrays, *tail) == _lib.OK
    torch.cuda.synchronize()
    assert not bool(torch.isnan(one).any()) and torch.equal(one, many)
    # the same level twice, a level that the block size does not have, no level
    twice = (ctypes.c_int * n)(*([packs[0]] * n))
    assert lib.bsp_sdd_matmul_levels(*args(one), n, twice, *arrays[1:], *tail) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_sdd_matmul_levels(*args(one), 1, (ctypes.c_int * 1)(8), *arrays[1:], *tail) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_sdd_matmul_levels(*args(one), 0, *arrays, *tail) < 0


@pytest.mark.parametrize('block,dtype', [(16, torch.float32), (32, torch.float32), (32, torch.bfloat16), (64, torch.float32), (64, torch.float16), (128, torch.float32)])
@pytest.mark.parametrize('K', [784, 1600, 3120])
def test_few_blocks_over_a_long_reduction_run_in_parts(block, dtype, K):
    # 784: the first reductions that are cut at fp32; 3120 = 97.5 steps of 32: the last part is shorter, and half a step is past the end
    n = 4 if block < 128 else 2
    lay = torch.zeros(2, n, n, dtype=torch.int64)
    lay[0, :2, :2] = 1
    lay[:, n - 1, 1] = 1
    lay[1, 0, 0] = 1
    lib = _lib.load()
    for ta, tb_, Z in ((True, False, 1), (False, True, 2)):
        for rep in range(2):
            run_matmul_case('sdd', ta, tb_, block, dtype, Z=Z, H=2, M=n * block, N=n * block, K=K, layout=lay, dist='randn', scale=K ** -0.5, seed=K, backward=False)
    packs, n_groups = (ctypes.c_int * 1)(1), (ctypes.c_int64 * 1)(7)
    parts = lib.bsp_sdd_parts(_lib.DTYPES[dtype], block, 1, packs, n_groups, 1, K, 0)
    steps = -(-K // (16 if dtype == torch.float32 else 32))
    assert (parts > 1) == (steps >= (48 if dtype == torch.float32 else 96)) and (parts - 1) * -(-steps // parts) < steps
    assert lib.bsp_sdd_parts(_lib.DTYPES[dtype], block, 1, packs, n_groups, 1, K, _lib.FLAG_WHOLE_K) == 1


def test_parts_give_the_same_bits_every_time_and_refuse_a_small_workspace():
    torch.manual_seed(3)
    lay = _layout(32, 'all')
    luts, _, widths, packs = _sparse_matmul.make_sdd_lut(lay, 32, torch.float32, torch.device(DEV))
    K, nnz = 2000, int(lay.sum())
    a, b = torch.randn(2, 2, K, 256, device=DEV), torch.randn(2, 2, K, 256, device=DEV)
    lib, n, null, st = _lib.load(), len(luts), ctypes.c_void_p(0), _lib.stream_ptr(torch.device(DEV))
    valid = [getattr(t, 'valid', None) for t in luts]
    arrays = ((ctypes.c_int * n)(*packs), (ctypes.c_void_p * n)(*[t.data_ptr() for t in luts]),
              (ctypes.c_void_p * n)(*[None if v is None else v.data_ptr() for v in valid]), (ctypes.c_int64 * n)(*widths))

    def run(parts, ws_bytes=None):
        c = torch.full((2, nnz, 32, 32), float('nan'), device=DEV)
        need = lib.bsp_sdd_parts_workspace_bytes(32, nnz, 2, parts)
        ws = torch.full((max(need, 16),), 255, dtype=torch.uint8, device=DEV)         # (not a number, read as floats)
        rc = lib.bsp_sdd_matmul_levels(_lib.F32, _lib.ptr(a), _lib.ptr(b), _lib.ptr(c), 1, 0, 2, K, a.stride(0), a.stride(1), 256, b.stride(0), b.stride(1), 256,
                                       c.stride(0), 32, n, *arrays, null, 0, 0, parts, nnz, _lib.ptr(ws), need if ws_bytes is None else ws_bytes, 0, st)
        torch.cuda.synchronize()
        return rc, c

    rc, one = run(1)
    assert rc == _lib.OK
    for parts in (2, 5, 16):
        rc, c = run(parts)
        again = run(parts)[1]
        bound = 1e-5 * (a.abs().transpose(2, 3) @ b.abs()).max()
        assert rc == _lib.OK and torch.equal(c, again) and float((c - one).abs().max()) <= float(bound)
    assert run(4, 1024)[0] == _lib.ERR_CAPACITY
    assert run(126)[0] < 0 and run(125)[0] == _lib.OK                                 # (125 steps: 126 parts would leave one empty)


@pytest.mark.parametrize('block,dtype', [(32, torch.float32), (64, torch.float16), (128, torch.float16)])
@pytest.mark.parametrize('threads', [False, True])
def test_one_operator_on_two_streams_and_in_two_threads(block, dtype, threads):
    # products in parts, with nothing between the streams (threads: two of them on one stream): the bits of one call after the other
    lay = torch.zeros(1, 4, 4, dtype=torch.int64)
    lay[0, :2, :2] = lay[0, 3, 1:] = 1
    K, reps = 4096, 40
    torch.manual_seed(block)
    op = tb.MatMul(lay, block, 'sdd', trans_a=True)
    sets = [[torch.randn(1, 1, K, 4 * block, device=DEV).to(dtype) for _ in range(2)] for _ in range(2)]
    want = [op(*s) for s in sets]
    assert not torch.equal(*want)
    torch.cuda.synchronize()
    got = [[], []]
    if threads:
        def work(i):
            got[i] = [op(*sets[i]) for _ in range(reps)]
        both = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in both:
            t.start()
        for t in both:
            t.join()
    else:
        streams = [torch.cuda.Stream() for _ in range(2)]
        for _ in range(reps):
            for i in range(2):
                with torch.cuda.stream(streams[i]):
                    got[i].append(op(*sets[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == reps and all(torch.equal(c, want[i]) for c in got[i])


def test_a_longer_reduction_leaves_no_memory_behind():
    lin = tb.Linear(1280, 1280, 64, torch.ones(1, 20, 20, dtype=torch.int64)).to(DEV)
    held = []
    for tokens in (768, 1536, 6144, 24576):
        x = torch.randn(tokens, 1280, device=DEV, requires_grad=True)
        dw = torch.autograd.grad(lin(x), lin.weight, torch.ones(tokens, 1280, device=DEV))[0]
        del x, dw
        torch.cuda.synchronize()
        held.append(torch.cuda.memory_allocated())
    assert held == held[:1] * len(held)
