"""GPU: the dsd / dds kernel that works from chunks with lists of blocks (block 32, fp16 / bf16): against the general kernel in every
orientation, lines that do not fill a group, empty lines and groups, chunks of one block and of 24, ragged free dimensions; and the rule
that brings it into a product."""
import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib, matmul
from torch_blocksparse.matmul import GroupPlan, _sparse_matmul
from helpers import Guarded, assert_close, guard_allocations, random_layout

DEV = 'cuda'


def _layout(kind):
    if kind == 'one block':
        lay = torch.zeros(1, 3, 2, dtype=torch.int64)
        lay[0, 2, 1] = 1
        return lay
    if kind == 'full':                                    # one reduction block a chunk
        return torch.ones(2, 18, 33, dtype=torch.int64)
    lay = random_layout((2, 21, 37), 0.3, 5)              # a second group of five lines, a third of rows that are columns
    lay[1, 16:] = 0
    lay[0, :, 3] = 0
    return lay


@pytest.mark.parametrize('kind', ['one block', 'full', 'ragged'])
@pytest.mark.parametrize('rows', [False, True])
def test_chunks_hold_the_layout(kind, rows):
    lay = _layout(kind)
    H, R, C = lay.shape
    plan = GroupPlan.build_xsd_chunks(lay, rows, torch.device('cpu'), always=True)
    L = R if rows else C
    assert plan.n_groups == H * -(-L // 16) and plan.lines == L
    ids = torch.full(lay.shape, -1)
    ids[lay != 0] = torch.arange(int(lay.sum()))
    seen = torch.full(lay.shape, -1)
    heads, records = plan.table[:4 * plan.n_groups].view(-1, 4), plan.table[4 * plan.n_groups:].view(-1, 32)
    for h, line0, first, n in heads.tolist():
        last = -1
        for r in records[first:first + n].tolist():
            assert n == 1 if not r[0] else r[0] <= 4 and 1 <= r[1] <= 24 and r[4] > last
            last, at = r[3 + r[0]], 8                       # (an empty group: one record of zeros)
            for bit in range(64):
                if (r[2 + bit // 32] >> bit % 32) & 1:
                    l, k = line0 + bit // 4, r[4 + bit % 4]
                    seen[(h, l, k) if rows else (h, k, l)] = r[at]
                    at += 1
            assert at == 8 + r[1]
    assert torch.equal(seen, ids)


def _against_the_general_kernel(lay, dtype, N, Z, once=False):
    """every orientation from chunks, between guard bands, against the general kernel"""
    H, R, C = lay.shape
    dev, nnz = torch.device(DEV), int(lay.sum())
    lib, st = _lib.load(), _lib.stream_ptr(dev)
    torch.manual_seed(N)
    sp = torch.randn(Z, nnz, 32, 32, device=DEV).to(dtype)
    for dds in (False, True):
        for tsp in (0, 1):                                # the sparse operand transposed
            lines_are_rows = bool(tsp) if dds else not tsp
            L, K = (R, C) if lines_are_rows else (C, R)
            lut, _, width, _ = _sparse_matmul.make_dxx_lut(lay, 32, 16, lines_are_rows, dev)
            chunks = GroupPlan.build_xsd_chunks(lay, lines_are_rows, dev, always=True)
            for tdn in (0, 1):
                for tc in (0, 1):
                    # dense operand: dsd K x N, dds N x K
                    flip = bool(tdn) != dds
                    out_n_last = bool(tc) == dds
                    if N % 8 and (not flip or out_n_last):  # (such a free dimension lies along whole rows on both sides)
                        continue
                    dn = torch.randn((Z, H) + ((N, K * 32) if flip else (K * 32, N)), device=DEV).to(dtype) * K ** -0.5
                    shape = (Z, H) + ((L * 32, N) if out_n_last else (N, L * 32))
                    ref, out = torch.full(shape, float('nan'), device=DEV, dtype=dtype), Guarded(shape, dtype, fill=float('nan'))
                    got, what = out.t, 'chunks dds=%d tsp=%d tdn=%d tc=%d' % (dds, tsp, tdn, tc)

                    def call(c, plan, flags):
                        strides = (dn.stride(0), dn.stride(1), dn.stride(2))
                        tail = (c.stride(0), c.stride(1), c.stride(2), 32, _lib.ptr(lut), _lib.ptr(lut.planbuf), width, _lib.ptr(plan.table) if plan else None,
                                plan.n_groups if plan else 0, plan.lines if plan else 0, 0, None, 0, flags, st)
                        if dds:
                            return lib.bsp_dds_matmul(_lib.DTYPES[dtype], _lib.ptr(dn), _lib.ptr(sp), _lib.ptr(c), tdn, tsp, tc, Z, N, *strides, sp.stride(0), *tail)
                        return lib.bsp_dsd_matmul(_lib.DTYPES[dtype], _lib.ptr(sp), _lib.ptr(dn), _lib.ptr(c), tsp, tdn, tc, Z, N, sp.stride(0), *strides, *tail)

                    assert call(ref, None, _lib.FLAG_GENERAL_ONLY) == _lib.OK
                    assert call(got, chunks, _lib.FLAG_PLAN_TILES) == _lib.OK
                    out.check(what)
                    assert_close(got, ref, dtype, what)
                    if once:
                        continue
                    got.fill_(float('nan'))               # a product that they do not serve runs from its table
                    assert call(got, chunks, _lib.FLAG_PLAN_TILES | _lib.FLAG_GENERAL_ONLY) == _lib.OK
                    out.check(what)
                    assert torch.equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['one block', 'full', 'ragged'])
@pytest.mark.parametrize('dtype,N', [(torch.float16, 256), (torch.bfloat16, 136), (torch.float16, 392), (torch.float16, 257), (torch.bfloat16, 999)])
def test_chunks_against_the_general_kernel(kind, dtype, N):
    _against_the_general_kernel(_layout(kind), dtype, N, Z=2)


@pytest.mark.gpu
@pytest.mark.parametrize('kind,Z', [('one block', 300), ('ragged', 75)])
@pytest.mark.parametrize('dtype,N', [(torch.float16, 256), (torch.bfloat16, 256), (torch.bfloat16, 136), (torch.float16, 257)])
def test_workgroups_that_take_several_tiles(kind, Z, dtype, N):
    # 600 tiles and more for 256 workgroups: a tile's first chunk is on its way during the stores of the one before; whole tiles and partial
    # ones (lines and columns past the end), tiles of one chunk, tiles without blocks between others
    lay = _layout(kind)
    assert lay.shape[0] * -(-min(lay.shape[1:]) // 16) * -(-N // 128) * Z >= 600
    _against_the_general_kernel(lay, dtype, N, Z, once=True)


@pytest.mark.gpu
@pytest.mark.parametrize('lists', [True, False])
@pytest.mark.parametrize('M,Z', [(257, 16), (999, 8)])
def test_rows_that_divide_by_nothing_on_the_wide_kernels(M, Z, lists, monkeypatch):
    # y = x W and dx = dy W^T with M rows, from chunks and from groups of four lines
    if not lists:
        monkeypatch.setattr(GroupPlan, 'build_xsd_chunks', staticmethod(lambda *args, **kw: None))
    lay = random_layout((1, 48, 48), 0.3, 3)
    assert 48 // 4 * -(-M // 256) * Z >= 384                 # the launches that take the wide kernels
    op = tb.MatMul(lay, 32, 'dds')
    torch.manual_seed(M)
    x, dy = [torch.randn(Z, 1, M, 48 * 32, device=DEV).half() for _ in range(2)]
    w = torch.randn(Z, int(lay.sum()), 32, 32, device=DEV).half() / 16
    x.requires_grad_(True)

    def both():
        y = op(x, w)
        return y.detach(), torch.autograd.grad(y, x, dy)[0]

    with guard_allocations('wide'):
        got = both()
    luts = op.make_lut(torch.float16, x.device)
    assert [t.gplan_wide.flags for t in (luts[0], luts[4])] == [_lib.FLAG_PLAN_TILES if lists else 0] * 2
    monkeypatch.setattr(matmul, 'KERNEL_FLAGS', _lib.FLAG_GENERAL_ONLY)
    for one, two, what in zip(got, both(), ('y', 'dx')):
        assert_close(one, two, torch.float16, what)


@pytest.mark.gpu
def test_a_product_takes_them_at_its_densities(monkeypatch):
    torch.manual_seed(2)
    b = torch.randn(8, 8, 1024, 256, device=DEV).half()      # 512 workgroups of the wide kernels
    for density, rows, taken in ((0.25, 32, True), (0.6, 32, False), (0.08, 32, False), (0.25, 25, False)):
        lay = random_layout((8, rows, 32), density, 3)
        op = tb.MatMul(lay, 32, 'dsd')
        a = torch.randn(8, int(lay.sum()), 32, 32, device=DEV).half() / 16
        wide = GroupPlan.build_xsd_chunks(lay, True, b.device)
        assert (wide is not None) == taken
        with guard_allocations('dsd'):
            got, again = op(a, b), op(a, b)
        monkeypatch.setattr(matmul, 'KERNEL_FLAGS', _lib.FLAG_GENERAL_ONLY)
        assert_close(got, op(a, b), torch.float16, 'dsd')
        monkeypatch.undo()
        assert torch.equal(got, again)
        lut = op.make_lut(torch.float16, b.device)[0]
        assert taken == (lut.gplan_wide is not None and lut.gplan_wide.flags == _lib.FLAG_PLAN_TILES)
