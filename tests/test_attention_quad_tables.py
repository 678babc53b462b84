"""CPU: the tables of the attention kernels without sparse tensors (bsp_attention_tables_build, host code of the library)."""
import ctypes

import pytest
import torch

from torch_blocksparse import _lib
from torch_blocksparse.attention_core import AttentionCore, _ColumnTable, _QuadTables, _stored_tables


@pytest.mark.parametrize('block,H,R,C,density,dtype', [
    (64, 1, 1, 1, 1.0, torch.int64), (64, 5, 6, 9, 0.4, torch.int32), (64, 2, 70, 5, 0.5, torch.int64), (64, 9, 40, 40, 0.1, torch.bool),
    (32, 2, 8, 12, 0.3, torch.int64), (32, 3, 80, 6, 0.2, torch.int32), (16, 2, 12, 20, 0.1, torch.int64), (16, 5, 160, 8, 0.3, torch.bool)])
def test_tiles_cover_the_layout_once_in_both_views(block, H, R, C, density, dtype):
    torch.manual_seed(R * C + block)
    lay = torch.rand(H, R, C) < density
    lay[:, :, 0] = True                                  # a long column
    lay[0, R // 2] = False                               # an empty block-row in one head
    lay[H - 1, :, C - 1] = False                         # and an empty block-column
    S = 64 // block
    t = _QuadTables(lay.to(dtype), block, 'cpu')
    rows, items, split = t.rows.tolist(), t.items.tolist(), t.split.tolist() if t.n_split else []
    full = lay.repeat_interleave(block, 1).repeat_interleave(block, 2)
    assert t.lines == R // S and t.columns == C // S
    got = torch.zeros(full.shape, dtype=torch.int32)
    longest = 0
    for h in range(H):
        for line in range(t.lines):
            n, first = rows[2 * (h * t.lines + line):2 * (h * t.lines + line) + 2]
            longest = max(longest, n)
            for e in range(n):
                entry = rows[first + 8 * e:first + 8 * e + 8]
                assert all(0 <= p <= C * block - 16 and p % 16 == 0 for p in entry[:4]) and entry[5:] == [0, 0, 0] and entry[4]
                for piece in range(16):
                    if entry[4] >> piece & 1:
                        r, c = 64 * line + 16 * (piece // 4), entry[piece % 4]
                        got[h, r:r + 16, c:c + 16] += 1
    assert torch.equal(got, full.int()) and longest == t.longest
    got.zero_()
    slots, parts, keys_of = [], {}, {}
    for i in range(t.n_items):
        n, first, h, col, slot = items[12 * i:12 * i + 5]
        keys = items[12 * i + 8:12 * i + 12]
        assert items[12 * i + 5:12 * i + 8] == [0, 0, 0] and keys_of.setdefault((h, col), keys) == keys
        parts.setdefault((h, col), []).append((slot, n))
        slots += [slot] if slot >= 0 else []
        for e in range(n):
            entry = items[first + 8 * e:first + 8 * e + 8]
            assert all(0 <= p <= R * block - 16 and p % 16 == 0 for p in entry[:4]) and entry[4]
            for piece in range(16):
                if entry[4] >> piece & 1:
                    r, c = entry[piece // 4], keys[piece % 4]
                    got[h, r:r + 16, c:c + 16] += 1
    assert torch.equal(got, full.int())
    for h in range(H):                                   # the columns of a head partition its keys
        assert sorted(p for (hh, _), keys in keys_of.items() if hh == h for p in keys) == list(range(0, C * block, 16))
    assert sorted(slots) == list(range(t.n_slots))
    for i in range(t.n_split):
        h, col, first, n = split[8 * i:8 * i + 4]
        assert split[8 * i + 4:8 * i + 8] == keys_of[(h, col)]
        assert sorted(s for s, _ in parts[(h, col)]) == list(range(first, first + n)) and n > 1
        sizes = [c for _, c in parts[(h, col)]]
        assert max(sizes) - min(sizes) <= 1
    assert sum(len(p) > 1 for p in parts.values()) == t.n_split
    lengths = [items[12 * i] for i in range(t.n_items)]  # four heads at a time, the longest items first
    groups = [items[12 * i + 2] // 4 for i in range(t.n_items)]
    assert groups == sorted(groups) and all(a >= b for a, b, ga, gb in zip(lengths, lengths[1:], groups, groups[1:]) if ga == gb)
    ids = torch.full(lay.shape, -1, dtype=torch.int64)
    ids[lay] = torch.arange(int(lay.sum()))
    old = _ColumnTable(lay.long(), 'cpu', S=S, ids=ids)  # the same columns and parts as the kernels that read p take
    assert (old.n_items, old.n_slots, old.n_split) == (t.n_items, t.n_slots, t.n_split)


def test_errors():
    lib, info = _lib.load(), _lib.AttentionTables()
    lay, out = torch.ones(1, 4, 4, dtype=torch.bool), torch.empty(16, dtype=torch.int32)
    build = lambda lay, R, block, cap: lib.bsp_attention_tables_build(_lib.ptr(lay), 1, R, 4, block, _lib.ptr(out), cap, ctypes.byref(info))
    assert build(lay, 4, 64, 16) == _lib.ERR_CAPACITY and info.total > 16
    assert build(lay, 3, 16, 16) == _lib.ERR_UNSUPPORTED
    assert build(lay, 4, 128, 16) == _lib.ERR_UNSUPPORTED
    assert build(None, 4, 64, 16) != _lib.OK


@pytest.mark.parametrize('block,H,R,C', [(64, 3, 7, 70), (32, 2, 8, 10), (16, 2, 8, 7)])
def test_tables_of_the_kernels_that_store_p(block, H, R, C):
    """the rows' part (the softmax table at blocks of 64, tiles with the ids of their blocks below), made beside the other set by
    whichever call comes first; a layout whose columns do not divide into tiles gets no columns"""
    torch.manual_seed(C)
    lay = (torch.rand(H, R, C) < 0.3).long()
    lay[0, 1] = 0
    S = 64 // block
    host, info = _stored_tables(lay, block)
    assert info.lines == R // S and info.columns == (0 if C % S else C // S) and info.longest_line == max(
        -(-int(n) // S) for n in (lay.reshape(H, R // S, S, C).sum(2) > 0).sum(-1).flatten())
    seen = {}
    for h in range(H):
        for line in range(R // S):
            n, first = host[2 * (h * (R // S) + line):][:2].tolist()
            for e in range(n):
                if S == 1:
                    bid, c, r, hh = host[first + 4 * e:][:4].tolist()
                    assert (r, hh) == (line, h)
                    seen[bid] = (h, r, c)
                else:
                    entry = host[first + (8 + S * S) * e:][:8 + S * S].tolist()
                    for i, bid in enumerate(entry[8:]):
                        if bid >= 0:
                            seen[bid] = (h, S * line + i // S, entry[4 + i % S])
    assert [list(seen[i]) for i in range(len(seen))] == lay.nonzero().tolist()
    core = AttentionCore(lay, block)
    if C % S:
        assert core.tables('cpu') is None and core.quad('cpu') is None
    else:
        assert torch.equal(core.tables('cpu')[0], host) and core.quad('cpu').lines == R // S
    odd = ctypes.c_int64(0)
    assert _lib.load().bsp_attention_stored_tables_build(_lib.ptr(lay.bool()), None, H, R, C, block, 0, ctypes.byref(odd), 1, ctypes.byref(info)) == _lib.ERR_CAPACITY
    assert info.total == host.numel()


@pytest.mark.parametrize('block,H,R,C,density', [(64, 2, 6, 9, 0.4), (32, 3, 8, 12, 0.3), (16, 2, 16, 8, 0.1)])
def test_counts_that_fp32_calls_are_routed_by(block, H, R, C, density):
    """tiles and pieces as the tables have them, also in operators saved before these were kept"""
    torch.manual_seed(block)
    lay = torch.rand(H, R, C) < density
    core = AttentionCore(lay, block)
    t = core.quad('cpu')
    rows = t.rows.tolist()
    lines = [(rows[2 * i], rows[2 * i + 1]) for i in range(H * t.lines)]
    assert t.tiles == sum(n for n, _ in lines)
    assert t.pieces == sum(bin(rows[first + 8 * e + 4] & 0xffff).count('1') for n, first in lines for e in range(n))
    kept = t.tiles, t.pieces
    del t.tiles, t.pieces
    again = AttentionCore.__new__(AttentionCore)
    again.__setstate__(core.__dict__)
    assert (again.quad('cpu').tiles, again.quad('cpu').pieces) == kept


def test_fp32_calls_take_the_faster_way():
    def pays(lay, block, Z, D, backward=True):
        return _QuadTables(lay, block, 'cpu').pays_f32(Z, D, backward)
    dense, diagonal = torch.ones(8, 32, 32, dtype=torch.int64), torch.eye(64, dtype=torch.int64).expand(16, 64, 64)
    few = (torch.rand((8, 128, 128), generator=torch.Generator().manual_seed(1)) < 0.05).long() | torch.eye(128, dtype=torch.int64)
    for D in (64, 128):
        assert pays(dense, 64, 2, D) and pays(dense, 64, 2, D, False)
        assert not pays(diagonal, 64, 4, D) and not pays(few, 16, 2, D)
    assert pays(dense[:, :8, :8], 64, 1, 64, False) and pays(dense[:, :3, :3], 64, 1, 128, True)
    assert not pays(dense[:, :3, :3], 64, 1, 128, False)
