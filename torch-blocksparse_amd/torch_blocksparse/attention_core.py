"""The chain scores -> softmax -> context of the attention modules, in one launch per direction where that is possible.

The reference's modules call three operators, sparse_dot_sdd_nt(q, k), sparse_softmax(...), sparse_dot_dsd_nn(p, v)
(deepspeedsparseselfattention.py:152-157; attention.py:190-202).  `attention_chain` takes the same three operator
objects and the same arguments and returns the same context tensor; when the operators are this package's, built on
one layout with blocks of 16, 32 or 64, and the tensors are fp16 / bf16 with a head dimension of 64 or 128, it runs fused
kernels instead; in fp32 it does so without relative position embedding and attention mask, for layouts that make it pay
(_QuadTables.pays_f32; bsp_attention_f32_fwd, bsp_attention_f32_bwd: class _attention_f32).  In 16 bits, without relative position embedding and attention mask no sparse tensor exists (bsp_attention_rows_fwd,
bsp_attention_rows_bwd, bsp_attention_cols_bwd: class _attention_quad); with one of them the softmax is stored for the backward pass
(bsp_attention_fwd, bsp_attention_bwd, bsp_attention_bwd_kv: class _attention_core).
In every other case, and with FUSED = False, it calls the three operators one after the other.
"""
import ctypes
import os

import torch

from . import _lib
from .matmul import MatMul
from .softmax import Softmax, _sparse_softmax

FUSED = os.environ.get('BSP_FUSED_ATTENTION', '1') != '0'
MAX_ROW_BLOCKS = 8          # BSP_ATTENTION_MAX_ROW_BLOCKS: longer rows are streamed (the library decides)
fused_calls = 0             # forward calls that took the fused kernels for 16-bit tensors; tests read it
fused_f32_calls = 0         # ... and those for fp32
# dk and dv from a column kernel (bsp_attention_cols_bwd, bsp_attention_bwd_kv), which computes the softmax gradient again instead
# of reading it; False: the row kernel stores the gradient and the two products are ordinary dsd operators
FUSED_KV = os.environ.get('BSP_FUSED_ATTENTION_KV', '1') != '0'


def _stored_tables(layout, block, ids=None, part=0):
    """(tables, sizes): the tables of the kernels that store p, in host memory (bsp_attention_stored_tables_build)"""
    lay = (layout != 0).cpu().contiguous()
    H, R, C = lay.shape
    S = 64 // block
    info = _lib.AttentionTables()
    cap = 2 * H * R + 20 * H * C + (20 if S == 1 else 28 + 2 * S * S) * int(torch.count_nonzero(lay))
    host = torch.empty(max(cap, 1), dtype=torch.int32)
    ids = None if ids is None else ids.to(torch.int32).contiguous()
    _lib.check(_lib.load().bsp_attention_stored_tables_build(_lib.ptr(lay), _lib.ptr(ids), H, R, C, block, part, _lib.ptr(host), cap,
                                                             ctypes.byref(info)), 'bsp_attention_stored_tables_build')
    return host[:info.total], info


class _GatheredTiles:
    """64 x 64 tiles over a layout of small blocks (S = 64 / block a side).  A *line* of tiles is S consecutive block-rows;
    a tile takes the line's S block-rows and S block-columns gathered from anywhere in the line: the columns in which
    any of the line's block-rows holds a block, in ascending order, S per tile.  (Tiles cut from a fixed grid would be
    mostly holes wherever the layout has single block-columns, like the global columns of the 'fixed' layouts: a
    kernel that works on whole tiles then does S times the work.)
    sizes / starts: tiles per line and the line's first tile, lines in (head, line) order; cols [tiles, S]: the
    block-columns of a tile (slots past the end of a line repeat the tile's first column); ids [tiles, S, S]: the id of
    the block at (block-row i of the line, gathered column g), -1 where the layout has none or the slot is padding."""

    def __init__(self, lay, ids, S):
        host, info = _stored_tables(lay, 64 // S, ids)
        self.lines, self.heads = info.lines, lay.size(0)
        n, ints = self.lines * self.heads, 8 + S * S
        self.sizes = host[0:2 * n:2].long()
        self.starts = (host[1:2 * n:2].long() - 2 * n) // ints
        self._entries = host[2 * n:info.items_offset].reshape(-1, ints).long()
        self.n_tiles = self._entries.size(0)
        self.cols = self._entries[:, 4:4 + S]
        self.ids = self._entries[:, 8:].reshape(-1, S, S)

    def entries(self):
        """per tile 8 + S * S ints: (tile, 0, line, head, then the tile's block-columns, the last repeated up to four, then
        the ids of its blocks, [block-row of the line][gathered block-column])"""
        return self._entries


class _ColumnTable:
    """The tables of the column kernel: the layout read along columns, cut into work items.
    items: per item twelve ints (entries, offset of its entries, head, column, slot of its partial sums or -1, 0, 0, 0, then
    the column's block-columns, the last repeated up to four), then the entries, a column's by row.  Blocks of 64: a
    column is a block-column, an entry (id, row, column, head); the ids are the positions in the row-major order of the
    nonzero blocks, as everywhere.  Smaller blocks: a column is S block-columns whose blocks lie in the same block-rows as
    far as possible, so that the block-rows gathered into a tile hold blocks in most of them (the long ones of a head
    together, longest first, the others as they lie: neighbours share their rows in banded layouts), its entries the tiles
    of _GatheredTiles over the transposed layout (S block-rows gathered per tile): 8 + S * S ints, the last S * S the ids
    of the tile's blocks, [gathered block-row][block-column of the group].  A column of more than `part` entries (None: 16
    and twice the average, every part costs a slot written and read) is cut into parts of near-equal size, each with a slot;
    split: per such column eight ints (head, column, first slot, parts, then its block-columns)."""

    def __init__(self, layout, device, part=None, S=1, ids=None):
        self._take(*_stored_tables(layout, 64 // S, ids, part or 0), device)

    def _take(self, host, info, device):
        """the columns' part of the tables, in one piece on `device`; -> all of it there"""
        tables = host.to(device)
        self.items = tables[info.items_offset:info.split_offset]
        self.split = tables[info.split_offset:] if info.n_split else None
        self.columns, self.n_items, self.n_slots, self.n_split = info.columns, info.n_items, info.n_slots, info.n_split
        return tables


class _QuadTables:
    """The tables of the kernels without sparse tensors (bsp_attention_tables_build), made on the host in one call and copied
    to `device` in one piece: rows (forward and row kernel), items and split (column kernel), and their sizes."""
    _native = None

    def __init__(self, layout, block, device):
        lay = (layout != 0).cpu().contiguous()
        H, R, C = lay.shape
        lib = _lib.load()
        info = _lib.AttentionTables()
        blocks = int(torch.count_nonzero(lay))
        cap = 32 * H * (R + C) + 16 * blocks + 64
        host = torch.empty(cap, dtype=torch.int32)
        _lib.check(lib.bsp_attention_tables_build(_lib.ptr(lay), H, R, C, block, _lib.ptr(host), cap, ctypes.byref(info)),
                   'bsp_attention_tables_build')
        self.rows = host[:info.total].to(device)
        self.items = self.rows[info.items_offset:]
        self.split = self.rows[info.split_offset:] if info.n_split else None
        self.lines, self.longest, self.columns = info.lines, info.longest_line, info.columns
        self.n_items, self.n_slots, self.n_split = info.n_items, info.n_slots, info.n_split
        self.shape = (H, R, C, block)
        self._count(blocks)

    def _count(self, blocks):
        """tiles of the lines (what lies between the lines' heads and the items, eight ints each), and the 16 x 16 pieces of score that have a block"""
        self.tiles = (self.rows.numel() - self.items.numel() - 2 * self.shape[0] * self.lines) // 8
        self.pieces = blocks * (self.shape[3] // 16) ** 2

    def pays_f32(self, Z, D, backward):
        """Is a call in fp32 faster here than through the three operators?  The kernels work on whole tiles and have a cost a line, the
        operators work on blocks alone.  Fitted to layouts of all kinds (random ones of a hundredth to a quarter of the blocks, fixed,
        transformer, BigBird, dense; blocks of 16 to 64; 64 to 8192 lines in the launch).  Head dimension 64, training / inference, us of operators and
        kernels: per 1000 lines 29 and 79 / 8 and 24, per 10000 pieces 35 / 11, per 1000 tiles 21 / 5.  Beside the line, training: 2048 lines of
        2.5 tiles with 12.8 pieces each 352 and 331, 4096 of 1.6 with 16 405 and 499, 4096 of 13 with 4.2 1040 and 1539, 512 of 23 with 5.8 306
        and 337, of 15 with 9.0 286 and 261.  Head dimension 128, one workgroup a compute unit: 512 lines of 6 tiles with 16 pieces 347 and 395, of 10
        with 15.2 452 and 396, 2048 of 3 with 16 667 and 953, of 6 with 16 1131 and 1098, 8192 of 4 with 16 3247 and 3423; the operators take longer
        over blocks of 16 (2048 lines of 5.2 with 13.7: 1542 and 1063).  A short training pass waits for the host, which makes five launches
        for eleven: 64 lines of 3 tiles with head dimension 128 163 and 127, 512 lines of 2.6 with 64, 3.5 pieces a tile, 172 and 125."""
        lines, tiles, pieces = [Z * n for n in (self.shape[0] * self.lines, self.tiles, self.pieces)]
        if D == 64:
            return (backward and tiles + 4 * lines <= 4000) or pieces > 6 * tiles + 20 * lines - 8000
        return (backward and lines <= 128) or pieces * (1.1 if self.shape[3] == 16 else 1.) > 12 * tiles + 10 * lines + 7000

    def __getstate__(self):
        return {k: v for k, v in self.__dict__.items() if k != '_native'}

    def native(self):
        """what the native launcher (csrc/launch.cpp) wants to know of the tables, made once"""
        if self._native is None:
            dev = self.rows.device.index if self.rows.device.index is not None else torch.cuda.current_device()
            self._native = _lib.native().make_attn(self.rows, self.rows.data_ptr(), self.items.data_ptr(), 0 if self.split is None else self.split.data_ptr(), self.lines,
                                                   self.columns, self.n_items, self.n_slots, self.n_split, dev, self.longest, *self.shape)
        return self._native


def _vec_ok(t):
    """16-byte vector accesses of a 4-dimensional tensor: unit inner stride, every other stride a multiple of 8 elements, aligned
    base, rows that do not overlap (a gradient expanded along the positions has rows 0 apart)."""
    z, h, row, inner = t.stride()
    return inner == 1 and not (z | h | row) % 8 and row >= t.size(3) and not t.data_ptr() % 16


def _packed(t):
    """a copy in storage of its own (contiguous() returns a tensor at an odd address, or of batch size 1 with an odd stride, as it is)"""
    return t.clone(memory_format=torch.contiguous_format)


def _vec(t):
    return t if _vec_ok(t) else _packed(t)


def _near(t):
    """... and the rows of a head within 4 GiB of its first, as the kernels without sparse tensors address them"""
    return t if _vec_ok(t) and t.stride(2) * t.size(2) * t.element_size() < 2 ** 32 else _packed(t)


class AttentionCore:
    """What the fused kernels need beside the tensors: the tables of the layout's 64 x 64 tiles along lines of rows and along
    columns, for the kernels without sparse tensors and for those that store the softmax, and the two products that are
    ordinary operators in the backward pass when the column kernel is not used (dv = p^T . do and dk = ds^T . q)."""

    def __init__(self, layout, block):
        self.layout = layout
        self.block = block
        self.spdims = tuple(layout.shape)
        self.dsd_tn = MatMul(layout, block, 'dsd', trans_a=True, trans_b=False)
        self.nnz = None
        self._tables = dict()

    def __setstate__(self, state):
        self.__dict__.update(state)
        for quad, _ in self._tables.values():              # (saved before the tables kept their shape, or their counts)
            if quad is not None and not hasattr(quad, 'shape'):
                quad.shape = tuple(int(n) for n in self.spdims) + (self.block,)
            if quad is not None and not hasattr(quad, 'pieces'):
                quad._count(self.blocks())

    def blocks(self):
        if self.nnz is None:
            self.nnz = int((self.layout != 0).sum())
        return self.nnz

    def quad(self, device):
        """the tables of the kernels without sparse tensors on `device`, or None when the layout does not divide into tiles"""
        return (self._tables.get(str(device)) or self._made(device))[0]

    def tables(self, device):
        """(table, longest row, None, rows of the table's layout, present blocks per present tile as a share,
        tables of the column kernel) on `device`, or None when the layout does not divide into 64 x 64 tiles: what the kernels
        that store p need"""
        return (self._tables.get(str(device)) or self._made(device))[1]

    def _made(self, device):
        """Both sets of tables: a call with per-element masks and one without need different ones, and either may be the one
        that is captured after a warm-up step of the other kind."""
        S = 64 // self.block
        H, R, C = self.spdims
        made = (None, None)
        if not (R % S or C % S):
            lay = (self.layout != 0).cpu().contiguous()
            self.nnz = int(torch.count_nonzero(lay))
            host, info = _stored_tables(lay, self.block)
            columns = _ColumnTable.__new__(_ColumnTable)
            lut = columns._take(host, info, device)
            n_tiles = (info.items_offset - 2 * H * info.lines) // (4 if S == 1 else 8 + S * S)
            made = (_QuadTables(lay, self.block, device),
                    (lut, info.longest_line, None, info.lines, self.blocks() / max(1, n_tiles * S * S), columns))
        self._tables[str(device)] = made
        return made

    def usable(self, q, k, v, dropout_p=0.):
        """Can this call take the fused kernels?  (Shapes that do not fit the layout are left to the operators, which
        raise the reference's errors.)"""
        if not FUSED or self.block not in (16, 32, 64) or dropout_p:
            return False
        tables = self._tables.get(str(q.device)) if q.is_cuda else None
        if tables is not None and tables[0] is not None:
            usable = _lib.native().attn_usable(tables[0].native(), q, k, v)
            if usable is not None:
                return usable
        if not (q.is_cuda and q.dtype in (torch.float16, torch.bfloat16) and self._fits(q, k, v)):
            return False
        t = self.quad(q.device)
        if t is None or t.longest <= 0:
            return False
        return t.longest * 64 < 32768                           # the softmax operator's bound on a row (softmax.py:225-227)

    def _fits(self, q, k, v):
        """three operands of one type that fit the layout, of a head dimension that there are kernels for"""
        if k.dtype != q.dtype or v.dtype != q.dtype or q.dim() != 4 or k.dim() != 4 or v.dim() != 4 or q.size(3) not in (64, 128):
            return False
        H, R, C = self.spdims
        Z, D, b = q.size(0), q.size(3), self.block
        return tuple(q.shape) == (Z, H, R * b, D) and tuple(k.shape) == (Z, H, C * b, D) and tuple(v.shape) == (Z, H, C * b, D)

    def usable_f32(self, q, k, v, rpe=None, attn_mask=None, dropout_p=0.):
        """The same for fp32: calls without per-element masks, where the kernels are faster.  FUSED_KV = False asks for the gradients through
        stored softmax gradients, which only the operators have here."""
        if not (FUSED and FUSED_KV) or rpe is not None or attn_mask is not None or dropout_p or self.block not in (16, 32, 64) or not q.is_cuda:
            return False
        if str(q.device) not in self._tables and not self._fits(q, k, v):
            return False                                        # (no tables for calls that never use them)
        tables = self.quad(q.device)
        if tables is None or _lib.native().attn_usable(tables.native(), q, k, v) is not True:
            return False
        return tables.pays_f32(q.size(0), q.size(3), torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad))

    def __call__(self, q, k, v, scale=1., rpe=None, key_padding_mask=None, attn_mask=None,
                 key_padding_mask_mode='add', attn_mask_mode='add'):
        for name, m in (('relative position embedding', rpe), ('Attention mask', attn_mask), ('Key padding mask', key_padding_mask)):
            if m is not None and m.dtype != q.dtype:      # softmax.py:348-353
                raise ValueError('%s must be %s' % (name, q.dtype))
        if rpe is None and attn_mask is None:
            if key_padding_mask is not None:
                self._check_masks(q, None, key_padding_mask, None)
            chain = _attention_f32 if q.dtype == torch.float32 else _attention_quad
            return chain.apply(q, k, v, float(scale), key_padding_mask, key_padding_mask_mode, self, torch.is_grad_enabled())
        lut, maxlut, _, rows = self.tables(q.device)[:4]
        # p is kept for the backward pass; a forward pass that no backward pass can follow does not store it
        keep_p = torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad)
        return _attention_core.apply(q, k, v, float(scale), rpe, key_padding_mask, attn_mask, key_padding_mask_mode,
                                     attn_mask_mode, self, lut, maxlut, keep_p, rows)


    def _check_masks(self, q, rpe, key_padding_mask, attn_mask):
        """the masks against the layout, exactly as the softmax operator checks them (the kernels take every address from the table)"""
        nnz, block = self.blocks(), self.block
        _sparse_softmax._check_shapes(torch.empty((q.size(0), nnz, block, block), device='meta'), rpe, key_padding_mask, attn_mask, self.spdims, block, nnz)


class _attention_quad(torch.autograd.Function):
    """The chain without per-element masks: no sparse tensor is kept for the backward pass, two floats per row are (the
    logarithm of the row's sum of exponentials, and what its rounding left out), from which the backward kernels compute
    the softmax again."""

    @staticmethod
    def forward(ctx, q, k, v, scale, key_padding_mask, kp_mask_mode, core, grad_enabled):
        global fused_calls
        H, R, C = core.spdims
        Z, D = q.size(0), q.size(3)
        tables = core.quad(q.device)
        lines = tables.lines
        keep = grad_enabled and any(ctx.needs_input_grad[:3])
        kpm = None
        if key_padding_mask is not None:                   # element (z, c), softmax.py:60-62, 274
            kpm = _sparse_softmax._strided16(key_padding_mask, 'key_padding_mask')
            if keep and kpm.data_ptr() == key_padding_mask.data_ptr():
                kpm = _packed(kpm[:, :k.size(2)])          # the backward pass reads it again, the caller may fill it with the next mask until then
        ctx.kpm_args = (kpm.stride(0) if kpm is not None and kpm.size(0) > 1 else 0, int(kp_mask_mode == 'mul'))
        launch, native = _lib.native(), tables.native()
        made = launch.attn_fwd(native, q, k, v, scale, kpm, *ctx.kpm_args, keep)
        if made is None:                                   # operands that the kernels cannot address are copied to memory of their own
            q, k, v = _near(q), _near(k), _near(v)
            made = launch.attn_fwd(native, q, k, v, scale, kpm, *ctx.kpm_args, keep)
            if made is None:
                raise _lib.BlocksparseLibraryError('attention: operands %s, %s, %s do not fit the layout' % (tuple(q.shape), tuple(k.shape), tuple(v.shape)))
        o, lse = made                                      # lse [Z, H, 2, rows]: and what its rounding left out
        fused_calls += 1
        if keep:
            ctx.save_for_backward(q, k, v, o, lse, kpm)
            ctx.core, ctx.scale, ctx.tables, ctx.kp_mask_mode = core, scale, tables, kp_mask_mode
        return o

    @staticmethod
    def rows_kernel(ctx, saved, do, delta):
        """dq, and into delta (if given) the negative of the rows' sums sum_d do . o"""
        q, k, v, o, lse, kpm = saved
        Z, H, D = q.size(0), q.size(1), q.size(3)
        dq = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        rc = _lib.load().bsp_attention_rows_bwd(
            _lib.DTYPES[q.dtype] | _lib.ROWS_WITH_REST, _lib.ptr(do), _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(o), _lib.ptr(lse), _lib.ptr(dq), _lib.ptr(delta), Z, H,
            ctx.tables.lines, k.size(2), D, do.stride(0), do.stride(1), do.stride(2), q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
            v.stride(0), v.stride(1), v.stride(2), o.stride(0), o.stride(1), o.stride(2), dq.stride(0), dq.stride(1), dq.stride(2),
            ctx.tables.lines * 128, ctx.scale, _lib.ptr(ctx.tables.rows), _lib.ptr(kpm), *ctx.kpm_args, _lib.stream_ptr(q.device))
        _lib.check(rc, 'bsp_attention_rows_bwd')
        return dq

    @staticmethod
    def columns_kernel(ctx, saved, do, delta):
        """dk and dv"""
        q, k, v, o, lse, kpm = saved
        Z, H, D = q.size(0), q.size(1), q.size(3)
        ct = ctx.tables
        dk = torch.empty(k.shape, dtype=k.dtype, device=k.device)
        dv = torch.empty(v.shape, dtype=v.dtype, device=v.device)
        partial = torch.empty((Z, ct.n_slots, 2, 64, D), dtype=torch.float32, device=q.device) if ct.n_slots else None
        rc = _lib.load().bsp_attention_cols_bwd(
            _lib.DTYPES[q.dtype] | _lib.ROWS_WITH_REST, _lib.ptr(do), _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(lse), _lib.ptr(delta), _lib.ptr(dk), _lib.ptr(dv), Z, H,
            ct.columns, q.size(2), D, do.stride(0), do.stride(1), do.stride(2), q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
            v.stride(0), v.stride(1), v.stride(2), dk.stride(0), dk.stride(1), dk.stride(2), dv.stride(0), dv.stride(1), dv.stride(2),
            ctx.tables.lines * 128, ctx.scale, _lib.ptr(ct.items), ct.n_items, _lib.ptr(partial), ct.n_slots, _lib.ptr(ct.split), ct.n_split,
            _lib.ptr(kpm), *ctx.kpm_args, _lib.stream_ptr(q.device))
        _lib.check(rc, 'bsp_attention_cols_bwd')
        return dk, dv

    @staticmethod
    def through_stored_gradient(ctx, saved, do, need_k, need_v):
        """dk and dv the other way (FUSED_KV = False): softmax and softmax gradient as sparse tensors, then the dsd operators; each
        only where its result is asked for"""
        q, k, v, o, lse, kpm = saved
        core = ctx.core
        lut, maxlut, _, lines = core.tables(q.device)[:4]
        stored = _StoredSoftmax()
        _attention_core.forward(stored, q, k, v, ctx.scale, None, kpm, None, ctx.kp_mask_mode, 'add', core, lut, maxlut, True, lines)
        p = stored.saved_tensors[3]
        dk = dv = None
        if need_k:
            ds = torch.empty_like(p)
            _attention_core.rows_kernel(stored, do, ds, None)
            dk = core.dsd_tn(ds, q)                        # ds^T . q and p^T . do, as the operators' backward passes do (matmul.py:598-601)
        if need_v:
            dv = core.dsd_tn(p, do)
        return dk, dv

    @staticmethod
    def backward(ctx, do):
        saved = ctx.saved_tensors                          # (unpacked once: non-reentrant checkpoints allow no more)
        q = saved[0]
        need_q, need_k, need_v = ctx.needs_input_grad[:3]
        if FUSED_KV:
            made = _lib.native().attn_bwd(ctx.tables.native(), do, *saved[:5], ctx.scale, saved[5], *ctx.kpm_args, need_q, need_k, need_v)
            if made is not None:
                return made + (None,) * 5
        do = _near(do)
        dq = dk = dv = None
        rows = (q.size(0), q.size(1), 2, ctx.tables.lines * 64)      # (the rows of a head as far apart as those of lse; the second half is not used)
        delta = None
        if need_k:
            delta = torch.empty(rows, dtype=torch.float32, device=q.device)
        elif need_v and FUSED_KV:
            delta = torch.zeros(rows, dtype=torch.float32, device=q.device)        # (dk is computed beside dv, and dropped)
        if need_q or need_k:
            dq = _attention_quad.rows_kernel(ctx, saved, do, delta if need_k else None)
        if need_k or need_v:
            dk, dv = (_attention_quad.columns_kernel(ctx, saved, do, delta) if FUSED_KV else
                      _attention_quad.through_stored_gradient(ctx, saved, do, need_k, need_v))
        return (dq if need_q else None, dk if need_k else None, dv if need_v else None) + (None,) * 5


def _vec32(t):
    """fp32 operands: unit inner stride, every other stride a multiple of 4 elements, aligned base, rows that do not overlap"""
    z, h, row, inner = t.stride()
    return t if inner == 1 and not (z | h | row) % 4 and row >= t.size(3) and not t.data_ptr() % 16 else _packed(t)


class _attention_f32(torch.autograd.Function):
    """The chain without per-element masks in fp32: what the backward pass needs of q, k and v are their bfloat16 parts, which the
    forward pass has made, and of the softmax two floats per row."""

    @staticmethod
    def forward(ctx, q, k, v, scale, key_padding_mask, kp_mask_mode, core, grad_enabled):
        global fused_f32_calls
        tables = core.quad(q.device)
        keep = grad_enabled and any(ctx.needs_input_grad[:3])
        kpm = None
        if key_padding_mask is not None:
            kpm = _sparse_softmax._strided16(key_padding_mask, 'key_padding_mask')
            if keep and kpm.data_ptr() == key_padding_mask.data_ptr():
                kpm = _packed(kpm[:, :k.size(2)])          # (as in _attention_quad)
        kpm_args = (kpm.stride(0) if kpm is not None and kpm.size(0) > 1 else 0, int(kp_mask_mode == 'mul'))
        launch, native = _lib.native(), tables.native()
        made = launch.attn32_fwd(native, q, k, v, scale, kpm, *kpm_args, keep)
        if made is None:                                   # operands that the kernels cannot address are copied to memory of their own
            made = launch.attn32_fwd(native, _vec32(q), _vec32(k), _vec32(v), scale, kpm, *kpm_args, keep)
            if made is None:
                raise _lib.BlocksparseLibraryError('attention: operands %s, %s, %s do not fit the layout' % (tuple(q.shape), tuple(k.shape), tuple(v.shape)))
        o, planes, stats, o_copy = made
        fused_f32_calls += 1
        if keep:                                           # (a copy of o: a program may add to the result in place, which none of the operators reads again)
            ctx.save_for_backward(planes, o_copy, stats, kpm)
            ctx.scale, ctx.tables, ctx.kpm_args = scale, tables, kpm_args
        return o

    @staticmethod
    def backward(ctx, do):
        planes, o, stats, kpm = ctx.saved_tensors
        args = (planes, stats, ctx.scale, kpm, *ctx.kpm_args, *ctx.needs_input_grad[:3])
        launch, native = _lib.native(), ctx.tables.native()
        made = launch.attn32_bwd(native, do, o, *args)
        if made is None:
            made = launch.attn32_bwd(native, _vec32(do), _vec32(o), *args)
            if made is None:
                raise _lib.BlocksparseLibraryError('attention: gradient %s does not fit the result %s' % (tuple(do.shape), tuple(o.shape)))
        return made + (None,) * 5


class _StoredSoftmax:
    """stands in for the autograd context of _attention_core where its kernels are called one by one"""

    def save_for_backward(self, *tensors):
        self.saved_tensors = tensors


class _attention_core(torch.autograd.Function):

    @staticmethod
    def forward(ctx, q, k, v, scale, rpe, key_padding_mask, attn_mask, kp_mask_mode, attn_mask_mode, core, lut, maxlut, keep_p, rows):
        global fused_calls
        H, R, C = core.spdims
        Z, D, block = q.size(0), q.size(3), core.block
        nnz = core.blocks()
        if rpe is not None or key_padding_mask is not None or attn_mask is not None:
            core._check_masks(q, rpe, key_padding_mask, attn_mask)
        q, k, v = _vec(q), _vec(k), _vec(v)
        null = ctypes.c_void_p(0)
        rpe_args = (null, 0, 0, 0)
        if rpe is not None:                                # element (z, h, r, c), softmax.py:50-55, 265
            while rpe.dim() < 4:
                rpe = rpe.unsqueeze(0)
            rpe = _sparse_softmax._strided16(rpe.expand(Z, H, rpe.size(2), rpe.size(3)), 'rpe')
            rpe_args = (_lib.ptr(rpe), rpe.stride(0), rpe.stride(1), rpe.stride(2))
        kpm_args = (null, 0)
        if key_padding_mask is not None:                   # element (z, c), softmax.py:60-62, 274
            key_padding_mask = _sparse_softmax._strided16(key_padding_mask, 'key_padding_mask')
            kpm_args = (_lib.ptr(key_padding_mask), key_padding_mask.stride(0) if key_padding_mask.size(0) > 1 else 0)
        attn_args = (null, 0)
        if attn_mask is not None:                          # element (r, c), softmax.py:67-70, 283
            attn_mask = _sparse_softmax._strided16(attn_mask, 'attn_mask')
            attn_args = (_lib.ptr(attn_mask), attn_mask.stride(0))
        p = torch.empty((Z, nnz, block, block), dtype=q.dtype, device=q.device) if keep_p else None
        o = torch.empty((Z, H, R * block, D), dtype=q.dtype, device=q.device)
        rc = _lib.load().bsp_attention_fwd(
            _lib.DTYPES[q.dtype], _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(p), _lib.ptr(o), Z, H, rows, D,
            q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2),
            o.stride(0), o.stride(1), o.stride(2), p.stride(0) if keep_p else 0, block, scale, _lib.ptr(lut), maxlut,
            rpe_args[0], rpe_args[1], rpe_args[2], rpe_args[3], kpm_args[0], kpm_args[1], int(kp_mask_mode == 'mul'),
            attn_args[0], attn_args[1], int(attn_mask_mode == 'mul'), _lib.stream_ptr(q.device))
        _lib.check(rc, 'bsp_attention_fwd')
        fused_calls += 1
        ctx.save_for_backward(q, k, v, p, o, lut)
        ctx.core, ctx.scale, ctx.maxlut, ctx.rows = core, scale, maxlut, rows
        ctx.columns = core.tables(q.device)[5]
        return o

    @staticmethod
    def rows_kernel(ctx, do, ds, delta, saved=None):
        """dq; with it the softmax gradient ds (if a tensor is given) and / or the rows' sums delta = sum_d do . o"""
        q, k, v, p, o, lut = saved or ctx.saved_tensors
        core = ctx.core
        Z, H, D = q.size(0), q.size(1), q.size(3)
        dq = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        rc = _lib.load().bsp_attention_bwd(
            _lib.DTYPES[q.dtype], _lib.ptr(do), _lib.ptr(v), _lib.ptr(k), _lib.ptr(p), _lib.ptr(o), _lib.ptr(ds), _lib.ptr(dq), Z, H, ctx.rows, D,
            do.stride(0), do.stride(1), do.stride(2), v.stride(0), v.stride(1), v.stride(2), k.stride(0), k.stride(1), k.stride(2),
            o.stride(0), o.stride(1), o.stride(2), dq.stride(0), dq.stride(1), dq.stride(2), p.stride(0), ds.stride(0) if ds is not None else 0,
            core.block, ctx.scale, _lib.ptr(lut), ctx.maxlut, _lib.ptr(delta), delta.stride(1) if delta is not None else 0,
            _lib.stream_ptr(q.device))
        _lib.check(rc, 'bsp_attention_bwd')
        return dq

    @staticmethod
    def columns_kernel(ctx, do, delta, saved=None):
        """dk and dv, the softmax gradient computed again from p and delta"""
        q, k, v, p, o, lut = saved or ctx.saved_tensors
        Z, H, D = q.size(0), q.size(1), q.size(3)
        ct = ctx.columns
        dk = torch.empty(k.shape, dtype=k.dtype, device=k.device)
        dv = torch.empty(v.shape, dtype=v.dtype, device=v.device)
        partial = torch.empty((Z, ct.n_slots, 2, 64, D), dtype=torch.float32, device=q.device) if ct.n_slots else None
        rc = _lib.load().bsp_attention_bwd_kv(
            _lib.DTYPES[q.dtype], _lib.ptr(do), _lib.ptr(q), _lib.ptr(v), _lib.ptr(p), _lib.ptr(delta), _lib.ptr(dk), _lib.ptr(dv), Z, H, ct.columns, D,
            do.stride(0), do.stride(1), do.stride(2), q.stride(0), q.stride(1), q.stride(2), v.stride(0), v.stride(1), v.stride(2),
            dk.stride(0), dk.stride(1), dk.stride(2), dv.stride(0), dv.stride(1), dv.stride(2), p.stride(0), delta.stride(1),
            ctx.core.block, ctx.scale, _lib.ptr(ct.items), ct.n_items, _lib.ptr(partial), ct.n_slots, _lib.ptr(ct.split), ct.n_split,
            _lib.stream_ptr(q.device))
        _lib.check(rc, 'bsp_attention_bwd_kv')
        return dk, dv

    @staticmethod
    def backward(ctx, do):
        saved = ctx.saved_tensors                          # (unpacked once, as above)
        q, k, v, p, o, lut = saved
        core = ctx.core
        do = _vec(do)
        need_q, need_k, need_v = ctx.needs_input_grad[:3]
        dq = dk = dv = None
        if need_k and FUSED_KV:
            # two launches: rows (dq, delta), then columns (dk and dv)
            delta = torch.empty((q.size(0), q.size(1), ctx.rows * 64), dtype=torch.float32, device=q.device)
            dq = _attention_core.rows_kernel(ctx, do, None, delta, saved)
            dk, dv = _attention_core.columns_kernel(ctx, do, delta, saved)
        else:
            if need_v:
                dv = core.dsd_tn(p, do)                    # p^T . do, as the dsd operator's backward does (matmul.py:598-601)
            if need_k:
                ds = torch.empty_like(p)
                dq = _attention_core.rows_kernel(ctx, do, ds, None, saved)
                dk = core.dsd_tn(ds, q)                    # ds^T . q (matmul.py:598-601 of the sdd operator)
            elif need_q:
                dq = _attention_core.rows_kernel(ctx, do, None, None, saved)
        return (dq if need_q else None, dk, dv if need_v else None) + (None,) * 11


def _core_for(sdd_nt, softmax, dsd_nn):
    """The fused core that stands for this triple of operators, or None when they are not such a triple."""
    if not (isinstance(sdd_nt, MatMul) and isinstance(dsd_nn, MatMul) and isinstance(softmax, Softmax)):
        return None
    core = getattr(softmax, '_attention_core', None)
    if core is not None and core[0] is sdd_nt and core[1] is dsd_nn:
        return core[2]
    ok = (sdd_nt.mode == 'sdd' and not sdd_nt.trans_a and sdd_nt.trans_b and dsd_nn.mode == 'dsd' and not dsd_nn.trans_a
          and not dsd_nn.trans_b and sdd_nt.block == softmax.block == dsd_nn.block and softmax.block in (16, 32, 64))
    if ok:
        for other in (sdd_nt.layout, dsd_nn.layout):
            ok = ok and (other is softmax.layout or (other.shape == softmax.layout.shape and bool((other == softmax.layout).all())))
    made = AttentionCore(softmax.layout, softmax.block) if ok else None
    softmax._attention_core = (sdd_nt, dsd_nn, made)
    return made


def attention_chain(sdd_nt, softmax, dsd_nn, q, k, v, scale=1., rpe=None, key_padding_mask=None, attn_mask=None,
                    key_padding_mask_mode='add', attn_mask_mode='add', dropout_p=0.):
    """dsd_nn(softmax(sdd_nt(q, k), ...), v): fused when the operators and tensors allow it, else the three calls."""
    core = _core_for(sdd_nt, softmax, dsd_nn)
    if core is not None and (core.usable_f32(q, k, v, rpe, attn_mask, dropout_p) if q.dtype == torch.float32 else core.usable(q, k, v, dropout_p)):
        return core(q, k, v, scale, rpe, key_padding_mask, attn_mask, key_padding_mask_mode, attn_mask_mode)
    w = sdd_nt(q, k)
    kwargs = dict(dropout_p=dropout_p) if dropout_p else {}
    w = softmax(w, scale=scale, rpe=rpe, key_padding_mask=key_padding_mask, attn_mask=attn_mask,
                key_padding_mask_mode=key_padding_mask_mode, attn_mask_mode=attn_mask_mode, **kwargs)
    return dsd_nn(w, v)
