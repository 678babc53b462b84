"""The host side of the launches without a GPU: what a call allocates, keeps and passes on.  Tensors are stand-ins, and every call of
the library below is one that it refuses, or that a stand-in takes, before anything is launched."""
import ctypes
import os
import pickle
import resource
import subprocess
import sys
import threading
import types

import pytest
import torch

from torch_blocksparse import _lib, matmul
from torch_blocksparse.attention_core import AttentionCore
from torch_blocksparse.matmul import GroupPlan, SddTables, _sparse_matmul


class FakeTensor:
    """what csrc/launch.cpp asks of a tensor"""

    def __init__(self, shape, dtype, ptr=1 << 20, device='cuda:0'):
        self.shape, self.dtype, self.device, self._ptr = tuple(shape), dtype, device, ptr

    def get_device(self):
        return 0

    def stride(self):
        out = [1]
        for n in self.shape[:0:-1]:
            out.insert(0, out[0] * n)
        return tuple(out)

    def data_ptr(self):
        return self._ptr


@pytest.fixture
def launcher():
    """csrc/launch.cpp on stand-ins: the module, what it allocated, and the statuses of the library that it raised"""
    module, made, raised = _lib.native(), [], []

    def empty(shape, dtype, device):
        # (memory for parts at an odd address: the library refuses such a call before it launches anything)
        made.append((shape, dtype))
        return FakeTensor(shape, dtype, 1 << 20 | (8 if dtype == 'uint8' else 0))

    def check(code, what):
        raised.append((what, code))
        raise ValueError(what)

    fake = types.SimpleNamespace(Tensor=FakeTensor, float16='float16', bfloat16='bfloat16', float32='float32', uint8='uint8', empty=empty)
    module.setup(fake, check, lambda dev: 0, FakeTensor, _sparse_matmul)
    yield types.SimpleNamespace(module=module, made=made, raised=raised)
    _lib._native = None                                    # (the next caller sets it up again)


def _sdd_tables(launch, block, dtype, n):
    """tables of n single blocks, the first of 4 x 4"""
    at = 1 << 21
    return launch.make_sdd((None,), block, dtype, 0, n, 1, 4, 4, (0, 0, 0, 0), (0, 0, 0, 0), 0, 0, 0, 0, (0, 0, 0, 0), 0, 150, 22, ((1, at, 0, n),))


@pytest.mark.parametrize('block,dtype,name', [(32, _lib.F32, 'float32'), (64, _lib.F16, 'float16'), (128, _lib.F16, 'float16')])
def test_every_sdd_in_parts_has_memory_of_its_own(launcher, block, dtype, name):
    lib, n, K = _lib.load(), 7, 4096
    tables = _sdd_tables(launcher.module, block, dtype, n)
    a = FakeTensor((1, 1, K, 4 * block), name)
    if block == 128:
        need = lib.bsp_sdd_splitk_workspace_bytes(1, n, 16)
    else:
        parts = lib.bsp_sdd_parts(dtype, block, 1, (ctypes.c_int * 1)(1), (ctypes.c_int64 * 1)(n), 1, K, 0)
        assert parts > 1
        need = lib.bsp_sdd_parts_workspace_bytes(block, n, 1, parts)
    assert need > 0
    for call in range(2):
        with pytest.raises(ValueError):
            launcher.module.sdd(tables, a, a, True, False, False, 0)
    assert launcher.made == [((1, n, block, block), name), ((need,), 'uint8')] * 2
    assert [code for _, code in launcher.raised] == [-1, -1]


@pytest.mark.parametrize('need', [(True, True, True), (True, False, False), (False, True, True)])
def test_attention_backward_allocates_in_front_of_each_launch(launcher, need):
    # delta and dq, then the row kernel (refused here: no lse), then dk, dv and the parts of long columns for the column kernel
    H, L, D, lines = 2, 256, 64, 4
    tables = launcher.module.make_attn((), 1 << 21, 1 << 21, 1 << 21, lines, 4, 8, 3, 1, 0, 4, H, 4, 4, 64)
    t = FakeTensor((3, H, L, D), 'float16')
    with pytest.raises(ValueError):
        launcher.module.attn_bwd(tables, t, t, t, t, t, FakeTensor((3, H, 2, 64 * lines), 'float32', 0), 1., None, 0, 0, *need)
    assert launcher.raised == [('bsp_attention_rows_bwd', -1)]
    assert launcher.made == [((3, H, 2, 64 * lines), 'float32')] * need[1] + [((3, H, L, D), 'float16')]


def _softmax_flags():
    """flags that run Python code when they are asked (as the results of an overloaded comparison may): in a process of its own"""
    asked = []

    class Flag:
        def __bool__(self):
            asked.append(sys._getframe(1).f_code.co_name)
            return True

    class NoFlag:
        def __bool__(self):
            raise KeyError('no flag')

    module, raised = _lib.native(), []
    fake = types.SimpleNamespace(Tensor=FakeTensor, float16='float16', bfloat16='bfloat16', float32='float32')

    def check(code, what):
        raised.append(code)
        raise ValueError(what)

    module.setup(fake, check, lambda dev: 0, FakeTensor, _sparse_matmul)
    rows = module.make_rows((), 0, 2, 0, 4, 1, 2, 2, 32)          # (no table: the library refuses the call)
    x = FakeTensor((1, 4, 32, 32), 'float16')
    for flags, error in (((Flag(), Flag()), ValueError), ((True, False), ValueError), ((NoFlag(), True), KeyError)):
        try:
            module.softmax_fwd(rows, x, 1., None, None, None, *flags)
        except error:
            continue
        raise AssertionError(flags)
    assert asked == ['_softmax_flags'] * 2 and raised == [-1, -1]


def _alone(name):
    """a function of this file in a process of its own, which it may end"""
    here = os.path.dirname(os.path.abspath(__file__))
    done = subprocess.run([sys.executable, '-c', 'import test_launch_host as t; t.%s()' % name], cwd=here, env=dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path)),
                          capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, (done.returncode, done.stderr[-2000:])


def test_the_softmax_reads_its_flags_with_the_lock_held():
    _alone('_softmax_flags')


@pytest.mark.parametrize('block,dtype', [(32, torch.float32), (128, torch.float16)])
def test_calls_that_overlap_share_no_memory(block, dtype, monkeypatch):
    # the general host side: a second thread's call while the first one is between its two launches
    real, K, nnz = _lib.load(), 4096, 3
    places, inner = [], []

    def launch(*args):
        ws, need = [(a.value, n) for a, n in zip(args, args[1:]) if hasattr(a, 'value') and a.value and isinstance(n, int) and n > 4096][-1]
        places.append((ws, need))
        if len(places) == 1:
            t = threading.Thread(target=lambda: inner.append(product()))
            t.start()
            t.join(60)
        return _lib.OK

    class Library:
        bsp_sdd_matmul_levels = bsp_sdd_matmul_splitk = staticmethod(launch)

        def __getattr__(self, name):
            return getattr(real, name)

    monkeypatch.setattr(_lib, 'load', lambda: Library())
    monkeypatch.setattr(_lib, 'stream_ptr', lambda device: None)
    tables = SddTables([torch.zeros(4 * nnz, dtype=torch.int32)])
    tables.nnz, tables.spdims, tables.widths, tables.packs = nnz, (1, 4, 4), [nnz], [1]
    a = torch.zeros(1, 1, K, 4 * block, dtype=dtype)
    product = lambda: _sparse_matmul._sdd_matmul(a, a, True, False, False, (1, 4, 4), block, tables, None, None, None, False, [None])
    product()
    (one, need), (two, again) = places
    assert inner and need == again and (one + need <= two or two + need <= one)


def test_a_linear_layer_takes_any_number_of_tokens_whenever_its_tables_were_built(monkeypatch):
    # made ahead (make_lut), or by a call of the product itself, which reduces over multiples of 16 only
    lin = matmul.Linear(64, 96, 32, torch.ones(1, 2, 3, dtype=torch.int64))
    key = (torch.float32, torch.device('cpu'))
    tables = SddTables()
    lin.matmul.lut_cache[key] = (None,) * 8 + (tables, None, None, None)
    first = lin.matmul._product(*key)
    assert lin.matmul._product(*key) is first and not tables.any_k
    seen = []

    def call(op, a, b):
        product = op._product(*key)
        seen.append((product.luts[8].any_k, op._product(*key) is product))
        return a.new_zeros(1, 1, a.size(2), 96)

    monkeypatch.setattr(matmul.MatMul, '__call__', call)
    lin(torch.zeros(7, 64))
    assert seen == [(True, True)]


def test_copies_of_ragged_operands_only_where_they_pay():
    whole = _lib.load().bsp_sdd_whole_steps
    for dtype, block, side, density, K, copies in (
            (_lib.F16, 128, 4096, .5, 8176, 0), (_lib.BF16, 64, 4096, .5, 8176, 0), (_lib.F32, 32, 4096, .5, 8176, 0), (_lib.F16, 32, 4096, .5, 8192, 0),
            (_lib.F16, 32, 4096, .1, 8176, 0), (_lib.F16, 32, 4096, .25, 8176, 1), (_lib.F16, 32, 4096, .25, 1040, 0), (_lib.F16, 32, 1024, .5, 8176, 0), (_lib.F16, 32, 2048, .5, 8176, 0),
            (_lib.F16, 16, 4096, .1, 2032, 1), (_lib.F16, 16, 4096, .1, 1040, 0), (_lib.F16, 16, 1024, .5, 8176, 0), (_lib.F16, 16, 65536, .5, 255, 0)):
        assert whole(dtype, block, int(density * (side // block) ** 2), side, side, K) == copies, (dtype, block, side, density, K)


def _builders_without_memory():
    """the builders of tables on the host with no memory left for their lists: in a process of its own"""
    lib = _lib.load()
    wide = ctypes.create_string_buffer(1 << 24)            # 16 Mi cells of a layout, none there
    out, n, m, info = (ctypes.c_int32 * 1024)(), ctypes.c_int64(0), ctypes.c_int(0), _lib.AttentionTables()
    with open('/proc/self/statm') as f:
        used = int(f.read().split()[0]) * resource.getpagesize()
    resource.setrlimit(resource.RLIMIT_AS, (used + (24 << 20),) * 2)
    assert lib.bsp_sdd_tiles_build(wide, 1, 1 << 24, 1, out, 1024, ctypes.byref(n)) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_xsd_chunks_build(wide, 1, 4096, 4096, 1, out, 1024, ctypes.byref(m), ctypes.byref(n)) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_attention_tables_build(wide, 1, 1, 1 << 24, 64, out, 1024, ctypes.byref(info)) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_attention_stored_tables_build(wide, None, 1, 1, 1 << 24, 64, 0, out, 1024, ctypes.byref(info)) == _lib.ERR_UNSUPPORTED
    assert lib.bsp_sdd_tiles_build(wide, 1, 64, 64, out, 1024, ctypes.byref(n)) == _lib.OK and n.value == 0


def test_builders_report_that_memory_is_short():
    _alone('_builders_without_memory')


def test_a_product_follows_the_operator_as_it_is_at_the_call():
    op = matmul.MatMul(torch.ones(1, 2, 2, dtype=torch.int64), 32, 'dds')
    key = (torch.float32, torch.device('cpu'))
    op.lut_cache[key] = (None,) * 8 + (SddTables(), None, None, None)
    first = op._product(*key)
    assert op._product(*key) is first
    op.trans_a = True                                      # (the tables of dds do not depend on it)
    turned = op._product(*key)
    assert turned.trans_a and not first.trans_a
    op.trans_a, op.bench = False, True
    assert op._product(*key).bench and not op._product(*key).trans_a


def test_operators_saved_without_what_the_native_launches_keep_can_be_loaded():
    core = AttentionCore(torch.ones(1, 2, 2, dtype=torch.int64), 64)
    quad = core._made(torch.device('cpu'))[0]
    shape = quad.__dict__.pop('shape')
    loaded = pickle.loads(pickle.dumps(core))
    got = loaded._tables['cpu'][0]
    assert got.shape == shape == (1, 2, 2, 64) and got._native is None and torch.equal(got.rows, quad.rows)
    # a product's tables: no length of the longest segment, plans without flags
    plan = GroupPlan(torch.zeros(8, dtype=torch.int32), 1, 2)
    plan.__dict__.pop('flags', None)
    lut = torch.zeros(64, dtype=torch.int32)
    lut.planbuf, lut.nnz, lut.gplan, lut.gplan_wide = torch.zeros(64, dtype=torch.int32), 4, plan, None
    lut, plan = pickle.loads(pickle.dumps((lut, plan)))
    assert lut.gplan.flags == plan.flags == 0
    op = matmul.MatMul(torch.ones(1, 2, 2, dtype=torch.int64), 64, 'dsd')
    op.lut_cache[torch.float32, torch.device('cuda', 0)] = (lut, 0, 2, None) + (SddTables(), None, None, None) + (lut, 0, 2, None)
    product = op._product(torch.float32, torch.device('cuda', 0))
    assert product._tables(0) is not None and product._tables(2) is not None


def test_tables_that_another_thread_builds_meanwhile_are_seen_by_the_next_call(monkeypatch):
    lut = torch.zeros(64, dtype=torch.int32)
    lut.planbuf, lut.nnz, lut.longest, lut.gplan, lut.gplan_wide = torch.zeros(64, dtype=torch.int32), 4, 2, None, None
    lut.build_wide = lambda: None
    op = matmul.MatMul(torch.ones(1, 2, 2, dtype=torch.int64), 32, 'dsd')
    key = (torch.float16, torch.device('cuda', 0))
    op.lut_cache[key] = (lut, 0, 2, None) + (SddTables(), None, None, None) + (lut, 0, 2, None)
    real = _lib.native()

    def make_xsd(*args):
        made = real.make_xsd(*args)
        lut.gplan_wide = GroupPlan(torch.zeros(8, dtype=torch.int32), 1, 2)      # the other thread
        return made

    monkeypatch.setattr(_lib, 'native', lambda: types.SimpleNamespace(make_xsd=make_xsd))
    product = op._product(*key)
    assert product._tables(0) is not None and product.built[0] != product._on_demand(0)
