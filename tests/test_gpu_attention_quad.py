"""GPU: the attention kernels that keep no sparse tensor (bsp_attention_rows_fwd, bsp_attention_rows_bwd,
bsp_attention_cols_bwd behind attention_chain) at the points where they can go wrong: numbers of heads that do not divide
by the heads a launch takes together, lines of one tile and of many, tiles with missing pieces, a running maximum that
moves at every tile or starts at -inf, negative and zero scale, operands far apart in memory.  Tolerance: assert_close, the
bounds every fp16 / bf16 comparison with the fp32 oracle uses."""
import ctypes

import pytest
import torch

import torch_blocksparse as tb
from torch_blocksparse import _lib, attention_core as ac
from oracle import dense_oracle as D
from helpers import assert_close, guard_allocations

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _run(layout, block, q, k, v, do, **kw):
    ops = (tb.MatMul(layout, block, 'sdd', trans_b=True), tb.Softmax(layout, block), tb.MatMul(layout, block, 'dsd'))
    ts = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
    before = ac.fused_calls
    with guard_allocations('attention without sparse tensors'):
        o = ac.attention_chain(ops[0], ops[1], ops[2], *ts, **kw)
        o.backward(do)
        torch.cuda.synchronize()
    assert ac.fused_calls == before + 1
    return [o.detach()] + [t.grad for t in ts]


def _check(got, ref, dtype):
    for name, g, r in zip(('o', 'dq', 'dk', 'dv'), got, ref):
        assert not bool(torch.isnan(g).any()), name
        assert_close(g, r, dtype, name)


@pytest.mark.parametrize('Z,H,block,R,C,d,dtype', [
    (1, 1, 64, 1, 1, 64, torch.float16),
    (1, 3, 64, 2, 5, 128, torch.bfloat16),
    (5, 1, 32, 6, 4, 64, torch.bfloat16),
    (3, 3, 16, 8, 12, 64, torch.float16),
    (1, 6, 16, 4, 20, 128, torch.float16),
    (2, 2, 64, 40, 3, 64, torch.float16),       # columns of 40 tiles: parts and their sum
])
def test_shapes_at_the_edges(Z, H, block, R, C, d, dtype):
    torch.manual_seed(R * C + d)
    lay = (torch.rand(H, R, C) < 0.6).long()
    lay[:, :, 0] = 1
    q, do = [torch.randn(Z, H, R * block, d, device=DEV).to(dtype) for _ in range(2)]
    k, v = [torch.randn(Z, H, C * block, d, device=DEV).to(dtype) for _ in range(2)]
    kpm = torch.zeros(Z, C * block, device=DEV, dtype=dtype)
    kpm[-1, 5:9] = float('-inf')
    got = _run(lay, block, q, k, v, do, scale=d ** -0.5, key_padding_mask=kpm)
    _check(got, D.attention(q, k, v, lay, block, d ** -0.5, key_padding_mask=kpm, attn_mask_mode='add', do=do), dtype)


@pytest.mark.parametrize('down', [False, True])
@pytest.mark.parametrize('block,d', [(64, 64), (16, 128)])
def test_a_maximum_that_moves_at_every_tile(block, d, down):
    """Logits that rise (fall) by 10 from tile to tile, 2^14 in the exponentials: every tile (none but the first) moves the
    running maximum.  The first 64 keys are masked: the maximum starts at -inf.  The scores are exact in fp16."""
    torch.manual_seed(d)
    Z, H, R, C = 1, 2, 2 * 64 // block, 6 * 64 // block
    lay = torch.ones(H, R, C, dtype=torch.int64)
    n = torch.arange(C * block)
    logit = 10. * ((C * block - 1 - n) // 64 if down else n // 64) + 0.5 * (n % 3)
    q, k = torch.zeros(Z, H, R * block, d), torch.zeros(Z, H, C * block, d)
    q[..., 0] = 8.
    k[..., 0] = logit
    q, k = q.half().to(DEV), k.half().to(DEV)
    v, do = torch.randn(Z, H, C * block, d, device=DEV).half(), torch.randn(Z, H, R * block, d, device=DEV).half()
    kpm = torch.zeros(Z, C * block, device=DEV).half()
    kpm[:, :64] = float('-inf')
    got = _run(lay, block, q, k, v, do, scale=0.125, key_padding_mask=kpm)
    ref = D.attention(q, k, v, lay, block, 0.125, key_padding_mask=kpm, attn_mask_mode='add', do=do)
    # dq sums ds k over the row with k up to 51: its error follows the size of what was summed, ds rounded to 2^-11
    for name, g, r in zip(('o', 'dk', 'dv'), (got[0], got[2], got[3]), (ref[0], ref[2], ref[3])):
        assert_close(g, r, torch.float16, name)
    p = torch.softmax((q.float() @ k.float().transpose(2, 3).contiguous() * 0.125).cpu() + kpm.float().cpu()[:, None, None], -1)
    terms = (p * ((do.float() @ v.float().transpose(2, 3).contiguous()).cpu().abs() + 40.) * 0.125) @ k.float().cpu().abs()
    assert bool(((got[1].float().cpu() - ref[1]).abs() <= 2 ** -10 * terms + 1e-2 * ref[1].abs() + 1e-2).all())


def test_negative_and_zero_scale():
    torch.manual_seed(2)
    Z, H, R, block, d = 2, 3, 5, 64, 64
    lay = torch.tril(torch.ones(H, R, R)).long()
    q, k, v, do = [torch.randn(Z, H, R * block, d, device=DEV).half() for _ in range(4)]
    o, dq, dk, dv = D.attention(q, -k, v, lay, block, 0.125, attn_mask_mode='add', do=do)
    _check(_run(lay, block, q, k, v, do, scale=-0.125), (o, dq, -dk, dv), torch.float16)
    got = _run(lay, block, q, k, v, do, scale=0.)
    zero = torch.zeros_like(q)
    o, _, _, dv = D.attention(zero, k, v, lay, block, 1., attn_mask_mode='add', do=do)
    assert not bool(got[1].any()) and not bool(got[2].any())
    _check((got[0], got[3]), (o, dv), torch.float16)


def test_gradients_without_those_of_the_keys():
    torch.manual_seed(4)
    lay = torch.tril(torch.ones(2, 4, 4)).long()
    q, k, v, do = [torch.randn(1, 2, 256, 64, device=DEV).half() for _ in range(4)]
    full = _run(lay, 64, q, k, v, do, scale=0.125)
    core = ac.AttentionCore(lay, 64)
    for need in ((True, False, False), (False, False, True), (True, False, True)):
        ts = [t.clone().requires_grad_(n) for t, n in zip((q, k, v), need)]
        core(*ts, scale=0.125).backward(do)
        for t, n, f in zip(ts, need, full[1:]):
            assert (t.grad is not None) == n and (not n or torch.equal(t.grad, f))


def test_c_abi_argument_checks():
    lib = _lib.load()
    t = torch.zeros(1, 1, 64, 64, device=DEV, dtype=torch.float16)
    o, lse = t.clone(), torch.zeros(1, 1, 64, device=DEV)
    table = ac.AttentionCore(torch.ones(1, 1, 1, dtype=torch.int64), 64).quad(torch.device(DEV)).rows
    null, st = ctypes.c_void_p(0), (t.stride(0), t.stride(1))

    def fwd(dtype=0, q=t, D=64, ldk=64, keys=64, lse_sh=64):
        return lib.bsp_attention_rows_fwd(dtype, _lib.ptr(q), _lib.ptr(t), _lib.ptr(t), _lib.ptr(o), _lib.ptr(lse), 1, 1, 1, keys, D,
                                          *st, 64, *st, ldk, *st, 64, *st, 64, lse_sh, 1.0, _lib.ptr(table), null, 0, 0, _lib.stream_ptr(torch.device(DEV)))
    assert fwd() == _lib.OK
    assert fwd(dtype=_lib.F32) == _lib.ERR_UNSUPPORTED
    assert fwd(D=96) == _lib.ERR_UNSUPPORTED
    assert fwd(q=None) != _lib.OK
    assert fwd(ldk=60) != _lib.OK
    assert fwd(keys=0) != _lib.OK
    assert fwd(keys=2 ** 25) != _lib.OK                 # 2^25 rows of 128 bytes: beyond the 32-bit offsets
    assert fwd(lse_sh=32) != _lib.OK
    torch.cuda.synchronize()


def _padded_rows(block, dtype, pad, R=512):
    """Causal layout, left padding of finite values over the first 128 keys of one sequence and over all keys of the other:
    rows 0 .. 127 of the one and every row of the other see nothing but padded keys."""
    lay = torch.tril(torch.ones(2, R // block, R // block)).long()
    kpm = torch.zeros(2, R)
    kpm[0, :128] = pad
    kpm[1] = pad
    return lay, kpm.to(dtype).to(DEV)


@pytest.mark.parametrize('block,d,dtype,pad', [
    (64, 64, torch.float16, -1e4), (16, 64, torch.float16, -65504.), (32, 128, torch.float16, -65504.),
    (64, 128, torch.bfloat16, -1e6), (16, 64, torch.bfloat16, -1e9), (64, 64, torch.bfloat16, -1e9)])
def test_shares_of_rows_that_see_only_padded_keys_add_up_to_one(block, d, dtype, pad):
    """do is a one in row 2 j + 1, column j: sum_c dv[c, j] is the sum of that row's shares as the backward pass has them.  Each
    share is rounded to the operand type once (2^-11, 2^-8 of it, or 2^-25 in fp16's subnormals); one is what they add up to."""
    torch.manual_seed(d + block)
    lay, kpm = _padded_rows(block, dtype, pad)
    q, k, v = [torch.randn(2, 2, 512, d, device=DEV).to(dtype) for _ in range(3)]
    do = torch.zeros(2, 2, 512, d, device=DEV)
    do[:, :, 2 * torch.arange(min(d, 64)) + 1, torch.arange(min(d, 64))] = 1.
    got = _run(lay, block, q, k, v, do.to(dtype), scale=d ** -0.5, key_padding_mask=kpm)
    sums = got[3].double().sum(2)[..., :min(d, 64)]
    unit = 2. ** -11 if dtype == torch.float16 else 2. ** -8
    assert float((sums - 1.).abs().max()) <= unit + 512 * 2. ** -25 + 2. ** -16
    if dtype == torch.float16:
        do = torch.randn(2, 2, 512, d, device=DEV).to(dtype)
        got = _run(lay, block, q, k, v, do, scale=d ** -0.5, key_padding_mask=kpm)
        _check(got, D.attention(q, k, v, lay, block, d ** -0.5, key_padding_mask=kpm, attn_mask_mode='add', do=do), dtype)


def test_the_rest_of_lse_is_part_of_the_row_buffers_only_when_asked_for():
    lib = _lib.load()
    t, lse = torch.zeros(1, 1, 64, 64, device=DEV, dtype=torch.float16), torch.full((128,), 7., device=DEV)
    table = ac.AttentionCore(torch.ones(1, 1, 1, dtype=torch.int64), 64).quad(torch.device(DEV)).rows
    null, st = ctypes.c_void_p(0), (t.stride(0), t.stride(1), 64)
    for flag, stride, ok in ((0, 64, True), (0, 128, True), (_lib.ROWS_WITH_REST, 64, False), (_lib.ROWS_WITH_REST, 128, True)):
        lse.fill_(7.)
        o = torch.empty_like(t)
        rc = lib.bsp_attention_rows_fwd(flag, _lib.ptr(t), _lib.ptr(t), _lib.ptr(t), _lib.ptr(o), _lib.ptr(lse), 1, 1, 1, 64, 64, *st, *st, *st, *st,
                                        stride, 1.0, _lib.ptr(table), null, 0, 0, _lib.stream_ptr(torch.device(DEV)))
        assert (rc == _lib.OK) == ok
        if ok:
            assert lse[:64].tolist() == [6.] * 64 and lse[64:].tolist() == [0. if flag else 7.] * 64
    torch.cuda.synchronize()


@pytest.mark.parametrize('block,d,dtype,why', [
    (16, 64, torch.float16, 'padded'), (32, 64, torch.bfloat16, 'padded'), (16, 128, torch.bfloat16, 'padded'), (32, 128, torch.float16, 'padded'),
    (16, 64, torch.float16, 'overflow'), (32, 128, torch.float16, 'overflow')])
def test_rows_without_a_softmax_reach_only_the_keys_they_attend_to(block, d, dtype, why):
    """Causal layout whose first block-row sees nothing but its own keys, all padded (or one of whose rows has scores beyond the
    type): these rows are NaN, and the gradients of the keys of their block; the other keys of the same 64 x 64 tiles have no block there."""
    torch.manual_seed(block + d)
    lay = torch.tril(torch.ones(2, 256 // block, 256 // block)).long()
    q, k, v, do = [torch.randn(2, 2, 256, d, device=DEV).to(dtype) for _ in range(4)]
    kw = dict(scale=d ** -0.5)
    if why == 'padded':
        kw['key_padding_mask'] = torch.zeros(2, 256, device=DEV).to(dtype)
        kw['key_padding_mask'][0, :block] = float('-inf')
        do[0, 1, :block] = 0.
    else:
        q[0, :, 3] = 6e4
    got = _run(lay, block, q, k, v, do, **kw)
    old = ac.FUSED
    try:
        ac.FUSED = False
        ops = (tb.MatMul(lay, block, 'sdd', trans_b=True), tb.Softmax(lay, block), tb.MatMul(lay, block, 'dsd'))
        ts = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = ac.attention_chain(*ops, *ts, **kw)
        o.backward(do)
    finally:
        ac.FUSED = old
    for name, g, r in zip(('o', 'dq', 'dk', 'dv'), got, [o.detach()] + [t.grad for t in ts]):
        assert torch.equal(torch.isnan(g), torch.isnan(r)), name
        assert bool(torch.isnan(r).any()) and not bool(torch.isnan(r[1]).any()) and not bool(torch.isnan(r[0, :, block:]).any()), name
        assert_close(g, r, dtype, name)


@pytest.mark.parametrize('block,d', [(64, 64), (16, 128), (32, 64), (64, 128)])
def test_padding_values_beyond_the_scores(block, d):
    """-1e9 in bf16: in rows that see nothing else, fp32 rounds the scores away beside it and every key gets the same share, in
    the oracle, in the three operators and in the fused kernels."""
    torch.manual_seed(d)
    lay, kpm = _padded_rows(block, torch.bfloat16, -1e9)
    q, k, v, do = [torch.randn(2, 2, 512, d, device=DEV).bfloat16() for _ in range(4)]
    kw = dict(scale=d ** -0.5, key_padding_mask=kpm)
    got = _run(lay, block, q, k, v, do, **kw)
    _check(got, D.attention(q, k, v, lay, block, d ** -0.5, key_padding_mask=kpm, attn_mask_mode='add', do=do), torch.bfloat16)
    ops = (tb.MatMul(lay, block, 'sdd', trans_b=True), tb.Softmax(lay, block), tb.MatMul(lay, block, 'dsd'))
    ts = [t.clone().requires_grad_(True) for t in (q, k, v)]
    o = ops[2](ops[1](ops[0](ts[0], ts[1]), **kw), ts[2])
    o.backward(do)
    _check(got, [o.detach()] + [t.grad for t in ts], torch.bfloat16)


@pytest.mark.parametrize('block', [64, 16])
@pytest.mark.parametrize('masked_first', [False, True])
def test_capture_of_the_kind_of_call_that_the_warm_up_was_not(block, masked_first):
    """Calls with per-element masks run other kernels on other tables than calls without.  Operators that have met one kind
    only are captured with the other; every replay against operators that run it eagerly."""
    torch.manual_seed(block)
    L = 256
    lay = torch.tril(torch.ones(2, L // block, L // block)).long()
    make = lambda: (tb.MatMul(lay, block, 'sdd', trans_b=True), tb.Softmax(lay, block), tb.MatMul(lay, block, 'dsd'))
    masks = dict(rpe=(0.3 * torch.randn(L, L, device=DEV)).half())
    ops, others = make(), make()

    def chain(ops, tensors, kw):
        ts = [t.detach().clone().requires_grad_(True) for t in tensors[:3]]
        before = ac.fused_calls
        o = ac.attention_chain(*ops, *ts, scale=0.125, **kw)
        assert ac.fused_calls == before + 1
        return (o.detach(),) + torch.autograd.grad(o, ts, tensors[3])
    static_in = [torch.randn(2, 2, L, 64, device=DEV).half() for _ in range(4)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        chain(ops, static_in, masks if masked_first else {})
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    kw = {} if masked_first else masks
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_out = chain(ops, static_in, kw)
    for _ in range(3):
        fresh = [torch.randn_like(t) for t in static_in]
        eager = chain(others, fresh, kw)
        torch.cuda.synchronize()
        for s, f in zip(static_in, fresh):
            s.copy_(f)
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(('o', 'dq', 'dk', 'dv'), static_out, eager):
            assert torch.equal(a, b), name


@pytest.mark.parametrize('which', ['do over positions', 'k of one position', 'odd address', 'odd stride of a single batch', 'rows apart', 'overlapping rows'])
@pytest.mark.parametrize('masked', [False, True])
def test_operands_that_the_kernels_cannot_address_are_copied(which, masked):
    """Tensors that are contiguous or aligned in the wrong way, or whose rows overlap (a gradient that reaches every position
    through a sum has rows 0 apart), against the same values in memory of their own."""
    torch.manual_seed(5)
    Z, L, d = (1 if 'batch' in which else 2), 256, 64
    lay = torch.tril(torch.ones(2, L // 32, L // 32)).long()
    q, k, v, do = [torch.randn(Z, 2, L, d, device=DEV).half() for _ in range(4)]
    if which == 'do over positions':
        do = torch.randn(Z, 2, d, device=DEV).half()[:, :, None].expand(-1, -1, L, -1)
    elif which == 'k of one position':
        k = k[:, :, :1].expand(-1, -1, L, -1)
    elif which == 'odd address':
        q, do = [torch.randn(Z * 2 * L * d + 1, device=DEV).half()[1:].view(Z, 2, L, d) for _ in range(2)]
    elif which == 'odd stride of a single batch':
        v, do = [t.as_strided(t.shape, (2 * L * d + 3,) + t.stride()[1:]) for t in (v, do)]
    elif which == 'rows apart':
        q, k, v, do = [torch.randn(Z, L, 2, 3 * d, device=DEV).half()[..., d:2 * d].transpose(1, 2) for _ in range(4)]
    else:
        v = torch.randn(Z * 2 * L * 32 + 32, device=DEV).half().as_strided((Z, 2, L, d), (2 * L * 32, L * 32, 32, 1))
    kw = dict(scale=0.125, rpe=(0.3 * torch.randn(L, L, device=DEV)).half()) if masked else dict(scale=0.125)

    def grads(q, k, v, do):
        ops = (tb.MatMul(lay, 32, 'sdd', trans_b=True), tb.Softmax(lay, 32), tb.MatMul(lay, 32, 'dsd'))
        ts = [t.detach().requires_grad_(True) for t in (q, k, v)]
        before = ac.fused_calls
        o = ac.attention_chain(*ops, *ts, **kw)
        assert ac.fused_calls == before + 1
        return (o,) + torch.autograd.grad(o, ts, do)
    for name, a, b in zip(('o', 'dq', 'dk', 'dv'), grads(q, k, v, do), grads(*[t.clone(memory_format=torch.contiguous_format) for t in (q, k, v, do)])):
        assert torch.equal(a, b), name


@pytest.mark.parametrize('d,dtype,block', [(64, torch.float16, 64), (128, torch.bfloat16, 64), (64, torch.bfloat16, 16)])
def test_operands_far_apart_in_memory(d, dtype, block):
    """Rows 2.9 MB apart, so that the last ones of the tensors that are fetched tile by tile lie just below 4 GiB from the first: byte
    offsets beyond 2^31, and the largest row stride that 1472 positions allow."""
    torch.manual_seed(d + block)
    L = 1472
    ld = 2 ** 32 // (2 * L) // 8 * 8
    assert 2 * L * ld < 2 ** 32 <= 2 * L * (ld + 8)
    lay = (torch.rand(2, L // block, L // block) < 0.3).long()
    lay[:, :, 0] = lay[:, :, -1] = 1
    buf = torch.empty(L * ld, device=DEV, dtype=dtype)
    near = [torch.randn(1, 2, L, d, device=DEV).to(dtype) for _ in range(4)]
    far = [buf.as_strided((1, 2, L, d), (16, 4 * d, ld, 1), i * d) for i in range(4)]
    for f, n in zip(far, near):
        f.copy_(n)
    core = ac.AttentionCore(lay, block)
    results = []
    for q, k, v, do in (far, near):
        assert all(ac._near(t) is t for t in (q, k, v, do))
        ts = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = core(*ts, scale=d ** -0.5)
        results.append((o,) + torch.autograd.grad(o, ts, do))
    for name, a, b in zip(('o', 'dq', 'dk', 'dv'), *results):
        assert torch.equal(a, b), name


@pytest.mark.parametrize('layout_of', [lambda m: m, lambda m: m[:1], lambda m: torch.cat((m, m), 1)[:, :256], lambda m: m[0].expand(2, -1),
                                       lambda m: torch.cat((m, m), 1)[:, :260]])
def test_a_mask_buffer_may_be_refilled_before_the_backward_pass(layout_of):
    torch.manual_seed(6)
    lay = torch.tril(torch.ones(2, 4, 4)).long()
    q, k, v, do = [torch.randn(2, 2, 256, 64, device=DEV).half() for _ in range(4)]
    mask = torch.zeros(2, 256, device=DEV).half()
    mask[0, 3:40] = float('-inf')
    mask = layout_of(mask)
    results = []
    for refill in (False, True):
        core = ac.AttentionCore(lay, 64)
        ts = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = core(*ts, scale=0.125, key_padding_mask=mask)
        if refill:
            (mask if mask.stride(0) or mask.size(0) == 1 else mask[0]).fill_(1.)
        results.append((o.detach(),) + torch.autograd.grad(o, ts, do))
    for name, a, b in zip(('o', 'dq', 'dk', 'dv'), *results):
        assert torch.equal(a, b), name


@pytest.mark.parametrize('block,kpm', [(64, False), (16, True)])
def test_a_scale_that_is_not_a_number(block, kpm):
    torch.manual_seed(7)
    lay = torch.tril(torch.ones(2, 256 // block, 256 // block)).long()
    q, k, v = [torch.randn(2, 2, 256, 64, device=DEV).half().requires_grad_(True) for _ in range(3)]
    kw = dict(key_padding_mask=torch.zeros(2, 256, device=DEV).half()) if kpm else {}
    core = ac.AttentionCore(lay, block)
    o = core(q, k, v, scale=float('nan'), **kw)
    for t in (o,) + torch.autograd.grad(o, (q, k, v), torch.ones_like(o)):
        assert bool(torch.isnan(t).all())


@pytest.mark.parametrize('which', ['dq', 'dk'])
@pytest.mark.parametrize('block,d,scale', [(64, 64, 8.), (16, 64, -8.), (32, 128, 64.), (64, 64, 1e5)])
def test_small_gradients_under_a_scale_above_one(which, block, d, scale):
    """fp16 gradients so small that ds without the scale lies in the subnormals.  ds with it is rounded in steps of 2^-24 there, an
    error of 2^-24 / sqrt(12) an element that the product takes on as relative to its root mean square; beside it the result's own
    rounding, 2^-11 or half a step of 2^-24, and of what ds is made of."""
    torch.manual_seed(d)
    L = 512
    lay = torch.ones(2, L // block, L // block, dtype=torch.int64)
    small = 0.64 / (abs(scale) * d ** 0.5)                # scores of about 0.64, so that the shares are spread
    q, k = torch.randn(1, 2, L, d, device=DEV), torch.randn(1, 2, L, d, device=DEV)
    q, k = (q * small, k) if which == 'dq' else (q, k * small)
    v, do = torch.randn(1, 2, L, d, device=DEV), torch.randn(1, 2, L, d, device=DEV) * 2. ** -12 / min(abs(scale), 64.)
    q, k, v, do = [t.half() for t in (q, k, v, do)]
    got = _run(lay, block, q, k, v, do, scale=scale)[1 if which == 'dq' else 2].double()
    Q, K, V, dO = [t.double() for t in (q, k, v, do)]
    P = torch.softmax(Q @ K.transpose(2, 3).contiguous() * scale, -1)
    dP = dO @ V.transpose(2, 3).contiguous()
    dS = P * (dP - (P * dP).sum(-1, keepdim=True)) * scale
    ref = dS @ K if which == 'dq' else dS.transpose(2, 3).contiguous() @ Q
    step, rms = 2. ** -24 / 12 ** 0.5, lambda t: float(t.pow(2).mean().sqrt())
    assert 4 * rms(dS) / abs(scale) < 2. ** -14 and rms(ref) > 2. ** -16
    bound = step / rms(dS) + step / rms(ref) + 3 * 2. ** -11
    assert float((got - ref).norm() / ref.norm()) < 1.25 * bound


@pytest.mark.parametrize('masks', [(), ('key_padding_mask',), ('rpe',)])
def test_under_a_non_reentrant_checkpoint(masks):
    """which lets a backward pass unpack what was saved once"""
    from torch.utils.checkpoint import checkpoint
    torch.manual_seed(8)
    core = ac.AttentionCore(torch.tril(torch.ones(2, 4, 4)).long(), 64)
    q, k, v, do = [torch.randn(2, 2, 256, 64, device=DEV).half() for _ in range(4)]
    values = dict(key_padding_mask=(0.5 * torch.randn(2, 256, device=DEV)).half(), rpe=(0.3 * torch.randn(256, 256, device=DEV)).half())
    kw = dict(scale=0.125, **{m: values[m] for m in masks})
    results = []
    for wrap in (lambda f, *ts: f(*ts), lambda f, *ts: checkpoint(f, *ts, use_reentrant=False)):
        ts = [t.clone().requires_grad_(True) for t in (q, k, v)]
        o = wrap(lambda a, b, c: core(a, b, c, **kw), *ts)
        results.append((o.detach(),) + torch.autograd.grad(o, ts, do))
    for name, a, b in zip(('o', 'dq', 'dk', 'dv'), *results):
        assert torch.equal(a, b), name


def test_stored_gradient_way_computes_what_is_asked_for(monkeypatch):
    """FUSED_KV = False: one product for one gradient, the same values as where both are asked for"""
    torch.manual_seed(9)
    core = ac.AttentionCore(torch.tril(torch.ones(2, 4, 4)).long(), 64)
    q, k, v, do = [torch.randn(1, 2, 256, 64, device=DEV).half() for _ in range(4)]
    monkeypatch.setattr(ac, 'FUSED_KV', False)
    products, dsd = [], core.dsd_tn
    monkeypatch.setattr(core, 'dsd_tn', lambda *a: (products.append(a), dsd(*a))[1])

    def grads(need):
        ts = [t.clone().requires_grad_(n) for t, n in zip((q, k, v), need)]
        del products[:]
        core(*ts, scale=0.125).backward(do)
        assert len(products) == need[1] + need[2]
        return [t.grad for t in ts]
    full = grads((True, True, True))
    for need in ((False, False, True), (False, True, False), (True, False, False), (True, False, True)):
        for n, g, f in zip(need, grads(need), full):
            assert (g is not None) == n and (not n or torch.equal(g, f))
