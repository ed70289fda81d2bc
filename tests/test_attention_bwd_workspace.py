"""How much workspace the attention backward asks for (fo_attn_bwd_workspace_ex): dS only for the calls that keep it."""
import ctypes
import math
import time

import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention import flash_attention as fa
from fast_ops_amd.flash_attention.flash_attention import _AttnExtras

DEV = "cuda:0"
B, H, S = 1, 8, 2048
ROWS = 8 * B * H * S
DS = 2 * B * H * S * S
PART = 2 * 128 * 128 * 4                # one block's fp32 sums of dK and dV


def _asked(D, causal=False, bias=None, p=0.0):
    """bias: (address, strides, dtype)"""
    ex = _AttnExtras()
    if bias is not None:
        ex.bias, ex.bias_strides, ex.bias_dtype = bias[0], (ctypes.c_int64 * 3)(*bias[1]), bias[2]
    ex.dropout_p = p
    return _lib.load().fo_attn_bwd_workspace_ex(B, H, S, S, D, int(causal), ctypes.byref(ex))


KEY = (0x1000, (S, 0, 0), _lib.FO_DTYPE_F32)
TILES = (0x1000, (0, S * S, S), _lib.FO_DTYPE_BF16)
TILES32 = (0x1000, (0, S * S, S), _lib.FO_DTYPE_F32)
ODD_ROWS = (0x1000, (0, S * (S + 1), S + 1), _lib.FO_DTYPE_BF16)
ODD_BASE = (0x1002, (0, S * S, S), _lib.FO_DTYPE_BF16)


@pytest.mark.parametrize("causal", [False, True])
def test_calls_that_keep_ds(causal):
    for D, bias, p in [(128, None, 0.0), (128, None, 0.3), (72, None, 0.0), (96, None, 0.0), (120, None, 0.0), (128, KEY, 0.0), (128, KEY, 0.3),
                       (128, TILES, 0.0), (128, TILES32, 0.0)]:
        n = _asked(D, causal, bias, p)
        assert n >= ROWS + DS and (n - ROWS - DS) % (B * H * PART) == 0, (D, bias, p)
        assert n <= _lib.load().fo_attn_bwd_workspace(B, H, S, S, D)
    assert _lib.load().fo_attn_bwd_workspace_ex(B, H, S, S, 128, int(causal), None) == _asked(128, causal)


@pytest.mark.parametrize("causal", [False, True])
def test_calls_that_do_not(causal):
    for D, bias, p in [(96, None, 0.3), (72, KEY, 0.0), (104, TILES, 0.0), (128, TILES, 0.3), (128, ODD_ROWS, 0.0), (128, ODD_BASE, 0.0), (64, None, 0.0),
                       (32, KEY, 0.3)]:
        assert _asked(D, causal, bias, p) == ROWS, (D, bias, p)
    _lib.tune_set("attn_bwd.variant", 0)
    try:
        assert _asked(128, causal) == ROWS
    finally:
        _lib.tune_set("attn_bwd.variant", -1)


def test_sizes_at_which_ds_is_kept():
    """... are those where that is faster: with many heads only while the caches hold dS, with very many not beyond 512 keys."""
    lib = _lib.load()
    def kept(heads, Sq, Sk, D, causal=0, bias=None, p=0.0):
        ex = _AttnExtras()
        if bias is not None:
            ex.bias, ex.bias_strides, ex.bias_dtype = bias[0], (ctypes.c_int64 * 3)(*bias[1]), bias[2]
        ex.dropout_p = p
        room = lib.fo_attn_bwd_workspace(1, heads, Sq, Sk, D)
        got = lib.fo_attn_bwd_kernels(1, heads, Sq, Sk, D, causal, ctypes.byref(ex), room)
        assert got == lib.fo_attn_bwd_kernels(1, heads, Sq, Sk, D, causal, ctypes.byref(ex), 4 << 30)      # no call can use more
        return got & 1

    for shape in [(96, 2048, 4096, 128), (4, 1, 1536, 128), (160, 384, 2048, 128), (192, 1024, 1024, 104), (192, 2048, 2048, 128), (192, 1024, 1024, 128, 1),
                  (384, 512, 512, 128), (48, 3072, 4096, 96), (128, 128, 4096, 72), (384, 1024, 1024, 128, 0, None, 0.1), (384, 1024, 1024, 128, 1, TILES)]:
        assert kept(*shape) == 1, shape
    for shape in [(192, 384, 4096, 128), (192, 2048, 2048, 128, 1), (256, 128, 4096, 128), (384, 384, 2048, 104), (512, 256, 1024, 128),
                  (384, 1024, 1024, 128, 0, KEY), (16, 1024, 1024, 128), (2, 4096, 1535, 96),
                  (128, 384, 4096, 96), (160, 256, 2048, 96), (384, 1024, 1024, 72), (129, 1024, 1024, 96)]:
        assert kept(*shape) == 0, shape
    _lib.tune_set("attn_bwd.keep_ds", 1)
    try:
        assert kept(384, 1024, 1024, 72) == 1
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)


def test_shapes_that_are_not_taken():
    ask = lambda *a: (_lib.load().fo_attn_bwd_workspace_ex(*a, 0, None), _lib.load().fo_attn_bwd_workspace(*a))
    big = 2 ** 31 - 1
    for shape in [(0, 1, 1, 1, 64), (1, -1, 1, 1, 64), (1, 1, 0, 1, 64), (1, 1, 1, 0, 64), (1, 1, 1, 1, 12), (1, 1, 1, 1, 136), (big, big, big, 1, 128)]:
        assert ask(*shape) == (0, 0), shape


def test_shapes_in_turn_do_not_plan_anew():
    """Layers of several shapes ask in turn: how the key blocks are shared is worked out once for each, not at every call (2 to 40 us)."""
    ask = _lib.load().fo_attn_bwd_workspace_ex

    def per_call(lengths):
        best = math.inf
        for _ in range(7):
            t0 = time.perf_counter()
            for _ in range(100):
                for n in lengths:
                    ask(1, 4, n, n, 128, 1, None)
            best = min(best, (time.perf_counter() - t0) / (100 * len(lengths)))
        return best

    one = per_call([8192] * 4)
    assert per_call([8192, 7168, 6144, 5120]) < 3.0 * one


def test_a_workspace_that_does_not_fit_is_not_asked_for_again(monkeypatch):
    plan = fa._BwdPlan()
    plan.B, plan.H, plan.Sq, plan.Sk, plan.D, plan.ws_bytes = 1, 4, S, S, 128, {}
    full = _lib.load().fo_attn_bwd_workspace_ex(1, 4, S, S, 128, 1, None)
    rows = 8 * 4 * S
    ds = rows + 2 * 4 * S * S
    assert full > ds
    asked, fits = [], [rows]

    def empty(n, **kw):
        asked.append(n)
        if n > fits[0]:
            raise torch.OutOfMemoryError("no room")
        return n

    monkeypatch.setattr(fa.torch, "empty", empty)
    call = lambda: fa._bwd_workspace(plan, True, None, None, None, "cpu")
    assert call() == rows and asked == [full, ds, rows]
    asked.clear()
    for _ in range(fa._BWD_WS_RETRY):
        assert call() == rows
    assert set(asked) == {rows}
    asked.clear()
    fits[0] = ds
    assert call() == ds and asked == [full, ds]
    assert call() == ds and asked == [full, ds, ds]
    fits[0] = rows                       # less than before
    assert call() == rows and asked == [full, ds, ds, ds, rows]
    fits[0] = 0
    with pytest.raises(torch.OutOfMemoryError):
        call()


@pytest.mark.gpu
@pytest.mark.parametrize("room", ["dS", "rows"])
def test_backward_without_room(monkeypatch, room):
    """The gradients of a call whose workspace does not fit: with room for dS alone dQ is the same to the bit (and every block of
    keys whole), with room for the rows' values alone the call is the one that computes the scores again."""
    g = torch.Generator(device=DEV).manual_seed(5)
    t = [torch.randn(1, S, 4, 128, generator=g, device=DEV).to(torch.bfloat16).requires_grad_(True) for _ in range(3)]
    go = torch.randn(1, S, 4, 128, generator=g, device=DEV).to(torch.bfloat16)
    backward = lambda: torch.autograd.grad(flash_attn(*t, causal=True), t, go)
    full = _lib.load().fo_attn_bwd_workspace_ex(1, 4, S, S, 128, 1, None)
    ds = 8 * 4 * S + 2 * 4 * S * S
    assert full > ds
    free = backward()
    _lib.tune_set("attn_bwd.keep_ds" if room == "rows" else "attn_bwd.split", 0)
    try:
        expected = backward()
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)
        _lib.tune_set("attn_bwd.split", -1)
    real, refused = torch.empty, []

    def empty(*a, **kw):
        if kw.get("dtype") == torch.uint8 and a[0] > (ds if room == "dS" else ds - 1):
            refused.append(a[0])
            raise torch.OutOfMemoryError("no room")
        return real(*a, **kw)

    monkeypatch.setattr(fa.torch, "empty", empty)
    got = [backward() for _ in range(3)]
    monkeypatch.undo()
    assert refused == ([full] if room == "dS" else [full, ds])       # by the first call alone
    for grads in got:
        for a, b in zip(grads, expected):
            assert torch.equal(a, b)
    if room == "dS":
        assert torch.equal(got[0][0], free[0]) and not torch.equal(got[0][1], free[1])
    _lib.tune_set("attn_bwd.split", -1)      # (a new plan for whoever comes next)


@pytest.mark.gpu
@pytest.mark.parametrize("D,bias,p", [(96, None, 0.3), (96, "key", 0.0), (128, "rows", 0.3), (128, None, 0.0)])
def test_memory_of_a_backward(D, bias, p):
    g = torch.Generator(device=DEV).manual_seed(D)
    q, k, v, go = (torch.randn(B, S, H, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(4))
    if bias == "key":
        bias = torch.randn(B, 1, 1, S, generator=g, device=DEV)
    elif bias is not None:
        bias = torch.randn(1, 1, S, S, generator=g, device=DEV).to(torch.bfloat16)
    t = [x.requires_grad_(True) for x in (q, k, v)]
    o = flash_attn(*t, bias=bias, dropout_p=p, dropout_state=(1, 4) if p else None)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    torch.autograd.grad(o, t, go)
    torch.cuda.synchronize()
    used = torch.cuda.max_memory_allocated() - before
    grads = 3 * q.numel() * 2
    kept = D == 128 and bias is None
    assert (used >= grads + ROWS + DS) == kept, used
    if not kept:
        assert used <= grads + ROWS + (1 << 20), used
