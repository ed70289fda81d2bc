"""Dropout on every form of the kernels, at sizes where a wave's look at 1024 keys of its rows as a whole ends in each of
its outcomes: rows kept, rows dropped, and rows in which the mask changes (those are hashed element by element, in the
dK/dV kernel in a second visit of the tile). Against the oracle with the same mask; tolerances as in
test_attention_dropout_gpu.py."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from oracle.attention_oracle import attention_bwd_oracle, attention_fwd_oracle, dropout_keep_mask

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
O_ATOL, O_RTOL, LSE_ATOL = 2e-2, 1e-2, 1e-3


def _state_with_partial_rows(p, B, H, Sq, Sk, seed):
    """A generator offset at which the mask of this shape has kept rows, dropped rows and rows that are neither."""
    for off in range(4 * 1001, 1 << 32, (1 << 20) + 12344):
        keep = dropout_keep_mask(p, seed, off, B, H, Sq, Sk).reshape(-1, Sk)
        all_, any_ = keep.all(1), keep.any(1)
        if 0.2 < keep.mean() < 0.8 and (any_ & ~all_).any() and all_.any() and (~any_).any():
            return off
    raise AssertionError("no such offset")


# Sq and Sk off the tile sizes, several spans of 1024 keys, more than 64 query tiles in the last one
@pytest.mark.parametrize("variant", [-1, 0, 8, 32])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,dtype", [
    (1, 2, 700, 2200, 128, False, torch.bfloat16), (1, 3, 1100, 1100, 64, True, torch.float16),
    (2, 1, 1537, 1537, 128, True, torch.bfloat16), (1, 1, 4400, 200, 64, False, torch.bfloat16)])
def test_dropout_on_every_form(B, H, Sq, Sk, D, causal, dtype, bias, variant):
    p, seed = 0.4, 987654321
    off = _state_with_partial_rows(p, B, H, Sq, Sk, seed)
    g = torch.Generator().manual_seed(Sq + D)
    q, k, v, go = (torch.randn(B, H, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk, Sq))
    b = torch.randn(B, 1, 1, Sk, generator=g) if bias else None
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, causal=causal, dropout=(p, seed, off), bias=b)
    ref = attention_bwd_oracle(q, k, v, go, causal=causal, dropout=(p, seed, off), bias=b)
    t = [x.to(DEV).transpose(1, 2).requires_grad_(True) for x in (q, k, v)]
    _lib.tune_set("attn.variant", variant)
    _lib.tune_set("attn_bwd.variant", 0 if variant == 0 else -1)
    try:
        if variant >= 0:                     # the form asked for is the form that runs
            st = [(_lib.ctypes.c_int64 * 3)(x.stride(0), x.stride(2), x.stride(1)) for x in t[1:]]
            assert _lib.load().fo_attn_fwd_kernel(B, H, Sq, Sk, D, *st, causal, 2 if bias else 0, 1) == variant
        o, lse = flash_attn(*t, bias=None if b is None else b.to(DEV), causal=causal, dropout_p=p, return_lse=True, dropout_state=(seed, off))
        got = torch.autograd.grad(o, t, go.to(DEV).transpose(1, 2))
        torch.cuda.synchronize()
    finally:
        _lib.tune_set("attn.variant", -1)
        _lib.tune_set("attn_bwd.variant", -1)
    err = (o.detach().transpose(1, 2).float().cpu() - o_ref).abs()
    assert float((err - (O_ATOL + O_RTOL * o_ref.abs())).max()) <= 0, f"O: max abs err {float(err.max()):.3e}"
    assert float((lse.cpu() - lse_ref).abs().max()) <= LSE_ATOL
    for name, a, r in zip(("dQ", "dK", "dV"), got, ref):
        e = (a.transpose(1, 2).float().cpu() - r).abs().max().item()
        assert e <= 2e-2 * max(1.0, r.abs().max().item()), f"{name}: error {e:.3e} vs magnitude {r.abs().max().item():.3e}"


# a bias with a query stride: whole tiles of it and ragged ones, on 16-byte boundaries and off them
@pytest.mark.parametrize("bias_dtype", ["f32", "operand"])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,dtype", [
    (1, 2, 300, 1160, 128, False, torch.bfloat16), (1, 2, 700, 700, 128, True, torch.float16), (2, 1, 333, 1201, 128, False, torch.float16),
    (1, 2, 300, 1160, 64, False, torch.float16), (1, 2, 701, 701, 64, True, torch.bfloat16)])
def test_dropout_with_a_bias_per_query(B, H, Sq, Sk, D, causal, dtype, bias_dtype):
    p, seed = 0.4, 987654321
    off = _state_with_partial_rows(p, B, H, Sq, Sk, seed)
    g = torch.Generator().manual_seed(Sq + D)
    q, k, v, go = (torch.randn(B, H, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk, Sq))
    b = torch.randn(1, H, Sq, Sk, generator=g).to(torch.float32 if bias_dtype == "f32" else dtype)
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, causal=causal, dropout=(p, seed, off), bias=b)
    ref = attention_bwd_oracle(q, k, v, go, causal=causal, dropout=(p, seed, off), bias=b)
    t = [x.to(DEV).transpose(1, 2).requires_grad_(True) for x in (q, k, v)]
    o, lse = flash_attn(*t, bias=b.to(DEV), causal=causal, dropout_p=p, return_lse=True, dropout_state=(seed, off))
    got = torch.autograd.grad(o, t, go.to(DEV).transpose(1, 2))
    torch.cuda.synchronize()
    err = (o.detach().transpose(1, 2).float().cpu() - o_ref).abs()
    assert float((err - (O_ATOL + O_RTOL * o_ref.abs())).max()) <= 0, f"O: max abs err {float(err.max()):.3e}"
    assert float((lse.cpu() - lse_ref).abs().max()) <= LSE_ATOL
    for name, a, r in zip(("dQ", "dK", "dV"), got, ref):
        e = (a.transpose(1, 2).float().cpu() - r).abs().max().item()
        assert e <= 2e-2 * max(1.0, r.abs().max().item()), f"{name}: error {e:.3e} vs magnitude {r.abs().max().item():.3e}"


# P and dS are rounded to the operand type with the factor 1 / (1 - p). Sizes: dS of a kept element is about 6e-7 without that
# factor, which fp16 rounds to multiples of 2^-24 (error 2^-24 / sqrt(12) each: 1.8 % of dQ and dK, emulated in 64 bits; with the
# factor 0.2 %), and the gradients are about 1e-5 (0.2-0.3 % from their own rounding). The general dK/dV kernel (variant 0) and the pipelined one.
@pytest.mark.parametrize("variant", [-1, 0])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias", [None, "key", "query"])
def test_small_fp16_gradients_at_a_large_dropout_p(D, bias, variant):
    p, seed, off, S = 0.9, 12345, 1 << 20, 2048      # (kept, dropped and partly dropped rows; 27 % of the elements are kept)
    g = torch.Generator().manual_seed(D)
    q, k, v, go = (torch.randn(1, 1, S, D, generator=g) for _ in range(4))
    q, k, v, go = q.half(), k.half(), v.half(), (go * (1.2e-3 / D ** 0.5)).half()
    b = None if bias is None else torch.randn(1, 1, 1 if bias == "key" else S, S, generator=g)
    keep = torch.from_numpy(dropout_keep_mask(p, seed, off, 1, 1, S, S))
    x = [t.double().requires_grad_(True) for t in (q, k, v)]
    scores = x[0] @ x[1].transpose(2, 3).contiguous() / D ** 0.5 + (0 if b is None else b.double())
    ref = torch.autograd.grad((torch.softmax(scores, -1) * keep / (1 - p)) @ x[2], x, go.double())
    t = [y.to(DEV).transpose(1, 2).requires_grad_(True) for y in (q, k, v)]
    _lib.tune_set("attn_bwd.variant", variant)
    try:
        o = flash_attn(*t, bias=None if b is None else b.to(DEV), dropout_p=p, dropout_state=(seed, off))
        got = torch.autograd.grad(o, t, go.to(DEV).transpose(1, 2))
        torch.cuda.synchronize()
    finally:
        _lib.tune_set("attn_bwd.variant", -1)
    for name, a, r in zip(("dQ", "dK", "dV"), got, ref):
        e = float((a.transpose(1, 2).cpu().double() - r).norm() / r.norm())
        assert e <= 1e-2, f"{name}: relative error {e:.2e}"
