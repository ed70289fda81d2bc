"""Dropout on every form of the kernels, at sizes where a wave's look at 1024 keys of its rows as a whole ends in each of
its outcomes: rows kept, rows dropped, and rows in which the mask changes (those are hashed element by element, in the
dK/dV kernel in a second visit of the tile). Against the oracle with the same mask; tolerances as in
test_attention_dropout_gpu.py."""
import numpy as np
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


def _verdicts(first, seed, threshold):
    """The kernels' look at aligned blocks of 128 indices as a whole (dropout_block<7>): 0 dropped, 1 kept, 2 neither."""
    x = ((first ^ np.uint32(seed)) & np.uint32(0xFFFFFF80)).astype(np.uint32)
    y = (x ^ (x >> 4)) & np.uint32(0xFFFFFF80)
    z0 = ((y ^ np.uint32(0xDEADBEEF)) & np.uint32(0xFFFFFF80)) + (y << 5)
    a0, a1 = z0 >> 13, (z0 + np.uint32(33 * 127)) >> 13
    w0, w1, t = a0 ^ (a0 >> 11), a1 ^ (a1 >> 11), threshold >> 13
    return np.where((w0 > t) & (w1 > t), 1, np.where((w0 < t) & (w1 < t), 0, 2))


def _partly_dropped_block(p, seed):
    """The first index of an aligned block of 128 of which 32 to 96 are kept."""
    threshold = np.uint32(int(np.float32(p) * np.float32(4294967295)))
    for chunk in range(0, 1 << 32, 1 << 28):
        first = (np.arange(1 << 21, dtype=np.uint32) << np.uint32(7)) + np.uint32(chunk)
        for x in first[_verdicts(first, seed, threshold) == 2]:
            if 32 <= dropout_keep_mask(p, seed, int(x), 1, 1, 1, 128).sum() <= 96:
                return int(x)
    raise AssertionError("no such block")


# Rows of the dropout mask that are neither kept nor dropped over a workgroup's 128 keys take part in the dK/dV kernel's tile of
# gathered rows only: what they contribute is shown to be more than the tolerance forgives. Two keys: more than the 64 rows that fit
# that tile, so that it is worked on several times, and taken up again in the middle of a tile of rows. (block: which 128 keys.)
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (64, torch.float16), (128, torch.float16)])
@pytest.mark.parametrize("Sq,Sk,row,block,causal", [(300, 300, 200, 0, True), (300, 300, 290, 1, True), (300, 300, 77, 0, True),
                                                    (200, 520, 150, 3, False), (700, 2, 100, 0, False), (700, 2, 301, 0, True)])
def test_gathered_rows_of_the_key_gradients(Sq, Sk, row, block, causal, D, dtype):
    p, seed, B, H = 0.4, 987654321, 1, 2
    k_, scale = 1 / (1 - p), D ** -0.5
    off = (_partly_dropped_block(p, seed) - ((Sq + row) * Sk + 128 * block)) % (1 << 32)      # in the second head
    keep = torch.from_numpy(dropout_keep_mask(p, seed, off, B, H, Sq, Sk))
    seen = torch.ones(Sq, Sk, dtype=torch.bool)
    if causal:
        seen = seen.tril()
    g = torch.Generator().manual_seed(Sq + D)
    q, k, v, go = (torch.randn(B, H, n, D, generator=g) for n in (Sq, Sk, Sk, Sq))
    if Sk == 2:                                               # (the block lies over 64 rows)
        row += int(keep[0, 1, row:].any(-1).nonzero()[0])
    here = torch.nonzero(keep[0, 1, row] & seen[row])[:, 0]
    here = here[(here >= 128 * block) & (here < 128 * block + 128)]
    q[0, 1, row] = k[0, 1, here[len(here) // 2]] * (5.7 / D ** 0.5)       # about half of the row's probability on one of these keys
    q, k, v, go = (t.to(dtype) for t in (q, k, v, go))
    ref = attention_bwd_oracle(q, k, v, go, causal=causal, dropout=(p, seed, off))
    tol = [2e-2 * max(1.0, r.abs().max().item()) for r in ref]

    # what the gathered rows contribute
    threshold = np.uint32(int(np.float32(p) * np.float32(4294967295)))
    first = ((off + np.arange(H * Sq, dtype=np.int64)[:, None] * Sk + np.arange(0, Sk, 128)[None]) % (1 << 32)).astype(np.uint32)
    a, b = (_verdicts(f, seed, threshold) for f in (first, first + np.uint32(127)))
    mixed = torch.from_numpy((a != b) | (a == 2)).reshape(H, Sq, -1)
    assert mixed[1, row, block] and (Sk > 2 or mixed[1].sum() > 64)
    of_rows = (mixed.repeat_interleave(128, -1)[..., :Sk] & keep[0] & seen).float()
    scores = (q.float() @ k.float().transpose(2, 3).contiguous() * scale).masked_fill(~seen, float("-inf"))
    pz = torch.softmax(scores, -1) * of_rows * k_
    missing_v = pz.transpose(2, 3).contiguous() @ go.float()
    missing_k = (pz * (go.float() @ v.float().transpose(2, 3).contiguous())).transpose(2, 3).contiguous() @ q.float() * scale
    assert missing_k.abs().max() > 4 * tol[1] and missing_v.abs().max() > 4 * tol[2]

    t = [x.to(DEV).transpose(1, 2).requires_grad_(True) for x in (q, k, v)]
    o = flash_attn(*t, causal=causal, dropout_p=p, dropout_state=(seed, off))
    got = torch.autograd.grad(o, t, go.to(DEV).transpose(1, 2))
    torch.cuda.synchronize()
    for name, x, r, lim in zip(("dQ", "dK", "dV"), got, ref, tol):
        e = (x.transpose(1, 2).float().cpu() - r).abs().max().item()
        assert e <= lim, f"{name}: error {e:.3e} vs {lim:.3e}"
