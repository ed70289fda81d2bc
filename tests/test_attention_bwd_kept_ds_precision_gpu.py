"""How exact dQ of kept dS is, against the dQ kernel that computes the scores once more: the probabilities it is made of have
to be at least as good. (Kept dS comes from the dK/dV kernel, whose score accumulators used to start from -LSE / scale: an fp32 error of P
2.5 times as large as where the LSE joins in the exponent.)"""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention.flash_attention import attn_bwd_strided, attn_fwd_strided
from oracle.attention_oracle import attention_bwd_oracle
from test_attention_dropout_forms_gpu import _state_with_partial_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dq(t, go, keep, **kw):
    _lib.tune_set("attn_bwd.keep_ds", keep)
    _lib.tune_set("attn_bwd.split", 0)
    try:
        return torch.autograd.grad(flash_attn(*t, **kw), t[0], go)[0]
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)
        _lib.tune_set("attn_bwd.split", -1)


@pytest.mark.parametrize("H,Sq,Sk,D,causal,p,key_bias", [
    (3, 300, 1000, 128, False, 0.0, False), (3, 515, 515, 128, True, 0.0, False), (2, 333, 191, 80, False, 0.0, False), (2, 257, 300, 104, True, 0.0, False),
    (3, 300, 1000, 128, False, 0.0, True), (3, 515, 515, 128, True, 0.0, True), (2, 700, 1500, 128, False, 0.5, False),
    (3, 1100, 1100, 128, True, 0.5, False), (2, 700, 1500, 128, False, 0.5, True)])
def test_probabilities_are_the_same(H, Sq, Sk, D, causal, p, key_bias):
    """dO is 2 in one column, V and O are multiples of 1/64 there, 1 - p is a power of two: dP, delta and their difference are exact in
    either kernel, and what is left of dS is P. dQ is then the same to the bit, also in rows of which dropout keeps a part, which the dK/dV kernel
    visits twice. (bf16: the other kernel rounds P (dP - delta) to fp16 in one
    instruction, from the exact product.)"""
    dtype = torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(Sq + D)
    q, k, v = (torch.randn(1, H, n, D, generator=g, device=DEV).to(dtype) for n in (Sq, Sk, Sk))
    v = (v * 64).round() / 64
    drop = (p, 987654321, _state_with_partial_rows(p, 1, H, Sq, Sk, 987654321)) if p else None
    bias = None
    if key_bias:
        bias = torch.randn(1, 1, 1, Sk, generator=g, device=DEV)
        bias[..., Sk - Sk // 5:] = -10000.0
    o, lse = attn_fwd_strided(q, k, v, (0, 1, 2, 3), causal, None, drop, bias)
    o = (o * 64).round() / 64
    go = torch.zeros_like(o)
    go[..., 5] = 2.0
    grads = []
    _lib.tune_set("attn_bwd.split", 0)
    try:
        for keep in (1, 0):
            _lib.tune_set("attn_bwd.keep_ds", keep)
            grads.append(attn_bwd_strided(q, k, v, o, lse, go, (0, 1, 2, 3), causal, None, drop, bias))
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)
        _lib.tune_set("attn_bwd.split", -1)
    assert bool(grads[1][0].any())
    assert torch.equal(grads[0][0], grads[1][0])


@pytest.mark.parametrize("causal", [False, True])
def test_large_key_bias(causal):
    """A per-key bias that is large as a whole: the error of P is that of the exponent's terms (rel. 2^-24 of 5000 log2 e, 4e-4), of the
    order of fp16's rounding, and shows in dQ."""
    H, S, D = 4, 512, 128
    g = torch.Generator().manual_seed(7)
    q, k, v, go = (torch.randn(1, H, S, D, generator=g).to(torch.float16) for _ in range(4))
    bias = 5000.0 + torch.randn(1, 1, 1, S, generator=g)
    ref = attention_bwd_oracle(q, k, v, go, causal=causal, bias=bias, dtype=torch.float64)[0]
    t = [x.to(DEV).transpose(1, 2).requires_grad_(True) for x in (q, k, v)]
    errors = []
    for keep in (1, 0):
        dq = _dq(t, go.to(DEV).transpose(1, 2), keep, bias=bias.to(DEV), causal=causal).transpose(1, 2).double().cpu()
        errors.append((dq - ref).norm().item() / ref.norm().item())
    assert errors[0] <= 1.02 * errors[1], errors
