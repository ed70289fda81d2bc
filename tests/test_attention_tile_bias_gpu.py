"""A bias with a query stride whose tiles are copied into LDS (rows on 16-byte boundaries, a whole number of 16-byte pieces):
several whole tiles and ragged last ones, rows longer than the keys with NaN behind them, keys masked with -inf at either
end, broadcasting over batch and heads, and calls next to the rule's lines that the general kernels take. Against the
oracle; tolerances as in test_attention_bias_gpu.py."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention import flash_attention as surface
from oracle.attention_oracle import attention_bwd_oracle, attention_fwd_oracle
from test_attention_bias_gpu import DEV, _bshd, _check

pytestmark = pytest.mark.gpu


# (the last four: keys that are no whole number of 16-byte pieces)
@pytest.mark.parametrize("B,H,Sq,Sk", [(2, 2, 449, 456), (1, 3, 577, 584), (1, 2, 640, 640), (1, 2, 130, 8), (1, 1, 333, 1030), (2, 1, 300, 333), (1, 2, 515, 1021), (2, 1, 1021, 771)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias_f32", [False, True])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("causal,dtype", [(False, torch.float16), (True, torch.bfloat16), (False, torch.bfloat16)])
def test_tile_bias(B, H, Sq, Sk, D, bias_f32, packed, causal, dtype):
    g = torch.Generator().manual_seed(Sq + Sk + D)
    q, k, v, go = (torch.randn(B, H, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk, Sq))
    bias = (2.0 * torch.randn(1 if B == 2 else B, H, Sq, Sk, generator=g)).to(torch.float32 if bias_f32 else dtype)
    if not causal:
        bias[:, :, Sq // 2:, :Sk // 3] = float("-inf")        # whole tiles and parts of one, left ...
    bias[:, :, ::3, Sk - Sk // 4:] = float("-inf")            # ... and right padding
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, causal=causal, bias=bias)
    ref = attention_bwd_oracle(q, k, v, go, causal=causal, bias=bias)
    pad = -Sk % 8 + 8
    wide = torch.full(bias.shape[:-1] + (Sk + pad,), float("nan"), dtype=bias.dtype, device=DEV)
    wide[..., :Sk] = bias.to(DEV)
    if packed:                                                # rows without a gap: copied first where they are off 16-byte boundaries
        wide = bias.to(DEV)
    t = [_bshd(x.to(DEV)).requires_grad_(True) for x in (q, k, v)]
    o, lse = flash_attn(*t, bias=wide[..., :Sk], causal=causal, return_lse=True)
    got = torch.autograd.grad(o, t, _bshd(go.to(DEV)))
    torch.cuda.synchronize()
    _check(_bshd(o), lse, [_bshd(x) for x in got], o_ref, lse_ref, ref)


# Rows whose whole bias is large: only its difference to the LSE counts, which fp32 holds exactly here. Error of P and dS in fp16
# 2^-11 / sqrt(3) each, the same of the results: 5e-4 together. (Scores summed at the ulp of bias / scale: dQ 2e-3 to 1e-2.) dK and dV:
# and that of LSE / scale rounded to fp32 once, up to |LSE| 2^-24 of P. The LSE is given, rounded to fp32 once.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias_f32", [False, True])
@pytest.mark.parametrize("causal", [False, True])
def test_gradients_of_rows_with_a_large_bias(D, bias_f32, causal):
    S, scale = 456, D ** -0.5
    g = torch.Generator().manual_seed(D)
    q, k, v, go = (torch.randn(1, 2, S, D, generator=g).half() for _ in range(4))
    bias = torch.randn(1, 2, S, S, generator=g) - 1e5 if bias_f32 else torch.full((1, 2, S, S), -3e4).half()
    x = [t.double() for t in (q, k, v, go)]
    s = x[0] @ x[1].transpose(2, 3).contiguous() * scale + bias.double()
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool).triu(1), float("-inf"))
    lse = torch.logsumexp(s, -1).float()
    p = torch.exp(s - lse.double()[..., None])
    o = (p @ x[2]).half()
    ds = p * (x[3] @ x[2].transpose(2, 3).contiguous() - (x[3] * o.double()).sum(-1, keepdim=True)) * scale
    ref = (ds @ x[1], ds.transpose(2, 3).contiguous() @ x[0], p.transpose(2, 3).contiguous() @ x[3])
    d = [t.to(DEV) for t in (q, k, v, o, lse, go, bias)]
    got = surface.attn_bwd_strided(*d[:6], (0, 1, 2, 3), causal, scale, None, d[6])
    torch.cuda.synchronize()
    for name, a, r in zip(("dQ", "dK", "dV"), got, ref):
        e = float((a.cpu().double() - r).norm() / r.norm())
        assert e <= 1e-3 + (0 if name == "dQ" else float(lse.abs().max()) * 2.0 ** -24), f"{name}: relative error {e:.2e}"


# one to three query tiles, the last of them whole or not: where the first tiles' copies and the last ones' hand-overs meet
@pytest.mark.parametrize("Sq,Sk", [(33, 64), (64, 128), (65, 136), (128, 260), (192, 128)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias_f32", [False, True])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_bias_few_query_tiles(Sq, Sk, D, bias_f32, causal):
    test_tile_bias(1, 2, Sq, Sk, D, bias_f32, False, causal, torch.bfloat16)


# (the packed rows of 1021 elements are copied into aligned ones, by the forward and by the backward)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_no_copy_of_the_bias_lives_from_forward_to_backward(dtype):
    g = torch.Generator().manual_seed(5)
    t = [torch.randn(1, 1021, 4, 64, generator=g).to(dtype).to(DEV).requires_grad_(True) for _ in range(3)]
    bias = torch.randn(1, 4, 1021, 1021, generator=g).to(dtype).to(DEV)
    assert surface._aligned_bias(bias, t[0], t[1], False) is not bias and surface._aligned_bias(bias, t[0], t[1], True) is not bias
    before = torch.cuda.memory_allocated()
    o = flash_attn(*t, bias=bias)
    assert torch.cuda.memory_allocated() - before < bias.numel() * bias.element_size() // 2      # O and the LSE: an eighth of a copy
    torch.autograd.grad(o, t, torch.ones_like(o))


def test_bias_is_read_in_place_where_a_copy_finds_no_memory(monkeypatch):
    empty = torch.empty

    def no_room(*args, **kw):
        if args and isinstance(args[0], tuple) and args[0][-1] == 1024:
            raise torch.OutOfMemoryError("no room for the copy")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", no_room)
    test_tile_bias(1, 2, 515, 1021, 64, False, True, True, torch.bfloat16)


# few rows over many keys are copied for the forward, many rows over few keys are not (the copy costs more than it gains)
@pytest.mark.parametrize("B,H,S,bias_f32,copied", [(1, 4, 1021, True, True), (1, 64, 1021, True, False), (1, 64, 1021, False, False),
                                                   (1, 32, 1021, False, True), (1, 4, 725, True, False), (1, 4, 515, False, False), (1, 4, 725, False, True)])
def test_bias_rows_are_copied_where_that_gains(B, H, S, bias_f32, copied):
    g = torch.Generator(device=DEV).manual_seed(S)
    t = [torch.randn(B, S, H, 64, generator=g, device=DEV).to(torch.bfloat16) for _ in range(3)]
    bias = torch.randn(B, H, S, S, generator=g, device=DEV).to(torch.float32 if bias_f32 else torch.bfloat16)
    rows = surface._aligned_bias(bias, t[0], t[1], False)
    assert (rows is not bias) == copied
    assert torch.equal(rows, bias)
    if bias_f32 == (S > 515):                                  # (where the backward's line lies)
        assert surface._aligned_bias(bias, t[0], t[1], True) is not bias


def _unaligned_bias(form, B, H, S, dtype, g):
    if form == "heads":                                        # one bias for all heads, expanded
        return torch.randn(B, 1, S, S, generator=g).to(dtype).to(DEV).expand(B, H, S, S)
    if form == "batch":
        return torch.randn(1, H, S, S, generator=g).to(dtype).to(DEV)
    if form == "transposed":                                   # heads outside of the batch
        return torch.randn(H, B, S, S, generator=g).to(dtype).to(DEV).transpose(0, 1)
    return torch.randn(B, H, S, S + 15, generator=g).to(dtype).to(DEV)[..., 1:S + 1]      # rows and their base off 16 bytes


# the layouts a bias can come in before it is copied, and the calls whose other kernels read the copy: dropout, narrow head dims
@pytest.mark.parametrize("form", ["heads", "batch", "transposed", "sliced"])
@pytest.mark.parametrize("D,drop,bias_f32,causal", [(64, 0.0, False, True), (128, 0.0, True, False), (128, 0.3, False, False), (64, 0.3, True, True), (80, 0.0, False, False)])
def test_copied_bias_in_every_layout(form, D, drop, bias_f32, causal):
    B, H, S, dtype, state = 2, 2, 901, torch.bfloat16, (987654321, 4 << 20)
    g = torch.Generator().manual_seed(D + len(form))
    q, k, v, go = (torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4))
    bias = _unaligned_bias(form, B, H, S, torch.float32 if bias_f32 else dtype, g)
    t = [_bshd(x.to(DEV)).requires_grad_(True) for x in (q, k, v)]
    for backward in (False, True):
        rows = surface._aligned_bias(bias, t[0], t[1], backward)
        assert rows is not bias and torch.equal(rows.expand(bias.shape), bias)
        assert rows.data_ptr() % 16 == 0 and all(s * rows.element_size() % 16 == 0 for s in rows.stride()[:3])
        assert rows.numel() * (H if form == "heads" else 1) == bias.numel()
    opts = dict(causal=causal, dropout=(drop, *state)) if drop else dict(causal=causal)
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, bias=bias.cpu(), **opts)
    ref = attention_bwd_oracle(q, k, v, go, bias=bias.cpu(), **opts)
    call = lambda: flash_attn(*t, bias=bias, causal=causal, return_lse=True, dropout_p=drop, dropout_state=state if drop else None)
    with torch.no_grad():
        o_eval, _ = call()
    o, lse = call()
    got = torch.autograd.grad(o, t, _bshd(go.to(DEV)))
    torch.cuda.synchronize()
    assert torch.equal(o, o_eval)
    _check(_bshd(o), lse, [_bshd(x) for x in got], o_ref, lse_ref, ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 1, 1, 1), (2, 3, 5, 7), (1, 2, 33, 257), (2, 1, 3, 16)])
def test_rows_of_the_copy(B, H, Sq, Sk, dtype):
    bias = torch.randn(B, H, Sq, Sk + 3, device=DEV).to(dtype)[..., 2:Sk + 2]
    size, n = bias.element_size(), 16 // bias.element_size()
    row = -(-Sk // n) * n
    out = torch.full((B * H * Sq + 1, row), float("nan"), dtype=dtype, device=DEV)       # (a row behind the last that stays as it is)
    st = (_lib.ctypes.c_int64 * 3)(*bias.stride()[:3])
    assert _lib.load().fo_attn_bias_rows(bias.data_ptr(), st, size, B, H, Sq, Sk, out.data_ptr(), row, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(out[:-1, :Sk], bias.reshape(-1, Sk)) and bool((out[:-1, Sk:] == 0).all()) and bool(out[-1].isnan().all())
