"""The backward that keeps dS (fo_attn_bwd_ws with the workspace fo_attn_bwd_workspace asks for): dQ as one product of the dS that
the dK/dV kernel leaves in memory. Lengths around its tiles (32 keys, 64 queries) and blocks (128 of either), both mask kinds,
every bias form and dropout with rows that are partly dropped. The workspace holds NaN before the call, so that a value the call reads
without having written it shows. Against the oracle, and against the path that computes the scores once more (the same call
with the small workspace)."""
import ctypes
import math

import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention.flash_attention import attn_bwd_strided, attn_fwd_strided
from oracle.attention_oracle import attention_bwd_oracle
from test_attention_dropout_forms_gpu import _state_with_partial_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # B, H, Sq, Sk, D, causal, bias, dropout
    (1, 2, 1, 1, 128, False, None, 0.0), (2, 3, 31, 33, 128, False, None, 0.0), (1, 2, 64, 128, 128, True, None, 0.0),
    (1, 2, 65, 129, 128, True, None, 0.0), (2, 2, 129, 65, 128, True, None, 0.0), (1, 3, 300, 700, 128, True, None, 0.0),
    (1, 2, 700, 300, 128, True, None, 0.0), (2, 2, 193, 1250, 80, False, None, 0.0), (1, 2, 333, 191, 104, True, None, 0.0),
    (1, 2, 257, 95, 72, False, None, 0.0), (1, 2, 640, 640, 128, True, "key", 0.0), (1, 2, 130, 97, 128, False, "key", 0.0),
    (1, 3, 385, 385, 128, True, "rows", 0.0), (1, 2, 97, 224, 128, False, "rows", 0.0), (1, 2, 321, 352, 128, False, "rows32", 0.0),
    (1, 2, 200, 160, 128, True, "rows32", 0.0), (1, 2, 1100, 1100, 128, True, None, 0.4), (1, 2, 700, 2200, 128, False, "key", 0.4),
    (2, 1, 1537, 1537, 128, True, None, 0.4), (1, 1, 4400, 200, 128, False, None, 0.4),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}H{c[1]}q{c[2]}k{c[3]}d{c[4]}{'c' if c[5] else 'f'}{c[6] or ''}{c[7] or ''}")
def test_kept_ds(case, dtype):
    B, H, Sq, Sk, D, causal, bias_kind, p = case
    g = torch.Generator().manual_seed(Sq * 7 + Sk + D)
    q, k, v, go = (torch.randn(B, H, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk, Sq))
    bias = None
    if bias_kind == "key":
        bias = torch.randn(1, 1, 1, Sk, generator=g)
        bias[..., Sk - Sk // 4:] = -10000.0
    elif bias_kind is not None:                # rows on 16-byte boundaries, NaN behind the last key
        wide = torch.full((1, H, Sq, (Sk + 15) // 16 * 16), math.nan, dtype=torch.float32 if bias_kind == "rows32" else dtype)
        wide[..., :Sk] = torch.randn(1, H, Sq, Sk, generator=g).to(wide.dtype)
        bias = wide[..., :Sk]
    seed = 987654321
    drop = (p, seed, _state_with_partial_rows(p, B, H, Sq, Sk, seed)) if p else None
    ref = attention_bwd_oracle(q, k, v, go, causal=causal, dropout=drop, bias=None if bias is None else bias.float())
    bias_dev = None if bias is None else (wide.to(DEV)[..., :Sk] if bias_kind != "key" else bias.to(DEV))
    t = [x.to(DEV) for x in (q, k, v)]
    o, lse = flash_attn(*(x.transpose(1, 2) for x in t), bias=bias_dev, causal=causal, dropout_p=p, return_lse=True, dropout_state=None if drop is None else drop[1:])
    o, go_dev = o.transpose(1, 2).contiguous(), go.to(DEV)
    lib, ex = _lib.load(), None
    if bias is not None or drop is not None:
        from fast_ops_amd.flash_attention.flash_attention import _extras
        ex = ctypes.byref(_extras(None if bias is None else bias_dev.expand(B, H, Sq, Sk), drop))
    I3, P64 = ctypes.c_int64 * 3, ctypes.POINTER(ctypes.c_int64)

    def backward(ws_bytes):
        ws = torch.full((ws_bytes,), 255, dtype=torch.uint8, device=DEV)
        grads = [torch.full_like(x, math.nan) for x in t]
        arrays = [I3(*x.stride()[:3]) for x in (*t, o, go_dev, *grads)]
        strides = (P64 * 8)(*[ctypes.cast(a, P64) for a in arrays])
        status = lib.fo_attn_bwd_ws(*(x.data_ptr() for x in (*t, o, go_dev, lse, *grads)), B, H, Sq, Sk, D, strides, 1.0 / math.sqrt(D), int(causal),
                                    _lib.FO_DTYPE_BF16 if dtype == torch.bfloat16 else _lib.FO_DTYPE_F16, ex, ws.data_ptr(), ws_bytes,
                                    torch.cuda.current_stream().cuda_stream)
        assert status == 0
        torch.cuda.synchronize()
        return grads

    small = 8 * B * H * Sq
    _lib.tune_set("attn_bwd.keep_ds", 1)       # (also where it does not pay)
    try:
        full = lib.fo_attn_bwd_workspace(B, H, Sq, Sk, D)
        assert full >= small + 2 * B * H * Sq * Sk
        assert [lib.fo_attn_bwd_kernels(B, H, Sq, Sk, D, int(causal), ex, n) & 1 for n in (full, small)] == [1, 0]      # the forms that run below
        kept, again = backward(full), backward(small)
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)
    assert lib.fo_attn_bwd_ws(*([t[0].data_ptr()] * 9), B, H, Sq, Sk, D, (P64 * 8)(), 1.0, 0, 0, None, t[0].data_ptr(), small - 1, None) != 0
    for name, a, r in zip(("dQ", "dK", "dV"), kept, ref):
        e = (a.float().cpu() - r).abs().max().item()
        assert e <= 2e-2 * max(1.0, r.abs().max().item()), f"{name}: error {e:.3e} vs magnitude {r.abs().max().item():.3e}"
    # delta is summed in another order than in the dQ kernel: dS differs by its rounding (2^-8 in bf16) here and there. Where a
    # query attends one key, dS is a difference of two equal sums of 128 products: its fp32 rounding, 128 x 2^-24 x |dO.O| (below
    # 100 here), times K and the scale (below 0.5), is all there is of dQ.
    for name, a, b in zip(("dQ", "dK", "dV"), kept, again):
        a, b = a.float(), b.float()
        assert (a - b).norm().item() <= (2e-3 if dtype == torch.bfloat16 else 3e-4) * b.norm().item() + 4e-4, name


def _operand(kind, n, H, D, g, dtype):
    """[1, n, H, D] in memory as a program may have it: dense; one of three in a packed projection; heads first; one head seen by all;
    rows as far apart as 32-bit offsets do not reach."""
    new = lambda *shape: torch.randn(*shape, generator=g, device=DEV).to(dtype)
    if kind == "packed":
        return new(1, n, 3, H, D)[:, :, 1]
    if kind == "heads_first":
        return new(1, H, n, D).transpose(1, 2)
    if kind == "one_head":
        return new(1, n, 1, D).expand(1, n, H, D)
    if kind == "far_rows":
        far = torch.empty(((n - 1) << 23) + H * D, dtype=dtype, device=DEV).as_strided((1, n, H, D), (8, 1 << 23, D, 1))
        return far.copy_(new(1, n, H, D))
    return new(1, n, H, D)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_kind,kv_kind,go_kind,Sq,Sk,D,causal,p", [
    ("packed", "packed", "dense", 300, 300, 128, True, 0.0), ("heads_first", "heads_first", "heads_first", 129, 391, 80, False, 0.0),
    ("dense", "one_head", "packed", 257, 450, 128, False, 0.0), ("packed", "one_head", "heads_first", 333, 97, 104, True, 0.0),
    ("dense", "far_rows", "dense", 200, 70, 128, False, 0.0), ("far_rows", "dense", "far_rows", 70, 333, 96, False, 0.0),
    ("far_rows", "far_rows", "packed", 75, 75, 128, True, 0.4), ("packed", "heads_first", "heads_first", 700, 1300, 128, False, 0.4)])
def test_layouts(q_kind, kv_kind, go_kind, Sq, Sk, D, causal, p, dtype):
    H = 3
    g = torch.Generator(device=DEV).manual_seed(Sq + Sk + D)
    q, k, v = (_operand(kind, n, H, D, g, dtype) for kind, n in ((q_kind, Sq), (kv_kind, Sk), (kv_kind, Sk)))
    go = _operand(go_kind, Sq, H, D, g, dtype)
    drop = (p, 987654321, 4004 * 17) if p else None
    o, lse = attn_fwd_strided(q, k, v, (0, 2, 1, 3), causal, None, drop)
    grads = {}
    try:
        for keep, split in ((0, 0), (1, 0), (1, 3)):
            _lib.tune_set("attn_bwd.keep_ds", keep)
            _lib.tune_set("attn_bwd.split", split)
            grads[keep, split] = attn_bwd_strided(q, k, v, o, lse, go, (0, 2, 1, 3), causal, None, drop)
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)
        _lib.tune_set("attn_bwd.split", -1)
    for form in ((1, 0), (1, 3)):
        for name, a, b in zip(("dQ", "dK", "dV"), grads[form], grads[0, 0]):
            a, b = a.double(), b.double()
            assert bool(torch.isfinite(a).all()), (form, name)
            assert (a - b).norm().item() <= (2e-3 if dtype == torch.bfloat16 else 3e-4) * b.norm().item() + 4e-4, (form, name)      # (as above)
