"""The forward of few query rows over many keys: the keys of a row block dealt to waves and workgroups. Sizes at the edges of
the 32-key tiles and the 32-row blocks, keys in slices of a larger cache, multi-query K/V, one and several workgroups per
row block; against the oracle with the forward's tolerances."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn, multi_head_attention
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention import flash_attention as surface
from oracle.attention_oracle import attention_fwd_oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
O_ATOL, O_RTOL, LSE_ATOL = 2e-2, 1e-2, 1e-3


@pytest.mark.parametrize("split", [-1, 1, 2, 7])
@pytest.mark.parametrize("B,H,Sq,Sk,D,dtype,multi_query", [
    (1, 3, 1, 128, 64, torch.float16, False), (2, 5, 1, 129, 128, torch.bfloat16, False), (1, 2, 32, 1000, 64, torch.bfloat16, False),
    (3, 4, 17, 545, 128, torch.float16, False), (2, 8, 1, 4097, 128, torch.bfloat16, True), (1, 12, 5, 700, 64, torch.float16, True),
    (9, 1, 2, 300, 128, torch.bfloat16, False)])
def test_decode_against_oracle(B, H, Sq, Sk, D, dtype, multi_query, split):
    g = torch.Generator().manual_seed(Sk + D)
    Hk = 1 if multi_query else H
    q = torch.randn(B, H, Sq, D, generator=g).to(dtype)
    # what lies behind the filled part of the cache must not count
    cache = [torch.cat([torch.randn(B, Hk, Sk, D, generator=g), torch.full((B, Hk, 40, D), float("nan"))], dim=2).to(dtype) for _ in range(2)]
    # moving row maxima: the last keys score far above the others
    cache[0][:, :, Sk - 3:Sk] *= 6
    k, v = (t[:, :, :Sk].expand(B, H, Sk, D) for t in cache)
    o_ref, lse_ref = attention_fwd_oracle(q, k, v)
    kd, vd = (t.to(DEV)[:, :, :Sk].expand(B, H, Sk, D) for t in cache)
    assert _lib.tune_set("attn.decode_split", split) is None
    try:
        o, lse = multi_head_attention(q.to(DEV), kd, vd, return_lse=True)
        I3 = lambda t: (_lib.ctypes.c_int64 * 3)(*t.stride()[:3])
        assert _lib.load().fo_attn_fwd_kernel(B, H, Sq, Sk, D, I3(kd), I3(vd), 0, 0, 0) == _lib.FO_ATTN_KERNEL_DECODE
        torch.cuda.synchronize()
    finally:
        _lib.tune_set("attn.decode_split", -1)
    err = (o.float().cpu() - o_ref).abs()
    assert float((err - (O_ATOL + O_RTOL * o_ref.abs())).max()) <= 0, f"O: max abs err {float(err.max()):.3e}"
    assert float((lse.cpu() - lse_ref).abs().max()) <= LSE_ATOL


# K holds -inf in the column that Q holds 1 in: those keys score -inf. They fill whole tiles of some waves, all tiles of some
# waves, and (split 7) all tiles of some workgroups; the other keys of the row count as if they were alone.
@pytest.mark.parametrize("split", [-1, 1, 7])
@pytest.mark.parametrize("Sq,Sk,D,dtype,live", [(1, 2000, 128, torch.bfloat16, (0, 1000)), (8, 4096, 64, torch.float16, (0, 196)),
                                                (32, 1000, 64, torch.bfloat16, (600, 650)), (1, 1025, 128, torch.float16, (1024, 1025))])
def test_decode_with_keys_that_score_minus_infinity(Sq, Sk, D, dtype, live, split):
    g = torch.Generator().manual_seed(Sk)
    q, k, v = (torch.randn(2, 3, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk))
    q[..., 0] = 1
    k[..., 0] = float("-inf")
    k[:, :, live[0]:live[1], 0] = 0
    o_ref, lse_ref = attention_fwd_oracle(q, k, v)
    _lib.tune_set("attn.decode_split", split)
    try:
        o, lse = multi_head_attention(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True)
        torch.cuda.synchronize()
    finally:
        _lib.tune_set("attn.decode_split", -1)
    err = (o.float().cpu() - o_ref).abs()
    assert float((err - (O_ATOL + O_RTOL * o_ref.abs())).max()) <= 0, f"O: max abs err {float(err.max()):.3e}"
    assert float((lse.cpu() - lse_ref).abs().max()) <= LSE_ATOL


# The merge takes four splits with the references and eight at a time behind them: the edges of both, and the most there are.
@pytest.mark.parametrize("split", [3, 4, 5, 12, 13, 20, 64])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16)])
def test_decode_merges_any_number_of_splits(split, D, dtype):
    test_decode_against_oracle(1, 3, 2, 65 * 32 + 1, D, dtype, False, split)


# a shape's first call may fall into a time when another kernel, or fewer workgroups per row block, were asked for
@pytest.mark.parametrize("key,value", [("attn.variant", 0), ("attn.decode_split", 1)])
def test_workspace_follows_what_is_asked_for(key, value):
    q, k, v = (torch.randn(1, 4, n, 128, device=DEV, dtype=torch.bfloat16) for n in (1, 4352 + len(key), 4352 + len(key)))
    dims = (0, 1, 2, 3)
    _lib.tune_set(key, value)
    try:
        assert surface._fwd_plan(q, k, v, dims).ws_bytes == 0
    finally:
        _lib.tune_set(key, -1)
    assert surface._fwd_plan(q, k, v, dims).ws_bytes > 0


# the [B, S, H, D] layout, several rows per head; keys that all heads share with values of their own (only the keys' head stride is 0)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Sq,Sk,shared_keys", [(1, 1500, False), (7, 801, False), (1, 1500, True), (5, 801, True)])
def test_decode_layouts(Sq, Sk, D, shared_keys):
    g = torch.Generator().manual_seed(Sk + D)
    q, k, v = (torch.randn(2, n, 6, D, generator=g).to(torch.bfloat16) for n in (Sq, Sk, Sk))
    if shared_keys:
        k = k[:, :, :1].expand(2, Sk, 6, D)
    o_ref, lse_ref = attention_fwd_oracle(*(t.transpose(1, 2) for t in (q, k, v)))
    kd = k[:, :, :1].contiguous().to(DEV).expand(2, Sk, 6, D) if shared_keys else k.to(DEV)
    o, lse = flash_attn(q.to(DEV), kd, v.to(DEV), return_lse=True)
    I3 = lambda t: (_lib.ctypes.c_int64 * 3)(t.stride(0), t.stride(2), t.stride(1))
    assert _lib.load().fo_attn_fwd_kernel(2, 6, Sq, Sk, D, I3(kd), I3(v), 0, 0, 0) == _lib.FO_ATTN_KERNEL_DECODE
    torch.cuda.synchronize()
    err = (o.transpose(1, 2).float().cpu() - o_ref).abs()
    assert float((err - (O_ATOL + O_RTOL * o_ref.abs())).max()) <= 0, f"O: max abs err {float(err.max()):.3e}"
    assert float((lse.cpu() - lse_ref).abs().max()) <= LSE_ATOL
