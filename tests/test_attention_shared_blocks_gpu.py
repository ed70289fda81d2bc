"""Query blocks whose keys several workgroups of the pipelined 128-row forward kernel share (attn.split: every block in two, three and
four pieces): lengths off the tile sizes, causal blocks that end before the last key, blocks too short for that many pieces, both
kinds of bias - keys masked for a whole piece among them - and dropout, with too little scratch memory, in a captured graph. Against
the oracle; tolerances as in test_attention_bias_gpu.py."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn, multi_head_attention
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention import flash_attention as surface
from oracle.attention_oracle import attention_fwd_oracle, dropout_keep_mask
from test_attention_bias_gpu import DEV, _bshd, _check

pytestmark = pytest.mark.gpu


@pytest.fixture
def split():
    def use(pieces):
        _lib.tune_set("attn.split", pieces)
        _lib.tune_set("attn.variant", _lib.FO_ATTN_KERNEL_ROWS128_PIPE)
    yield use
    _lib.tune_set("attn.split", -1)
    _lib.tune_set("attn.variant", -1)


def _kernel(q, k, v, bias, causal, drop):
    """The kernel of this call with the scratch memory that it asks for."""
    plan = surface._fwd_plan(q, k, v, (0, 2, 1, 3))
    if bias is not None:
        bias = surface._expand_bias(bias, q, plan.B, plan.H, plan.Sq, plan.Sk)
    call = (plan.B, plan.H, plan.Sq, plan.Sk, plan.D, plan.ks, plan.vs, int(causal), _lib.ctypes.byref(surface._extras(bias, drop)))
    return _lib.load().fo_attn_fwd_kernel_ex(*call, _lib.load().fo_attn_fwd_workspace_ex(*call))


@pytest.mark.parametrize("pieces", [2, 3, 4])
@pytest.mark.parametrize("form", ["none", "key", "query", "dropout", "key + dropout"])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,dtype", [
    (1, 2, 130, 200, 128, False, torch.bfloat16), (1, 1, 300, 1160, 128, False, torch.float16), (2, 1, 700, 700, 128, True, torch.bfloat16),
    (1, 1, 1000, 600, 128, True, torch.float16), (1, 2, 260, 1000, 64, False, torch.bfloat16), (1, 3, 520, 520, 64, True, torch.float16)])
def test_shared_blocks(B, H, Sq, Sk, D, causal, dtype, form, pieces, split):
    g = torch.Generator().manual_seed(Sq + Sk + D)
    q, k, v = (torch.randn(B, H, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk))
    bias, drop = None, None
    if "key" in form:
        bias = torch.randn(B, 1, 1, Sk, generator=g).to(dtype)
        if not causal:
            bias[..., Sk // 4:] = float("-inf")                      # the last piece, or pieces, see no key that counts
    if "query" in form:
        bias = torch.randn(1, H, Sq, (Sk + 7) // 8 * 8, generator=g).to(dtype)[..., :Sk]
    if "dropout" in form:
        p, seed = 0.4, 987654321
        off = next(o for o in range(4004, 1 << 32, (1 << 20) + 12344) if 0.2 < dropout_keep_mask(p, seed, o, B, H, Sq, Sk).mean() < 0.8)
        drop = (p, seed, off)
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, causal=causal, bias=bias, dropout=drop)
    dev_bias = None
    if bias is not None:
        dev_bias = torch.empty(bias.shape[:-1] + ((Sk + 7) // 8 * 8,), dtype=dtype, device=DEV)[..., :Sk]
        dev_bias.copy_(bias)
    split(pieces)
    t = [_bshd(x.to(DEV)) for x in (q, k, v)]
    kw = {} if drop is None else dict(dropout_p=drop[0], dropout_state=drop[1:])
    o, lse = flash_attn(*t, bias=dev_bias, causal=causal, return_lse=True, **kw)
    torch.cuda.synchronize()
    _check(_bshd(o), lse, [], o_ref, lse_ref, [])
    assert _kernel(*t, dev_bias, causal, drop) == _lib.FO_ATTN_KERNEL_ROWS128_PIPE + _lib.FO_ATTN_KERNEL_SHARED_BLOCKS


def test_without_the_memory_the_blocks_are_whole(monkeypatch):
    q, k, v = (torch.randn(1, 4, 2048, 128, generator=torch.Generator().manual_seed(i)).to(DEV, torch.bfloat16) for i in range(3))
    shared = multi_head_attention(q, k, v, causal=True)
    monkeypatch.setattr(surface, "_host", lambda: None)
    monkeypatch.setattr(surface, "_scratch", lambda n, device: None)
    whole = multi_head_attention(q, k, v, causal=True)
    _lib.tune_set("attn.split", 0)
    try:
        assert torch.equal(whole, multi_head_attention(q, k, v, causal=True)) and not torch.equal(whole, shared)
    finally:
        _lib.tune_set("attn.split", -1)


def test_shared_blocks_in_a_graph():
    q, k, v = (torch.randn(1, 2048, 6, 128, generator=torch.Generator().manual_seed(i)).to(DEV, torch.bfloat16) for i in range(3))
    bias = torch.zeros(1, 1, 1, 2048, device=DEV)
    call = lambda: flash_attn(q, k, v, bias=bias, causal=True, dropout_p=0.1, dropout_state=(7, 4 << 20))
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = call()
    for i in range(3):
        q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(10 + i)))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, call())
