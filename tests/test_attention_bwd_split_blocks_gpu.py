"""Key blocks of the backward whose query tiles several workgroups share (attn_bwd.split, where dS is kept): the sums of a
block's pieces added by the dQ launch. Every block in 2 to 4 pieces, down to pieces of one 64-query tile and blocks of fewer tiles than pieces,
against the same call with a workgroup per block: dQ, from the same dS, to the bit; dK and dV to the rounding of their fp32 sums in another
order, and of dS where rows that are partly dropped are added a second time."""
import ctypes

import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention.flash_attention import _extras
from test_attention_dropout_forms_gpu import _state_with_partial_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # B, H, Sq, Sk, D, causal, bias, dropout
    (1, 2, 64, 200, 128, False, None, 0.0), (1, 3, 129, 65, 128, False, None, 0.0), (2, 2, 321, 129, 128, False, None, 0.0),
    (1, 2, 700, 1250, 80, False, None, 0.0), (1, 2, 257, 300, 104, True, None, 0.0), (1, 3, 515, 515, 128, True, None, 0.0),
    (1, 2, 320, 900, 128, True, None, 0.0), (1, 2, 900, 320, 128, True, None, 0.0), (2, 2, 640, 384, 128, False, "key", 0.0),
    (1, 2, 577, 577, 128, True, "rows", 0.0), (1, 2, 450, 260, 128, False, "rows", 0.0), (1, 2, 385, 400, 128, True, "rows32", 0.0),
    (1, 2, 450, 128, 128, False, "rows32", 0.0), (1, 2, 1100, 1100, 128, True, None, 0.4), (1, 2, 2200, 700, 128, False, "key", 0.4),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}H{c[1]}q{c[2]}k{c[3]}d{c[4]}{'c' if c[5] else 'f'}{c[6] or ''}{c[7] or ''}")
def test_split_blocks(case, dtype):
    B, H, Sq, Sk, D, causal, bias_kind, p = case
    g = torch.Generator().manual_seed(Sq * 7 + Sk + D)
    q, k, v, go = (torch.randn(B, n, H, D, generator=g).to(dtype).to(DEV) for n in (Sq, Sk, Sk, Sq))
    bias = None
    if bias_kind == "key":
        bias = torch.randn(1, 1, 1, Sk, generator=g).to(DEV)
    elif bias_kind is not None:
        wide = torch.randn(1, H, Sq, (Sk + 15) // 16 * 16, generator=g).to(torch.float32 if bias_kind == "rows32" else dtype)
        bias = wide.to(DEV)[..., :Sk]
    state = _state_with_partial_rows(p, B, H, Sq, Sk, 987654321) if p else None
    t = [x.requires_grad_(True) for x in (q, k, v)]
    drop = (p, 987654321, state) if p else None
    extras = None if bias is None and not p else ctypes.byref(_extras(None if bias is None else bias.expand(B, H, Sq, Sk), drop))

    lib = _lib.load()

    def backward(split):
        _lib.tune_set("attn_bwd.split", split)
        # the form asked for is the form that runs
        ws = lib.fo_attn_bwd_workspace_ex(B, H, Sq, Sk, D, int(causal), extras)
        shares = split > 0 and Sq > 64
        assert lib.fo_attn_bwd_kernels(B, H, Sq, Sk, D, int(causal), extras, ws) & 3 == (3 if shares else 1)
        assert (ws - whole_ws) % (B * H * 128 * 1024) == 0 and (ws > whole_ws) == shares
        o = flash_attn(*t, bias=bias, causal=causal, dropout_p=p, dropout_state=(987654321, state) if p else None)
        return torch.autograd.grad(o, t, go)

    _lib.tune_set("attn_bwd.keep_ds", 1)       # (also where it does not pay)
    try:
        _lib.tune_set("attn_bwd.split", 0)
        whole_ws = lib.fo_attn_bwd_workspace_ex(B, H, Sq, Sk, D, int(causal), extras)
        whole = backward(0)
        runs = {n: backward(n) for n in (2, 3, 4)}
    finally:
        _lib.tune_set("attn_bwd.keep_ds", -1)
        _lib.tune_set("attn_bwd.split", -1)
    for n, grads in runs.items():
        for name, a, b in zip(("dQ", "dK", "dV"), grads, whole):
            assert bool(torch.isfinite(a).all()), (n, name)
            if name == "dQ" and not p:
                assert torch.equal(a, b), (n, name)
                continue
            # sums that differ by fp32 rounding, each rounded to the operand type: now and then to its neighbour
            a, b = a.double(), b.double()
            assert (a - b).norm().item() <= (1e-3 if dtype == torch.bfloat16 else 1.5e-4) * b.norm().item(), (n, name)


# The library's own plans (256 compute units): blocks left whole beside blocks in pieces, and pieces of unequal length. (What such plans are: test_attention_bwd_plan.py)
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [
    (1, 12, 3072, 3072, 128, True), (1, 4, 4096, 4096, 128, True), (1, 5, 2050, 3000, 128, True), (1, 12, 3072, 3072, 128, False), (1, 12, 3072, 3072, 96, True)])
def test_chosen_plans(B, H, Sq, Sk, D, causal):
    lib = _lib.load()
    ws = lib.fo_attn_bwd_workspace_ex(B, H, Sq, Sk, D, int(causal), None)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert lib.fo_attn_bwd_kernels(B, H, Sq, Sk, D, int(causal), None, ws) & 3 == 3
    g = torch.Generator(device=DEV).manual_seed(Sq + D)
    t = [torch.randn(B, n, H, D, generator=g, device=DEV).to(torch.bfloat16).requires_grad_(True) for n in (Sq, Sk, Sk)]
    go = torch.randn(B, Sq, H, D, generator=g, device=DEV).to(torch.bfloat16)
    shared = torch.autograd.grad(flash_attn(*t, causal=causal), t, go)
    _lib.tune_set("attn_bwd.split", 0)
    try:
        whole = torch.autograd.grad(flash_attn(*t, causal=causal), t, go)
    finally:
        _lib.tune_set("attn_bwd.split", -1)
    for name, a, b in zip(("dK", "dV"), shared[1:], whole[1:]):
        a, b = a.double(), b.double()
        assert (a - b).norm().item() <= 1e-3 * b.norm().item(), name      # (as above)
    a, b = shared[0].double(), whole[0].double()                            # (sharing blocks may bring two teams to dQ)
    assert (a - b).norm().item() <= 1e-3 * b.norm().item()
