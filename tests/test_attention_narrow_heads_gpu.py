"""Head dims below the 64 and 128 columns the kernels are laid out for, over enough tiles that the copies which leave the
columns past head_dim alone follow those that zero them (the first tiles), up to ragged last tiles. Rows are wider than head_dim and hold NaN there:
a column read past head_dim shows. Against the oracle; criterion as in test_attention_bwd_gpu.py."""
import math

import pytest
import torch

from fast_ops.flash_attention.flash_attention import multi_head_attention
from oracle.attention_oracle import attention_bwd_oracle, attention_fwd_oracle
from test_attention_bwd_gpu import DEV, _check, _half_precision_torch, _inputs

pytestmark = pytest.mark.gpu


# 32, 64, 96 and 128 computed columns, the first and the last head_dim of each; tiles: several whole ones, a ragged one
@pytest.mark.parametrize("D", [8, 32, 40, 56, 72, 80, 96, 104, 120])
@pytest.mark.parametrize("Sq,Sk,causal,dtype", [(449, 333, False, torch.bfloat16), (577, 577, True, torch.float16), (384, 640, True, torch.bfloat16)])
def test_narrow_heads(D, Sq, Sk, causal, dtype):
    q, k, v, go = _inputs(1, 3, Sq, Sk, D, dtype, seed=D + Sq)
    sc = 1.0 / math.sqrt(D)
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, causal=causal)
    ref = attention_bwd_oracle(q, k, v, go, causal=causal)
    pt = _half_precision_torch(q, k, v, go, causal, sc)

    def wide(t):
        w = torch.full(t.shape[:-1] + (D + 8,), float("nan"), dtype=dtype, device=DEV)
        w[..., :D] = t.to(DEV)
        return w[..., :D]

    t = [wide(x).requires_grad_(True) for x in (q, k, v)]
    o, lse = multi_head_attention(*t, causal=causal, return_lse=True)
    got = torch.autograd.grad(o, t, wide(go))
    torch.cuda.synchronize()
    err = (o.detach().float().cpu() - o_ref).abs()
    assert float((err - (2e-2 + 1e-2 * o_ref.abs())).max()) <= 0, f"O: max abs err {float(err.max()):.3e}"
    assert float((lse.cpu() - lse_ref).abs().max()) <= 1e-3
    _check(got, ref, pt, f"D{D} Sq{Sq} Sk{Sk} causal={causal}")
