"""Values of a bias above a causal diagonal, which no row may see, whatever they are: NaN and infinities too. Against the oracle;
tolerances as in test_attention_bias_gpu.py."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from oracle.attention_oracle import attention_fwd_oracle
from test_attention_bias_gpu import DEV, _bshd, _check

pytestmark = pytest.mark.gpu
PLAIN, PIPE = _lib.FO_ATTN_KERNEL_ROWS128, _lib.FO_ATTN_KERNEL_ROWS128_PIPE


@pytest.fixture
def use():
    def kernel(variant, pieces=-1):
        _lib.tune_set("attn.variant", variant)
        _lib.tune_set("attn.split", pieces)
    yield kernel
    kernel(-1)


def _run(q, k, v, bias, causal):
    o_ref, lse_ref = attention_fwd_oracle(q, k, v, causal=causal, bias=bias)
    on = torch.empty(bias.shape[:-1] + ((bias.shape[-1] + 7) // 8 * 8,), dtype=bias.dtype, device=DEV)[..., :bias.shape[-1]]
    on.copy_(bias)                                                           # (rows on 16-byte boundaries)
    o, lse = flash_attn(*(_bshd(x.to(DEV)) for x in (q, k, v)), bias=on, causal=causal, return_lse=True)
    torch.cuda.synchronize()
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    _check(_bshd(o), lse, [], o_ref, lse_ref, [])


@pytest.mark.parametrize("above", [float("nan"), float("inf"), float("-inf"), 3e38])
@pytest.mark.parametrize("variant,pieces", [(PLAIN, -1), (PIPE, 0), (PIPE, 2)])
@pytest.mark.parametrize("D,bias_f32", [(64, False), (64, True), (128, False)])
def test_values_above_the_diagonal_are_not_seen(D, bias_f32, variant, pieces, above, use):
    S, dtype = 333, torch.bfloat16
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(1, 2, S, D, generator=g).to(dtype) for _ in range(3))
    bias = torch.randn(1, 2, S, S, generator=g)
    bias.masked_fill_(torch.ones(S, S, dtype=torch.bool).triu(1), above)
    use(variant, pieces)
    _run(q, k, v, bias.to(torch.float32 if bias_f32 else dtype), True)
