"""Rows all of whose keys carry a large finite mask value (-1e9, -1e30, -1e38): in fp32 every score of such a row is that value, so that O is
the mean of V over its keys and the LSE the value, whichever kernel a call gets and whatever stands before them - keys removed with
-inf, or nothing -, and a key that counts further on takes the whole row. And values above a causal diagonal, which no row may see: NaN
and infinities too. Against the oracle; tolerances of O as in test_attention_bias_gpu.py; the LSE has a few roundings of its own size."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from oracle.attention_oracle import attention_fwd_oracle
from test_attention_bias_gpu import DEV, _bshd, _check

pytestmark = pytest.mark.gpu
PLAIN, PIPE, W4 = _lib.FO_ATTN_KERNEL_ROWS128, _lib.FO_ATTN_KERNEL_ROWS128_PIPE, _lib.FO_ATTN_KERNEL_ROWS256_W4


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
    big = lse_ref.abs() > 1e4
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    # (four roundings: the value times log2 e, the score, the sum with log2 of the row sum, that times ln 2)
    assert float(((lse.cpu() - lse_ref).abs() / lse_ref.abs().clamp(min=1e-30))[big].max() if big.any() else 0.0) <= 4 * 2.0 ** -24
    _check(_bshd(o), torch.where(big, lse_ref, lse.cpu()), [], o_ref, lse_ref, [])


def _mask(shape, Sk, value, form, dtype):
    """Over the last dimension: every third row (or head, batch) as the form says, the others without a mask."""
    b = torch.zeros(shape)
    if form == "all":
        b[..., ::3, :] = value
    elif form == "behind removed keys":
        b[..., ::3, :] = value
        b[..., ::3, :Sk // 3] = float("-inf")
    elif form == "two values":
        b[..., ::3, :] = 2 * value
        b[..., ::3, 1::2] = value
    elif form == "a key at the end":
        b[..., ::3, :] = value
        b[..., ::3, Sk - 3] = 0.0
    return b.to(dtype)


FORMS = ["all", "behind removed keys", "two values", "a key at the end"]
VALUES = [-1e9, -1e30, -1e38]


@pytest.mark.parametrize("value", VALUES)
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("variant,pieces", [(PLAIN, -1), (PIPE, 0), (PIPE, 2), (PIPE, 3)])
@pytest.mark.parametrize("D,bias_f32,dtype", [(128, False, torch.bfloat16), (64, False, torch.bfloat16), (64, True, torch.float16)])
@pytest.mark.parametrize("Sq,Sk", [(130, 200), (140, 712)])
def test_bias_per_query(Sq, Sk, D, bias_f32, dtype, variant, pieces, form, value, use):
    g = torch.Generator().manual_seed(Sk + D)
    q, k, v = (torch.randn(1, 2, n, D, generator=g).to(dtype) for n in (Sq, Sk, Sk))
    use(variant, pieces)
    _run(q, k, v, _mask((1, 2, Sq, Sk), Sk, value, form, torch.float32 if bias_f32 else dtype), False)


@pytest.mark.parametrize("value", VALUES)
@pytest.mark.parametrize("variant,pieces", [(PLAIN, -1), (PIPE, 0), (PIPE, 2)])
@pytest.mark.parametrize("D", [64, 128])
def test_left_padding_under_a_causal_mask(D, variant, pieces, value, use):
    S, pad, dtype = 700, 150, torch.bfloat16
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(2, 2, S, D, generator=g).to(dtype) for _ in range(3))
    bias = torch.zeros(2, 1, S, S)
    bias[1, :, :, :pad] = value
    use(variant, pieces)
    _run(q, k, v, bias.to(dtype), True)


# (a bias per key is held divided by softmax_scale: beyond 3.4e38 times that it counts as -inf)
@pytest.mark.parametrize("value", [-1e9, -1e30, -1e36])
@pytest.mark.parametrize("causal,form", [(False, f) for f in FORMS] + [(True, f) for f in FORMS if f != "behind removed keys"])      # (there the first rows see no key)
@pytest.mark.parametrize("variant,pieces", [(PLAIN, -1), (PIPE, 0), (PIPE, 2), (PIPE, 3), (W4, -1)])
@pytest.mark.parametrize("D,bias_f32,dtype", [(128, False, torch.bfloat16), (64, False, torch.bfloat16), (64, True, torch.float16)])
def test_bias_per_key(causal, D, bias_f32, dtype, variant, pieces, form, value, use):
    S = 520
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(4, 1, S, D, generator=g).to(dtype) for _ in range(3))
    use(variant, pieces)
    _run(q, k, v, _mask((4, S), S, value, form, torch.float32 if bias_f32 else dtype).view(4, 1, 1, S), causal)


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
