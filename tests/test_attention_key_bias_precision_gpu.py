"""How exact the scores of the pipelined forward kernels are with a large bias per key, read off the LSE of rows that see one key each:
the bias joins a finished score, so that a score is rounded at the bias' size once and not once per product. And a bias that may be
anything at keys that a causal row does not see. Against float64."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
KERNELS = [_lib.FO_ATTN_KERNEL_ROWS128_PIPE, _lib.FO_ATTN_KERNEL_ROWS256_W4]


@pytest.fixture
def use():
    yield lambda variant: _lib.tune_set("attn.variant", variant)
    _lib.tune_set("attn.variant", -1)


@pytest.mark.parametrize("variant", KERNELS)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dropout_p", [0.0, 0.1])
def test_lse_of_one_key(D, variant, dropout_p, use):
    B, H, S = 24, 1, 512
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(B, S, H, D, generator=g).to(torch.bfloat16) for _ in range(3))
    at = torch.randint(0, S, (B,), generator=g)
    value = (520.0 + 200.0 * torch.rand(B, generator=g)) * (1 - 2 * (torch.arange(B) % 2))
    bias = torch.full((B, 1, 1, S), float("-inf"))
    bias[torch.arange(B), 0, 0, at] = value
    use(variant)
    _, lse = flash_attn(q.to(DEV), k.to(DEV), v.to(DEV), bias=bias.to(DEV), return_lse=True, dropout_p=dropout_p, dropout_state=(3, 8))
    exact = (q[:, :, 0].double() * k[torch.arange(B), at].double()).sum(-1) / D ** 0.5 + value.double()[:, None]
    off = float((lse[:, 0].double().cpu() - exact).square().mean().sqrt())
    # roundings of half an ulp at most, 0.29 ulp rms, here in nat: of bias / scale and of the score (below 8192 / sqrt(128) or 8192 / 8: 1.25e-5 and
    # 1.25e-5, or none and 1.8e-5), in base 2 (below 1024: 1.2e-5), of the LSE (below 1024: 1.8e-5). Together 2.8e-5. Rounded once per
    # product, the score alone takes it to 4.2e-5.
    assert off <= 3.4e-5, off


@pytest.mark.parametrize("variant", [_lib.FO_ATTN_KERNEL_ROWS128] + KERNELS)
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 3e38])
@pytest.mark.parametrize("D", [64, 128])
def test_keys_that_no_row_sees(D, value, variant, use):
    Sq, Sk = 300, 520
    g = torch.Generator().manual_seed(D)
    q = torch.randn(1, Sq, 2, D, generator=g).to(DEV, torch.bfloat16)
    k, v = (torch.randn(1, Sk, 2, D, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    bias = torch.randn(1, 1, 1, Sk, generator=g).to(DEV)
    use(variant)

    def same(some, as_these):
        # (other rows of a wave - ones that do see such a key, or stand past the end - may move the reference of all of them, against which
        # P is rounded: to 2^-9 of itself, as is O, whose values stay below 4)
        assert torch.allclose(some[0].float(), as_these[0].float(), rtol=2.0 ** -7, atol=2.0 ** -6)
        assert torch.allclose(some[1], as_these[1], rtol=0, atol=1e-4)

    want = flash_attn(q, k, v, bias=bias, causal=True, return_lse=True)
    bias[..., 20:] = value
    few = flash_attn(q, k, v, bias=bias, causal=True, return_lse=True)
    same((few[0][:, :20], few[1][:, :, :20]), (want[0][:, :20], want[1][:, :, :20]))
    bias[..., 20:Sq] = torch.randn(Sq - 20, generator=g).to(DEV)
    some = flash_attn(q, k, v, bias=bias, causal=True, return_lse=True)
    bias[..., Sq:] = 0.0
    same(some, flash_attn(q, k, v, bias=bias, causal=True, return_lse=True))
