"""dQ from stored dS where two teams of waves share a workgroup's keys (even and odd 32-key tiles, sums added at the end): launches of the
sizes that form is chosen at (257 to 320 blocks, causal up to 768, from 1536 keys), odd and even numbers of tiles, ragged last tiles, fewer
tiles than the rings hold (causal, the first blocks), and head dims off 128 in either form. Against the path that computes the scores once more."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # H, Sq, Sk, D, causal, bias
    (144, 129, 1536, 128, False, False), (144, 256, 1537, 128, False, False), (260, 1, 1567, 128, False, False), (144, 200, 1600, 128, False, True),
    (144, 200, 1537, 128, True, False), (260, 64, 1569, 128, True, False), (24, 1700, 1536, 128, True, False), (20, 1665, 1665, 128, True, True),
    (2, 150, 20, 72, False, False), (3, 150, 33, 80, False, False), (2, 300, 95, 104, True, False), (2, 130, 1249, 112, False, False), (4, 513, 257, 96, True, False),
    (144, 200, 1569, 72, False, False), (24, 1700, 1537, 104, True, False), (144, 256, 1600, 96, False, False), (20, 1665, 1665, 80, True, False),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"H{c[0]}q{c[1]}k{c[2]}d{c[3]}{'c' if c[4] else 'f'}{'b' if c[5] else ''}")
def test_dq_teams(case, dtype):
    H, Sq, Sk, D, causal, with_bias = case
    g = torch.Generator(device=DEV).manual_seed(Sq * 7 + Sk + D)
    q, k, v, go = (torch.randn(1, n, H, D, generator=g, device=DEV).to(dtype) for n in (Sq, Sk, Sk, Sq))
    bias = torch.randn(1, H, Sq, (Sk + 15) // 16 * 16, generator=g, device=DEV).to(dtype)[..., :Sk] if with_bias else None
    t = [x.requires_grad_(True) for x in (q, k, v)]

    def backward(keep):
        _lib.tune_set("attn_bwd.keep_ds", keep)
        try:
            return torch.autograd.grad(flash_attn(*t, bias=bias, causal=causal), t, go)
        finally:
            _lib.tune_set("attn_bwd.keep_ds", -1)

    # the same dS but for where delta's last bit (another order of its sum) rounds one to its neighbour, and one rounding of the result;
    # the absolute part is fp32's rounding of dP - delta where a query attends one key and both are equal (128 x 2^-24 x |dO.O| x |K| x scale)
    for name, a, b in zip(("dQ", "dK", "dV"), backward(1), backward(0)):
        a, b = a.double(), b.double()
        assert bool(torch.isfinite(a).all()), name
        assert (a - b).norm().item() <= (2e-3 if dtype == torch.bfloat16 else 3e-4) * b.norm().item() + 4e-4, name
