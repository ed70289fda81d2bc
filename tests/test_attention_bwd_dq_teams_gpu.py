"""dQ from stored dS where two teams of waves share a workgroup's keys (even and odd 32-key tiles, sums added at the end): launches of the
sizes that form is chosen at (257 to 320 blocks, causal up to 768, from 1536 keys), odd and even numbers of tiles, ragged last tiles, fewer
tiles than the rings hold (causal, the first blocks), and head dims off 128 in either form. Against the path that computes the scores once more,
and the two forms against each other wherever either can run."""
import ctypes

import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn
from fast_ops_amd import _lib
from fast_ops_amd.flash_attention.flash_attention import _extras

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # H, Sq, Sk, D, causal, bias
    (144, 129, 1536, 128, False, False), (144, 256, 1537, 128, False, False), (260, 1, 1567, 128, False, False), (144, 200, 1600, 128, False, True),
    (144, 200, 1537, 128, True, False), (260, 64, 1569, 128, True, False), (24, 1700, 1536, 128, True, False), (20, 1665, 1665, 128, True, True),
    (2, 150, 20, 72, False, False), (3, 150, 33, 80, False, False), (2, 300, 95, 104, True, False), (2, 130, 1249, 112, False, False), (4, 513, 257, 96, True, False),
    (144, 200, 1569, 72, False, False), (24, 1700, 1537, 104, True, False), (144, 256, 1600, 96, False, False), (20, 1665, 1665, 80, True, False),
]

TWO_TEAMS = [c for c in CASES if c[2] >= 1536 and (c[4] or c[0] * -(-c[1] // 128) <= 320)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"H{c[0]}q{c[1]}k{c[2]}d{c[3]}{'c' if c[4] else 'f'}{'b' if c[5] else ''}")
def test_dq_teams(case, dtype):
    H, Sq, Sk, D, causal, with_bias = case
    g = torch.Generator(device=DEV).manual_seed(Sq * 7 + Sk + D)
    q, k, v, go = (torch.randn(1, n, H, D, generator=g, device=DEV).to(dtype) for n in (Sq, Sk, Sk, Sq))
    bias = torch.randn(1, H, Sq, (Sk + 15) // 16 * 16, generator=g, device=DEV).to(dtype)[..., :Sk] if with_bias else None
    extras = None if bias is None else ctypes.byref(_extras(bias.expand(1, H, Sq, Sk), None))
    t = [x.requires_grad_(True) for x in (q, k, v)]

    def backward(keep, teams=-1):
        _lib.tune_set("attn_bwd.keep_ds", keep)
        _lib.tune_set("attn_bwd.dq_teams", teams)
        try:
            ws = lib.fo_attn_bwd_workspace_ex(1, H, Sq, Sk, D, int(causal), extras)
            kernels.append(lib.fo_attn_bwd_kernels(1, H, Sq, Sk, D, int(causal), extras, ws))
            return torch.autograd.grad(flash_attn(*t, bias=bias, causal=causal), t, go)
        finally:
            _lib.tune_set("attn_bwd.keep_ds", -1)
            _lib.tune_set("attn_bwd.dq_teams", -1)

    # the same dS but for where delta's last bit (another order of its sum) rounds one to its neighbour, and one rounding of the result;
    # the absolute part is fp32's rounding of dP - delta where a query attends one key and both are equal (128 x 2^-24 x |dO.O| x |K| x scale)
    lib, kernels = _lib.load(), []
    chosen, again, one, two = backward(1), backward(0), backward(1, 1), backward(1, 2)
    assert [k & 1 for k in kernels] == [1, 0, 1, 1] and [k & 4 for k in kernels[2:]] == [0, 4]      # the forms asked for are the forms that run
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (kernels[0] & 4 == 4) == (case in TWO_TEAMS)
    # the same dS and, within a workgroup of one team, the same order: dQ differs by fp32 sums taken in two halves, rounded once
    assert torch.equal(chosen[0], (two if kernels[0] & 4 else one)[0])
    a, b = one[0].double(), two[0].double()
    assert (a - b).norm().item() <= (1e-3 if dtype == torch.bfloat16 else 1.5e-4) * b.norm().item() + 1e-6
    for name, a, b in zip(("dQ", "dK", "dV"), chosen, again):
        a, b = a.double(), b.double()
        assert bool(torch.isfinite(a).all()), name
        assert (a - b).norm().item() <= (2e-3 if dtype == torch.bfloat16 else 3e-4) * b.norm().item() + 4e-4, name
