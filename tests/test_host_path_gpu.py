"""Calls through the compiled host path (csrc/host_path.cpp) against the same calls through the Python code: the same kernels with the
same arguments, so the same bits, in tensors of the same layout, over layouts, types, head dims, lengths, masks, both kinds of bias and
dropout; and what the library refuses is refused with the same words."""
import pytest
import torch

from fast_ops.flash_attention.flash_attention import flash_attn, multi_head_attention
from fast_ops_amd.flash_attention import flash_attention as surface

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _both(monkeypatch, call):
    assert surface._host() is not None
    here = call()
    with monkeypatch.context() as m:
        m.setattr(surface, "_host", lambda: None)
        there = call()
    return here, there


def _tensors(layout, B, H, Sq, Sk, D, dtype, bshd):
    g = torch.Generator(device=DEV).manual_seed(Sq + Sk + D)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)
    shape = lambda h, n: (B, n, h, D) if bshd else (B, h, n, D)
    if layout == "packed":
        x = r(B, Sq, 3, H, D)
        q, k, v = (x[:, :, i] if bshd else x[:, :, i].transpose(1, 2) for i in range(3))
    elif layout == "one kv head":
        q, k, v = r(*shape(H, Sq)), r(*shape(1, Sk)).expand(shape(H, Sk)), r(*shape(1, Sk)).expand(shape(H, Sk))
    elif layout == "transposed":
        q, k, v = (r(*((B, h, n, D) if bshd else (B, n, h, D))).transpose(1, 2) for h, n in ((H, Sq), (H, Sk), (H, Sk)))
    else:
        q, k, v = r(*shape(H, Sq)), r(*shape(H, Sk)), r(*shape(H, Sk))
    return q, k, v, r(*shape(H, Sq))


@pytest.mark.parametrize("layout,B,H,Sq,Sk,D,dtype", [
    ("dense", 2, 3, 130, 200, 64, torch.float16), ("dense", 1, 2, 1, 700, 128, torch.bfloat16), ("dense", 1, 1, 7, 5, 8, torch.bfloat16),
    ("packed", 2, 2, 257, 257, 128, torch.bfloat16), ("one kv head", 2, 4, 33, 300, 64, torch.bfloat16), ("transposed", 1, 3, 100, 90, 80, torch.float16),
    ("dense", 1, 4, 2048, 2048, 128, torch.bfloat16)])
@pytest.mark.parametrize("surface_of", ["bhsd", "bshd"])
@pytest.mark.parametrize("form", ["plain", "causal", "scaled", "key bias", "row bias", "fp32 bias", "dropout", "bias + dropout"])
def test_the_same_bits(layout, B, H, Sq, Sk, D, dtype, surface_of, form, monkeypatch):
    bshd = surface_of == "bshd"
    if "bias" in form and not bshd:
        pytest.skip("flash_attn's option")
    q, k, v, go = _tensors(layout, B, H, Sq, Sk, D, dtype, bshd)
    kw = {"causal": form in ("causal", "bias + dropout")}
    if form == "scaled":
        kw["softmax_scale"] = 0.3
    if form == "key bias":
        kw["bias"] = torch.randn(B, 1, 1, Sk, device=DEV).to(dtype)
    if form in ("row bias", "bias + dropout"):
        kw["bias"] = torch.randn(1, H, Sq, Sk, device=DEV).to(dtype)
    if form == "fp32 bias":
        kw["bias"] = torch.randn(B, 1, Sq, Sk, device=DEV)
    if "dropout" in form:
        kw.update(dropout_p=0.3, dropout_state=(5, (1 << 33) + 4004))
    call = flash_attn if bshd else multi_head_attention

    def run():
        t = [x.detach().requires_grad_(True) for x in (q, k, v)]
        with torch.no_grad():
            plain = call(q, k, v, return_lse=True, **kw)
        o, lse = call(*t, return_lse=True, **kw)
        return [*plain, o.detach(), lse, *torch.autograd.grad(o, t, go)]

    for a, b in zip(*_both(monkeypatch, run)):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and a.device == b.device and not a.requires_grad
        assert torch.equal(a, b)
    # the host path itself took both
    extras = [kw["causal"], kw.get("softmax_scale"), (kw["dropout_p"], *kw["dropout_state"]) if "dropout" in form else None, kw.get("bias")]
    taken = surface._host().fwd(q, k, v, bshd, *extras)
    assert taken is not None and surface._host().bwd(q, k, v, *taken, go, bshd, *extras) is not None


def test_refused_with_the_same_words(monkeypatch):
    q = torch.randn(1, 2, 16, 64, device=DEV).half()
    off = torch.randn(1 + 2 * 16 * 64, device=DEV).half()[1:].view(1, 2, 16, 64)          # not on a 16-byte boundary
    bad = [(off, q, q, {}), (q.float(), q.float(), q.float(), {}), (q, q[..., :32], q, {}), (q, q, q, dict(softmax_scale=-1.0)),
           (torch.randn(1, 2, 16, 136, device=DEV).half(),) * 3 + ({},), (q[..., ::2], q[..., ::2], q[..., ::2], {})]

    def words():
        out = []
        for a, b, c, kw in bad:
            with pytest.raises(RuntimeError) as e:
                multi_head_attention(a, b, c, **kw)
            out.append(str(e.value))
        return out

    here, there = _both(monkeypatch, words)
    assert here == there


def test_a_backward_without_any_memory():
    # its outputs find none: that is refused with torch's own error, and the next call is as ever (less than all: test_scratch_memory.py)
    q, k, v, go = _tensors("dense", 1, 4, 2048, 2048, 128, torch.bfloat16, False)
    t = [x.requires_grad_(True) for x in (q, k, v)]
    o = multi_head_attention(*t, causal=True)
    want = torch.autograd.grad(o, t, go, retain_graph=True)
    rest = []
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-4)          # nothing new
    try:
        # nor what is left of blocks that other tensors hold a part of
        size = 1 << 26
        while size >= 512:
            try:
                rest.append(torch.empty(size, dtype=torch.uint8, device=q.device))
            except torch.OutOfMemoryError:
                size //= 2
        with pytest.raises(torch.OutOfMemoryError):
            torch.autograd.grad(o, t, go, retain_graph=True)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        rest.clear()
    for a, b in zip(torch.autograd.grad(o, t, go), want):
        assert torch.allclose(a.float(), b.float(), atol=2e-2, rtol=2e-2)
