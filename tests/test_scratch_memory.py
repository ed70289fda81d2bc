"""Scratch memory that does not fit: a call does without, or with less, and so do the calls after it for a while, since a request that fails
makes the caching allocator give its cached blocks back. In the Python code, with an allocation that fails by hand, and in the compiled
host path, with a limit on what the process may allocate."""
import contextlib
import threading

import pytest
import torch

from fast_ops_amd.flash_attention import flash_attention as surface
from fast_ops.flash_attention.flash_attention import multi_head_attention

DEV = "cuda:0"


def test_a_forward_does_not_ask_again(monkeypatch):
    asked, fits = [], [100]

    def empty(n, **kw):
        asked.append(n)
        if n > fits[0]:
            raise torch.OutOfMemoryError("no room")
        return n

    monkeypatch.setattr(surface, "_refused", threading.local())
    monkeypatch.setattr(surface.torch, "empty", empty)
    assert surface._scratch(500, "a") is None and asked == [500]
    assert surface._scratch(50, "a") == 50 and surface._scratch(400, "b") is None          # less, and another device, are asked for
    assert surface._scratch(500, "a") is None and asked == [500, 50, 400, 500]             # (the last refusal counts)
    asked.clear()
    for i in range(surface._FWD_WS_RETRY):
        assert surface._scratch(500 + i, "a") is None
    assert asked == []
    fits[0] = 1000
    assert surface._scratch(500, "a") == 500 and asked == [500]
    # a thread's refusals are its own
    fits[0] = 0
    assert surface._scratch(500, "a") is None
    fits[0] = 1000
    got = []
    t = threading.Thread(target=lambda: got.append(surface._scratch(500, "a")))
    t.start()
    t.join()
    assert got == [500] and surface._scratch(500, "a") is None


@contextlib.contextmanager
def _room(n_bytes):
    """Lets the process have so many bytes more than what lives in it, and nothing that other tensors' blocks have left."""
    rest, total = [], torch.cuda.get_device_properties(0).total_memory
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-4)
    try:
        size = 1 << 26
        while size >= 512:
            try:
                rest.append(torch.empty(size, dtype=torch.uint8, device=DEV))
            except torch.OutOfMemoryError:
                size //= 2
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + n_bytes) / total)
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        rest.clear()


def _ooms():
    return torch.cuda.memory_stats()["num_ooms"]


def _in_a_thread(call):
    """What a thread was refused is its own: every test starts without any."""
    out = []

    def run():
        try:
            torch.cuda.set_device(0)
            call()
        except BaseException as e:
            out.append(e)

    t = threading.Thread(target=run)
    t.start()
    t.join()
    if out:
        raise out[0]


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["compiled", "Python"])
def test_a_forward_without_room(path, monkeypatch):
    # 8 MiB of O and 128 KiB of LSE: blocks of 20 and 2 MiB. The shared blocks' sums want more than what is left.
    q, k, v = (torch.randn(1, 4, 8192, 128, generator=torch.Generator().manual_seed(i)).to(DEV, torch.bfloat16) for i in range(3))
    few = [t[:, :2, :1024] for t in (q, k, v)]
    want, few_want = multi_head_attention(q, k, v, causal=True), multi_head_attention(*few, causal=True)
    host = surface._host()
    assert host is not None
    calls = []
    if path == "Python":
        monkeypatch.setattr(surface, "_host", lambda: None)
    else:                                                      # (declined calls would go to the Python code)
        monkeypatch.setattr(surface, "_fwd_plan", lambda *a: calls.append(a))

    def run():
        with _room(30 << 20):
            before = _ooms()
            got = multi_head_attention(q, k, v, causal=True)
            assert _ooms() == before + 1
            small = multi_head_attention(*few, causal=True)     # (whose sums fit)
            again = multi_head_attention(q, k, v, causal=True)
            assert _ooms() == before + 1
        assert torch.equal(got, again) and torch.equal(small, few_want)
        assert torch.allclose(got.float(), want.float(), atol=2e-2, rtol=1e-2)
        for _ in range(surface._FWD_WS_RETRY - 1):
            assert torch.equal(multi_head_attention(q, k, v, causal=True), got)
        assert torch.equal(multi_head_attention(q, k, v, causal=True), want)      # asked again, and given

    _in_a_thread(run)
    assert calls == []


@pytest.mark.gpu
def test_a_backward_without_room(monkeypatch):
    # 2 MiB of dQ, dK and dV each, one block of 20 MiB; dS would be 32 MiB, the rows' values are 64 KiB
    q, k, v, go = (torch.randn(1, 4, 2048, 128, generator=torch.Generator().manual_seed(i)).to(DEV, torch.bfloat16) for i in range(4))
    t = [x.requires_grad_(True) for x in (q, k, v)]
    o, lse = multi_head_attention(*t, causal=True, return_lse=True)
    args = [x.detach() for x in (q, k, v, o, lse, go)] + [False, True, None, None, None]
    host = surface._host()
    want = torch.autograd.grad(o, t, go, retain_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(host.bwd(*args), want))          # the compiled path takes it
    few = [x[:, :1, :256].contiguous() for x in args[:6]]
    asked = []
    monkeypatch.setattr(surface, "_BWD_PLANS", {})                                # (which keep what did not fit for a while)

    def run():
        with _room(24 << 20):
            before = _ooms()
            assert host.bwd(*args) is None and _ooms() == before + 1              # declined
            assert host.bwd(*args) is None and _ooms() == before + 1              # not asked for again
            got = surface.attn_bwd_strided(*args[:6], (0, 1, 2, 3), True, None)   # the Python code: less memory
            assert _ooms() > before + 1
            asked.append(_ooms())
            again = surface.attn_bwd_strided(*args[:6], (0, 1, 2, 3), True, None)
            assert _ooms() == asked[0]
            assert host.bwd(*few, *args[6:]) is not None                          # a smaller one is taken
        for a, b, c in zip(got, again, want):
            assert torch.equal(a, b) and torch.allclose(a.float(), c.float(), atol=2e-2, rtol=2e-2)
        for _ in range(256 - 3):
            assert host.bwd(*args) is None
        assert all(torch.equal(a, b) for a, b in zip(host.bwd(*args), want))

    _in_a_thread(run)
