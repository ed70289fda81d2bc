"""The compiled host path declines what is not an ordinary GPU call (csrc/host_path.cpp); the Python code then does or refuses it. On the
CPU: nothing here is an ordinary call. (Ordinary ones: test_host_path_gpu.py.)"""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from fast_ops.flash_attention.flash_attention import flash_attn, multi_head_attention
from fast_ops_amd.flash_attention import flash_attention as surface


@pytest.fixture
def host():
    return surface._host()


class Sub(torch.Tensor):
    pass


class Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_the_module_is_built(host):
    assert host is not None


@pytest.mark.parametrize("kind", ["cpu", "meta", "subclass", "none", "number", "sparse", "float32"])
def test_declined(host, kind):
    t = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)
    t = {"cpu": t, "meta": t.to("meta"), "subclass": t.as_subclass(Sub), "none": None, "number": 3, "sparse": t[0, 0].to_sparse(), "float32": t.float()}[kind]
    assert host.fwd(t, t, t, False, False, None, None, None) is None
    assert host.bwd(t, t, t, t, t, t, False, False, None, None, None) is None


def test_declined_arguments(host):
    t = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)
    assert host.fwd(t, t, t) is None and host.bwd(t) is None
    for odd in (1, None, torch.ones(2), "yes"):
        assert host.fwd(t, t, t, odd, odd, None, None, None) is None
    with Mode():
        assert host.fwd(t, t, t, False, False, None, None, None) is None


def test_who_replaces_torch_empty_sees_the_allocations(monkeypatch):
    assert surface._host() is not None
    monkeypatch.setattr(torch, "empty", lambda *a, **k: None)
    assert surface._host() is None


def test_refused_as_before():
    t = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)
    for call in (multi_head_attention, flash_attn):
        with pytest.raises(RuntimeError, match="GPU tensors"):
            call(t, t, t)
        with pytest.raises(RuntimeError, match="half-precision"):
            call(t.float(), t.float(), t.float())
        with pytest.raises(RuntimeError, match="same type"):
            call(t, t.half(), t)
