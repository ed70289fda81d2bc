"""FlashAttention forward for MI355X: drop-in for ``fast_ops.flash_attention.flash_attention``.

``multi_head_attention(Q, K, V)`` keeps the reference call (fast_ops/flash_attention/flash_attention.py:48-77):
[B, H, M, D] queries, [B, H, N, D] keys and values, fp16 or bf16, returns [B, H, M, D]. The reference's CUDA kernel
behind that call is unfinished and returns zeros (flash_attention_fwd.cu:120-151,158); this one computes
softmax(scale * Q K^T + mask) V with the numerics of the reference's working Triton forward
(flash_attention_triton.py:128-255) and can return the logsumexp that forward also produces (:255,771). The backward
the reference leaves unimplemented (flash_attention.py:40-45) is implemented too, after the Triton backward
(flash_attention_triton.py:832-958), so ``FlashAttentionFunction`` is trainable.

Keyword-only extras that the reference's README promises or its Triton surface already has
(flash_attention/README.md:34-38, flash_attention_triton.py:722-731): ``causal``, ``softmax_scale``, ``return_lse``.
``flash_attn`` is the [B, S, H, D] surface of ``flash_attn_triton``, with its additive bias and its dropout.
"""
from __future__ import annotations

import ctypes
import math
import threading
from typing import Optional, Tuple, Union

import numpy as np
import torch
from torch import Tensor
from torch.autograd import Function

from .. import _lib

_DTYPE_CODE = {torch.float16: _lib.FO_DTYPE_F16, torch.bfloat16: _lib.FO_DTYPE_BF16}
# the raw hipStream_t that is current on a device, without building a torch.cuda.Stream object around it
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (lambda dev: torch.cuda.current_stream(dev).cuda_stream)
_I64x3 = ctypes.c_int64 * 3
_BHSD, _BSHD = (0, 1, 2, 3), (0, 2, 1, 3)
_torch_empty = torch.empty
_host_module = False        # not asked for yet


def _host():
    """The compiled host path of ordinary calls (csrc/host_path.cpp), or None: where it was not built, or while torch.empty is not
    torch's own (who replaces it, to count or to refuse allocations, sees every one of them)."""
    global _host_module
    if _host_module is False:
        lib = _lib.load()
        try:
            from .. import _host as module
        except ImportError:
            module = None
        device = getattr(torch._C, "_cuda_getDevice", None)
        if module is not None:
            names = ("fo_attn_fwd_ex_ws", "fo_attn_fwd_workspace_ex", "fo_attn_bwd_ws", "fo_attn_bwd_workspace_ex", "fo_strerror")
            addresses = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in names}
            if device is None or not module.init(addresses, device, _raw_stream):
                module = None
        _host_module = module
    return _host_module if torch.empty is _torch_empty else None


def _check_inputs(q: Tensor, k: Tensor, v: Tensor) -> None:
    # the limits documented at flash_attention.py:61-70; violating them raises, as promised there
    if q.dim() != 4 or k.dim() != 4 or v.dim() != 4:
        raise RuntimeError("Q, K and V must be 4-dimensional")
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("All tensors must have the same type")
    if q.dtype not in _DTYPE_CODE:
        raise RuntimeError("Inputs must be half-precision floating points (float16 and bfloat16)")
    if not (q.is_cuda and k.is_cuda and v.is_cuda) or not (q.device == k.device == v.device):
        raise RuntimeError("Q, K and V must be GPU tensors on the same device (there is no CPU path)")
    if q.stride(-1) != 1 or k.stride(-1) != 1 or v.stride(-1) != 1:
        raise RuntimeError("The last dimension of Q, K and V must be contiguous")


Dropout = Tuple[float, int, int]   # (dropout_p, seed, generator offset)


class _AttnExtras(ctypes.Structure):    # fo_attn_extras
    _fields_ = [("bias", ctypes.c_void_p), ("bias_strides", ctypes.c_int64 * 3), ("bias_dtype", ctypes.c_int),
                ("dropout_p", ctypes.c_float), ("dropout_seed", ctypes.c_uint32), ("dropout_offset", ctypes.c_uint64)]


def _expand_bias(bias: Tensor, q: Tensor, B: int, H: int, Sq: int, Sk: int) -> Tensor:
    """The reference's checks and broadcast of the bias (flash_attention_triton.py:752-768): 4-dimensional, the dtype
    of q or fp32, last two dimensions (1, Sk) or (Sq, Sk), expanded (strides of 0) over batch, heads and queries."""
    if bias.dtype not in (q.dtype, torch.float32):
        raise RuntimeError("bias must have the dtype of q or float32")
    if not bias.is_cuda or bias.device != q.device:
        raise RuntimeError("bias must be on the device of q")
    if bias.dim() != 4:
        raise RuntimeError("bias must be 4-dimensional")
    if bias.stride(-1) != 1:
        bias = bias.contiguous()
    if tuple(bias.shape[2:]) not in ((1, Sk), (Sq, Sk)):
        raise RuntimeError("Last 2 dimensions of bias must be (1, seqlen_k) or (seqlen_q, seqlen_k)")
    return bias.expand(B, H, Sq, Sk)


# When _aligned_bias copies, without and with a backward's kernels to come. From so many (query, key) pairs on, by the bytes of an
# element: below, the launch and its host time (16 us) cost more than the copy gains (12 heads at head_dim 64, in place -> copied;
# forward 515 keys bf16 37 -> 29 us, 725 keys 49 -> 31 and fp32 50 -> 33, 1021 keys 66 -> 36 and 64 -> 44; forward + backward with both
# copied 515 keys bf16 155 -> 174, 725 keys 225 -> 175 and fp32 causal 145 -> 173, 1021 keys 434 -> 175 and 213 -> 174).
# Up to so many bytes of rows (rows x bytes of an element) in the forward, whose gain grows with the keys a workgroup walks (about
# 0.045 us per key) while the copy costs 0.45 us per MB: 12 heads x 3071 bf16 298 -> 162 us, causal 194 -> 145, 4 heads x 3071 fp32 184 ->
# 117; beyond, 64 heads x 1021 causal bf16 69 -> 81, fp32 68 -> 140, 12 heads x 2047 fp32 125 -> 130. The backward gains at every
# number of heads (64 heads x 1021, backward alone: bf16 412 -> 118, fp32 289 -> 245). And up to a copy of so many bytes: what
# the memory-side cache (256 MiB) holds for the forward.
_ALIGN_BIAS_FROM = {False: {2: 1 << 19, 4: 3 << 18}, True: {2: 1 << 18, 4: 1 << 19}}
_ALIGN_BIAS_ROW_BYTES = 80000
_ALIGN_BIAS_BYTES = {False: 256 << 20, True: 4 << 30}


def _aligned_bias(bias: Optional[Tensor], q: Tensor, k: Tensor, backward: bool) -> Optional[Tensor]:
    """A bias with a row per query whose rows do not start on 16-byte boundaries, copied (once for what is broadcast over batch
    or heads) into rows that do, which is what the kernels copy tiles from; any other bias as it is. (flash_attn's layout.)"""
    if bias is None:
        return bias
    shape = bias.shape
    # (fewer pairs than are asked for in any case: the usual end of a small call, and of a bias that is the same for every query)
    if len(shape) != 4 or shape[2] * shape[3] < 1 << 18 or shape[2] == 1 or q.dim() != 4 or k.dim() != 4:
        return bias                                            # (what does not fit is refused further on)
    if bias.dtype not in (q.dtype, torch.float32) or not bias.is_cuda or bias.device != q.device:
        return bias
    B, Sq, H, Sk = q.shape[0], q.shape[1], q.shape[2], k.shape[1]
    size = bias.element_size()
    if bias.stride(-1) != 1 or Sq * Sk < _ALIGN_BIAS_FROM[backward][size] or tuple(bias.shape[2:]) != (Sq, Sk) or bias.stride(2) == 0:
        return bias
    # (the forward reads four elements at a time where rows start on a multiple of four: 12 heads x 3068 bf16 148 us, copied 192)
    align = 16 if backward else 4 * size
    if bias.data_ptr() % align == 0 and not any(s * size % align for s, n in zip(bias.stride()[:3], bias.shape) if n > 1):
        return bias
    if bias.shape[0] not in (1, B) or bias.shape[1] not in (1, H):
        return bias
    nb, nh = (1 if bias.stride(i) == 0 else bias.shape[i] for i in (0, 1))
    row = -(-Sk * size // 16) * 16 // size
    if nb * nh * Sq * row * size > _ALIGN_BIAS_BYTES[backward] or (not backward and nb * nh * Sq * size > _ALIGN_BIAS_ROW_BYTES):
        return bias
    try:
        out = torch.empty((nb, nh, Sq, row), dtype=bias.dtype, device=bias.device)
    except torch.OutOfMemoryError:                             # no room for a copy: the kernels read the bias as it is
        return bias
    dev = bias.device.index
    # (as in attn_fwd_strided: the device is made current only when it is not)
    guard = torch.cuda.device(dev) if torch.cuda.current_device() != dev else None
    if guard is not None:
        guard.__enter__()
    try:
        status = _lib.load().fo_attn_bias_rows(bias.data_ptr(), _I64x3(*bias.stride()[:3]), size, nb, nh, Sq, Sk, out.data_ptr(), row, _raw_stream(dev))
    finally:
        if guard is not None:
            guard.__exit__(None, None, None)
    if status != 0:
        _lib.check(status, "fo_attn_bias_rows")
    return out[..., :Sk]


def _extras(bias: Optional[Tensor], dropout: Optional[Dropout]) -> _AttnExtras:
    ex = _AttnExtras()
    if bias is not None:
        ex.bias = bias.data_ptr()
        ex.bias_strides = _I64x3(bias.stride(0), bias.stride(1), bias.stride(2))
        ex.bias_dtype = _lib.FO_DTYPE_F32 if bias.dtype == torch.float32 else _DTYPE_CODE[bias.dtype]
    if dropout is not None:
        ex.dropout_p, ex.dropout_seed, ex.dropout_offset = float(dropout[0]), dropout[1] & 0xFFFFFFFF, dropout[2] % (1 << 64)
    return ex


def next_dropout_state(n_elements: int) -> Tuple[int, int]:
    """(seed, offset) for a dropout mask over ``n_elements`` attention probabilities, taken from torch's generator of the
    current device, whose offset is advanced past them: what increment_philox_state does in the reference
    (flash_attention_triton.py:641-665). The last 16 bytes of the generator state are (seed, offset) as two uint64."""
    state = torch.cuda.get_rng_state()
    words = state.numpy().view(np.uint64)
    seed, offset = int(words[-2]), int(words[-1])
    words[-1] = np.uint64((offset + 4 * math.ceil(n_elements / 4)) % (1 << 64))
    torch.cuda.set_rng_state(state)
    return seed, offset


def dropout_mask(
    dropout_p: float, batch_sz: int, n_heads: int, seqlen_q: int, seqlen_k: int, device: Union[str, torch.device],
    dropout_state: Optional[Tuple[int, int]] = None,
) -> Tensor:
    """The keep-mask (bool [B, H, Sq, Sk], True = kept) that the attention kernels apply for this dropout_p and state:
    triton_dropout_mask of the reference (flash_attention_triton.py:697-717). Without ``dropout_state`` the state comes
    from torch's generator, which is advanced exactly as an attention call of that shape advances it, so seeding, taking
    the mask, seeding again and calling the attention gives the attention's mask (tests/test_flash_attention_triton.py:
    93-103)."""
    if not 0.0 <= dropout_p < 1.0:
        raise RuntimeError(f"dropout_p must be in [0, 1), got {dropout_p}")
    device = torch.device(device)
    n = batch_sz * n_heads * seqlen_q * seqlen_k
    with torch.cuda.device(device):
        seed, offset = dropout_state if dropout_state is not None else next_dropout_state(n)
        keep = torch.empty((batch_sz, n_heads, seqlen_q, seqlen_k), dtype=torch.uint8, device=device)
        status = _lib.load().fo_dropout_mask(keep.data_ptr(), n, float(dropout_p), seed & 0xFFFFFFFF, offset % (1 << 64),
                                             torch.cuda.current_stream(device).cuda_stream)
    _lib.check(status, "fo_dropout_mask")
    return keep.view(torch.bool)


class _FwdPlan:
    """What a forward call of one (shapes, strides, dtype, device, layout) needs besides the data pointers: checked once,
    then reused - the checks, the stride arrays for the C ABI and the sizes cost more host time than a small kernel runs."""
    __slots__ = ("B", "H", "Sq", "Sk", "D", "qs", "ks", "vs", "os", "o_dense_like_q", "dtype_code", "device_index", "lse_shape", "ws_bytes", "ws_bytes_causal", "ws_forms")


_FWD_PLANS: dict = {}


def _fwd_plan(q: Tensor, k: Tensor, v: Tensor, dims: Tuple[int, int, int, int]) -> _FwdPlan:
    # (the scratch memory of a plan depends on what _lib.tune_set has set)
    key = (q.shape, q.stride(), k.shape, k.stride(), v.shape, v.stride(), q.dtype, k.dtype, v.dtype, q.device, k.device, v.device, dims, _lib.tune_generation)
    plan = _FWD_PLANS.get(key)
    if plan is not None:
        return plan
    _check_inputs(q, k, v)
    ib, ih, is_, id_ = dims
    B, H, Sq, D = q.shape[ib], q.shape[ih], q.shape[is_], q.shape[id_]
    Sk = k.shape[is_]
    if k.shape[ib] != B or k.shape[ih] != H or k.shape[id_] != D or v.shape != k.shape:
        raise RuntimeError(f"shape mismatch: Q {tuple(q.shape)}, K {tuple(k.shape)}, V {tuple(v.shape)}")
    if D > 128:
        raise RuntimeError("FlashAttention only support head dimensions up to 128")  # flash_attention_triton.py:745
    if D % 8 != 0:
        raise RuntimeError("head_dim must be a multiple of 8")                        # flash_attention.py:65-66
    plan = _FwdPlan()
    plan.B, plan.H, plan.Sq, plan.Sk, plan.D = B, H, Sq, Sk, D
    strides = lambda t: _I64x3(t.stride(ib), t.stride(ih), t.stride(is_))
    plan.qs, plan.ks, plan.vs = strides(q), strides(k), strides(v)
    o = torch.empty_like(q)
    plan.o_dense_like_q = o.stride() == q.stride()    # empty_like keeps dense layouts; anything else gets a plain contiguous output
    if not plan.o_dense_like_q:
        o = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    plan.os = strides(o)
    plan.dtype_code = _DTYPE_CODE[q.dtype]
    plan.device_index = q.device.index if q.device.index is not None else torch.cuda.current_device()
    plan.lse_shape = (B, H, Sq)
    with torch.cuda.device(plan.device_index):       # scratch memory of a call without bias and dropout, by the mask; other forms: _fwd_workspace
        plan.ws_bytes, plan.ws_bytes_causal = (_lib.load().fo_attn_fwd_workspace(B, H, Sq, Sk, D, plan.ks, plan.vs, causal) for causal in (0, 1))
    plan.ws_forms = {}
    if len(_FWD_PLANS) > 4096:
        _FWD_PLANS.clear()
    _FWD_PLANS[key] = plan
    return plan


def _fwd_workspace(plan: _FwdPlan, causal: bool, bias: Optional[Tensor], dropout: Optional[Dropout], extras) -> int:
    """Bytes of scratch memory that a call with a bias or dropout can use, worked out once per plan and form (as _bwd_workspace)."""
    form = (causal, dropout is not None and dropout[0] > 0.0, None if bias is None else (bias.stride(), bias.data_ptr() % 16, bias.dtype))
    n = plan.ws_forms.get(form)
    if n is None:
        n = _lib.load().fo_attn_fwd_workspace_ex(plan.B, plan.H, plan.Sq, plan.Sk, plan.D, plan.ks, plan.vs, 1 if causal else 0, extras)
        if len(plan.ws_forms) > 64:
            plan.ws_forms.clear()
        plan.ws_forms[form] = n
    return n


_FWD_WS_RETRY = 256                 # as _BWD_WS_RETRY
_refused = threading.local()        # (.fwd: device, bytes, calls) scratch memory that a thread's forward was refused: see _scratch


def _scratch(n_bytes: int, device) -> Optional[Tensor]:
    """Scratch memory of a forward, or None where there is none to be had: the call then does without, and so do the next _FWD_WS_RETRY that
    would ask for as much on that device."""
    refused = getattr(_refused, "fwd", None)
    if refused is not None and refused[2] > 0 and refused[0] == device and n_bytes >= refused[1]:
        refused[2] -= 1
        return None
    try:
        return torch.empty(n_bytes, dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        _refused.fwd = [device, n_bytes, _FWD_WS_RETRY]
        return None


def attn_fwd_strided(
    q: Tensor, k: Tensor, v: Tensor, dims: Tuple[int, int, int, int], causal: bool, softmax_scale: Optional[float],
    dropout: Optional[Dropout] = None, bias: Optional[Tensor] = None,
) -> Tuple[Tensor, Tensor]:
    """Launches fo_attn_fwd (fo_attn_fwd_ex when ``bias`` or ``dropout`` is given), with scratch memory where it helps. ``dims`` =
    positions of (batch, head, sequence, head_dim) in the tensors' shapes; ``bias`` is [B|1, H|1, Sq|1, Sk] whatever
    ``dims`` says. Returns (O with q's shape, dtype and layout; LSE fp32 [B, H, Sq])."""
    host = _host()
    if host is not None and (dims == _BHSD or dims == _BSHD):
        done = host.fwd(q, k, v, dims == _BSHD, causal, softmax_scale, dropout, bias)
        if done is not None:
            return done
    plan = _fwd_plan(q, k, v, dims)
    scale = float(softmax_scale) if softmax_scale else 1.0 / math.sqrt(plan.D)        # flash_attention_triton.py:750
    o = torch.empty_like(q) if plan.o_dense_like_q else torch.empty(q.shape, dtype=q.dtype, device=q.device)
    lse = torch.empty(plan.lse_shape, dtype=torch.float32, device=q.device)
    if bias is not None:
        bias = _expand_bias(bias, q, plan.B, plan.H, plan.Sq, plan.Sk)
    dev = plan.device_index
    lib = _lib.load()
    # (the launch goes to the stream that is current on the tensors' device; the device is made current only when it is not)
    guard = torch.cuda.device(dev) if torch.cuda.current_device() != dev else None
    if guard is not None:
        guard.__enter__()
    try:
        stream = _raw_stream(dev)
        args = (q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                plan.B, plan.H, plan.Sq, plan.Sk, plan.D, plan.qs, plan.ks, plan.vs, plan.os,
                scale, 1 if causal else 0, plan.dtype_code)
        if bias is None and (dropout is None or dropout[0] == 0.0):
            n = plan.ws_bytes_causal if causal else plan.ws_bytes
            ws = _scratch(n, q.device) if n else None
            if ws is not None:
                status = lib.fo_attn_fwd_ws(*args, ws.data_ptr(), n, stream)
            else:
                status = lib.fo_attn_fwd(*args, stream)
        else:
            extras = ctypes.byref(_extras(bias, dropout))
            n = _fwd_workspace(plan, causal, bias, dropout, extras)
            ws = _scratch(n, q.device) if n else None
            if ws is not None:
                status = lib.fo_attn_fwd_ex_ws(*args, extras, ws.data_ptr(), n, stream)
            else:
                status = lib.fo_attn_fwd_ex(*args, extras, stream)
    finally:
        if guard is not None:
            guard.__exit__(None, None, None)
    if status != 0:
        _lib.check(status, "fo_attn_fwd")
    return o, lse


class _BwdPlan:
    """What a backward call of one (shapes, strides, dtypes, devices, layout) needs besides the data pointers, as _FwdPlan.
    (Checks, stride arrays and the switch of the device took 12 of the 31 us such a call cost the host, and a training step of a
    small model waits for its host: B=8 H=12 S=1024 D=64 causal with dropout 132 -> 117 us per step.)"""
    __slots__ = ("B", "H", "Sq", "Sk", "D", "strides", "arrays", "dtype_code", "device_index", "ws_bytes")   # ws_bytes: see _bwd_workspace


_BWD_PLANS: dict = {}


def _bwd_plan(q: Tensor, k: Tensor, v: Tensor, o: Tensor, d_o: Tensor, dims: Tuple[int, int, int, int]) -> _BwdPlan:
    key = (q.shape, q.stride(), k.shape, k.stride(), v.shape, v.stride(), o.stride(), d_o.stride(), q.dtype, k.dtype, v.dtype,
           q.device, k.device, v.device, dims, _lib.tune_generation)      # (the workspace depends on what _lib.tune_set has set)
    plan = _BWD_PLANS.get(key)
    if plan is not None:
        return plan
    _check_inputs(q, k, v)
    ib, ih, is_, id_ = dims
    plan = _BwdPlan()
    plan.B, plan.H, plan.Sq, plan.D = q.shape[ib], q.shape[ih], q.shape[is_], q.shape[id_]
    plan.Sk = k.shape[is_]
    dense = [torch.empty(t.shape, device="meta") for t in (q, k, v)]      # dQ, dK and dV are dense
    plan.arrays = [_I64x3(t.stride(ib), t.stride(ih), t.stride(is_)) for t in (q, k, v, o, d_o, *dense)]
    plan.strides = (ctypes.POINTER(ctypes.c_int64) * 8)(*[ctypes.cast(a, ctypes.POINTER(ctypes.c_int64)) for a in plan.arrays])
    plan.dtype_code = _DTYPE_CODE[q.dtype]
    plan.device_index = q.device.index if q.device.index is not None else torch.cuda.current_device()
    plan.ws_bytes = {}
    if len(_BWD_PLANS) > 4096:
        _BWD_PLANS.clear()
    _BWD_PLANS[key] = plan
    return plan


# after a workspace did not fit: how many calls go without asking for so much again (asking makes the caching allocator give its
# cached blocks back, and the calls after it allocate anew)
_BWD_WS_RETRY = 256


def _bwd_workspace(plan: _BwdPlan, causal: bool, bias: Optional[Tensor], dropout: Optional[Dropout], extras, device) -> Tensor:
    """The workspace of a call: two values per row, and, in the forms of a call that keep it, dS, and behind that the partial sums
    of key blocks that several workgroups share. Without memory for all of that dS alone, or the rows' values. What is asked for
    is worked out once per plan and form (mask, dropout or none, layout of the bias)."""
    form = (causal, dropout is not None and dropout[0] > 0.0, None if bias is None else (bias.stride(), bias.data_ptr() % 16, bias.dtype))
    entry = plan.ws_bytes.get(form)
    if entry is None:
        n = _lib.load().fo_attn_bwd_workspace_ex(plan.B, plan.H, plan.Sq, plan.Sk, plan.D, 1 if causal else 0, extras)
        rows = (8 * plan.B * plan.H * plan.Sq + 255) // 256 * 256
        ds = rows + 2 * plan.B * plan.H * (-(-plan.Sq // 64) * 64) * (-(-plan.Sk // 128) * 128)
        if len(plan.ws_bytes) > 64:
            plan.ws_bytes.clear()
        entry = plan.ws_bytes[form] = [0, 0, [n] + [s for s in (ds, rows) if s < n]]      # first size to ask for, calls it is kept for, sizes
    sizes = entry[2]
    if entry[0]:
        entry[1] -= 1
        if entry[1] < 0:
            entry[0] = 0
    for i in range(entry[0], len(sizes)):
        try:
            return torch.empty(sizes[i], dtype=torch.uint8, device=device)
        except torch.OutOfMemoryError:
            if i + 1 == len(sizes):
                raise
            entry[0], entry[1] = i + 1, _BWD_WS_RETRY


def attn_bwd_strided(
    q: Tensor, k: Tensor, v: Tensor, o: Tensor, lse: Tensor, d_o: Tensor, dims: Tuple[int, int, int, int], causal: bool,
    softmax_scale: Optional[float], dropout: Optional[Dropout] = None, bias: Optional[Tensor] = None,
) -> Tuple[Tensor, Tensor, Tensor]:
    """Launches fo_attn_bwd_ws. Returns (dQ, dK, dV) with the shapes and dtypes of q, k, v (dense; a K/V whose heads are
    an expanded view gets a full-size gradient, which autograd then reduces)."""
    host = _host()
    if host is not None and (dims == _BHSD or dims == _BSHD):
        done = host.bwd(q, k, v, o, lse, d_o, dims == _BSHD, causal, softmax_scale, dropout, bias)
        if done is not None:
            return done
    if d_o.dtype != q.dtype or d_o.shape != q.shape:
        _check_inputs(q, k, v)
        raise RuntimeError(f"dO must have the output's shape and dtype, got {tuple(d_o.shape)} {d_o.dtype}")
    if not d_o.is_contiguous() and (d_o.stride(-1) != 1 or any(s % 8 for s in d_o.stride()[:-1])):
        d_o = d_o.contiguous()
    if o.stride(-1) != 1:
        o = o.contiguous()
    lse = lse.contiguous()
    plan = _bwd_plan(q, k, v, o, d_o, dims)
    scale = float(softmax_scale) if softmax_scale else 1.0 / math.sqrt(plan.D)
    device = q.device
    dq = torch.empty(q.shape, dtype=q.dtype, device=device)
    dk = torch.empty(k.shape, dtype=k.dtype, device=device)
    dv = torch.empty(v.shape, dtype=v.dtype, device=device)
    if bias is not None:
        bias = _expand_bias(bias, q, plan.B, plan.H, plan.Sq, plan.Sk)
    extras = None if bias is None and (dropout is None or dropout[0] == 0.0) else ctypes.byref(_extras(bias, dropout))
    lib = _lib.load()
    dev = plan.device_index
    # (as in the forward: the device is made current only when it is not)
    guard = torch.cuda.device(dev) if torch.cuda.current_device() != dev else None
    if guard is not None:
        guard.__enter__()
    try:
        stream = _raw_stream(dev)
        ws = _bwd_workspace(plan, causal, bias, dropout, extras, device)      # (asked with the device current: it depends on its compute units)
        status = lib.fo_attn_bwd_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse.data_ptr(),
                                    dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), plan.B, plan.H, plan.Sq, plan.Sk, plan.D, plan.strides, scale,
                                    1 if causal else 0, plan.dtype_code, extras, ws.data_ptr(), ws.numel(), stream)
    finally:
        if guard is not None:
            guard.__exit__(None, None, None)
    if status != 0:
        _lib.check(status, "fo_attn_bwd_ws")
    return dq, dk, dv


class FlashAttentionFunction(Function):
    @staticmethod
    def forward(ctx, Q: Tensor, K: Tensor, V: Tensor, causal: bool = False, softmax_scale: Optional[float] = None,
                return_lse: bool = False, dropout: Optional[Dropout] = None):
        """
        :param Q: (B, H, M, D) Query tensor.
        :param K: (B, H, N, D) Key tensor.
        :param V: (B, H, N, D) Value tensor.
        :returns: (B, H, M, D), and the (B, H, M) fp32 logsumexp when ``return_lse``
        """
        o, lse = attn_fwd_strided(Q, K, V, (0, 1, 2, 3), causal, softmax_scale, dropout)
        ctx.save_for_backward(Q, K, V, o, lse)   # what a backward pass needs (flash_attention_triton.py:826)
        ctx.causal = causal
        ctx.softmax_scale = softmax_scale
        ctx.dropout = dropout                    # (p, seed, offset): the backward regenerates the mask (:824-828)
        if return_lse:
            ctx.mark_non_differentiable(lse)
            return o, lse
        return o

    @staticmethod
    def backward(ctx, dO: Tensor, *unused):
        """:param dO: (B, H, M, D) Output gradient. The reference leaves this unimplemented (flash_attention.py:40-45);
        here it is what the reference's Triton backward computes (flash_attention_triton.py:832-958)."""
        Q, K, V, o, lse = ctx.saved_tensors
        dq, dk, dv = attn_bwd_strided(Q, K, V, o, lse, dO, (0, 1, 2, 3), ctx.causal, ctx.softmax_scale, ctx.dropout)
        return dq, dk, dv, None, None, None, None


class _FlashAttnBSHD(Function):
    """flash_attn's autograd node: the same kernels on [batch, seqlen, nheads, headdim] tensors."""

    @staticmethod
    def forward(ctx, q: Tensor, k: Tensor, v: Tensor, causal: bool, softmax_scale: Optional[float], return_lse: bool,
                dropout: Optional[Dropout], bias: Optional[Tensor] = None):
        o, lse = attn_fwd_strided(q, k, v, (0, 2, 1, 3), causal, softmax_scale, dropout, _aligned_bias(bias, q, k, False))
        # (the bias itself, not its copy: every layer that shares a bias would hold a copy of its own until its backward)
        ctx.save_for_backward(q, k, v, o, lse, bias)
        ctx.causal = causal
        ctx.softmax_scale = softmax_scale
        ctx.dropout = dropout
        if return_lse:
            ctx.mark_non_differentiable(lse)
            return o, lse
        return o

    @staticmethod
    def backward(ctx, dO: Tensor, *unused):
        q, k, v, o, lse, bias = ctx.saved_tensors
        if bias is not None and ctx.needs_input_grad[7]:
            raise RuntimeError("FlashAttention does not support bias gradient yet")   # flash_attention_triton.py:854
        dq, dk, dv = attn_bwd_strided(q, k, v, o, lse, dO, (0, 2, 1, 3), ctx.causal, ctx.softmax_scale, ctx.dropout,
                                      _aligned_bias(bias, q, k, True))
        return dq, dk, dv, None, None, None, None, None


def _dropout_arg(dropout_p: float, dropout_state: Optional[Tuple[int, int]], n_elements: int) -> Optional[Dropout]:
    if dropout_p == 0.0:
        return None
    if not 0.0 <= dropout_p < 1.0:
        raise RuntimeError(f"dropout_p must be in [0, 1), got {dropout_p}")
    seed, offset = dropout_state if dropout_state is not None else next_dropout_state(n_elements)
    return (float(dropout_p), int(seed), int(offset))


def multi_head_attention(
    Q: Tensor, K: Tensor, V: Tensor, *, causal: bool = False, softmax_scale: Optional[float] = None, return_lse: bool = False,
    dropout_p: float = 0.0, dropout_state: Optional[Tuple[int, int]] = None,
) -> Union[Tensor, Tuple[Tensor, Tensor]]:
    """FlashAttention forward (https://arxiv.org/abs/2205.14135), B = batch, H = heads, M = queries, N = keys, D = head dim.

    Limitations (violations raise RuntimeError): head_dim a multiple of 8 up to 128; the last dimension of Q, K, V contiguous and rows 16-byte aligned; inputs float16 or
    bfloat16; GPU tensors.

    :param Q: (B, H, M, D) Query tensor.
    :param K: (B, H, N, D) Key tensor.
    :param V: (B, H, N, D) Value tensor.
    :param causal: query i attends keys j <= i
    :param softmax_scale: multiplier of Q K^T, default 1/sqrt(D)
    :param return_lse: also return the (B, H, M) fp32 logsumexp of the scaled scores
    :param dropout_p: probability of dropping an attention probability (flash_attention_triton.py:216-219)
    :param dropout_state: (seed, offset) of the mask; default: taken from torch's generator, which is advanced
    :returns: (B, H, M, D)
    """
    drop = None if dropout_p == 0.0 else _dropout_arg(dropout_p, dropout_state, Q.shape[0] * Q.shape[1] * Q.shape[2] * K.shape[2])
    if not (torch.is_grad_enabled() and (Q.requires_grad or K.requires_grad or V.requires_grad)):
        # nothing to differentiate: no autograd node (its bookkeeping costs more host time than a small kernel runs)
        o, lse = attn_fwd_strided(Q, K, V, (0, 1, 2, 3), causal, softmax_scale, drop)
        return (o, lse) if return_lse else o
    return FlashAttentionFunction.apply(Q, K, V, causal, softmax_scale, return_lse, drop)


def flash_attn(
    q: Tensor, k: Tensor, v: Tensor, bias: Optional[Tensor] = None, causal: bool = False, dropout_p: float = 0.0,
    softmax_scale: Optional[float] = None, return_lse: bool = False, dropout_state: Optional[Tuple[int, int]] = None,
) -> Union[Tensor, Tuple[Tensor, Tensor]]:
    """The [batch, seqlen, nheads, headdim] surface of flash_attn_triton (flash_attention_triton.py:722-737,961),
    differentiable in q, k and v, with dropout and with an additive bias on the scaled scores: [B|1, H|1, 1, seqlen_k]
    or [B|1, H|1, seqlen_q, seqlen_k], the dtype of q or fp32 (:752-768). A bias that requires grad makes the backward
    raise, as in the reference (:854)."""
    drop = None if dropout_p == 0.0 else _dropout_arg(dropout_p, dropout_state, q.shape[0] * q.shape[2] * q.shape[1] * k.shape[1])
    if not (torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad or (bias is not None and bias.requires_grad))):
        rows = None if bias is None else _aligned_bias(bias, q, k, False)
        o, lse = attn_fwd_strided(q, k, v, (0, 2, 1, 3), causal, softmax_scale, drop, rows)
        return (o, lse) if return_lse else o
    return _FlashAttnBSHD.apply(q, k, v, causal, softmax_scale, return_lse, drop, bias)
