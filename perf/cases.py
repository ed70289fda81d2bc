"""The work this framework is measured on: attention (forward, and forward + backward) and the fused Lion step, called
through the public entry points of ``fast_ops`` as a user's program calls them.

``listed()`` names twelve cases, from the smallest call to the largest; ``draw(rng)`` gives further ones of the same
families with sizes spread over the whole range each family meets. A case is a dict of plain values, ``prepare`` builds
what a program holds before the call (inputs from the seed alone), ``run`` is one pass.
"""
import math

import torch

from fast_ops.flash_attention.flash_attention import flash_attn, multi_head_attention
from fast_ops.lion.lion_optimizer import Lion

DEVICE = "cuda:0"
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}

# No drawn case asks for more than these: the floating-point operations of the training step on long sequences and the
# bytes of the optimizer step over 1.3e9 parameters. Options that cost more time per operation get a smaller share.
MAX_FLOPS = 1.9e12
MAX_FLOPS_ENCODER = 1.09e12
MAX_FLOPS_OPTIONS = 6.0e11
MAX_LION_BYTES = 2.0e10


# ---------------------------------------------------------------------------------------------------------------------
# cases


def _attention(name=None, *, B, H, Sq, D, dtype, Sk=None, causal=False, train=False, surface="bhsd", bias="none",
               bias_dtype="float32", dropout=0.0, layout="dense", kv_heads="all"):
    """surface: "bhsd" = multi_head_attention on [B, H, S, D] tensors, "bshd" = flash_attn on [B, S, H, D] tensors.
    bias (flash_attn only): "none", "key" = [B, 1, 1, Sk] padding mask, "matrix" = [1, H, Sq, Sk] position bias.
    layout: "dense", "packed" = q, k, v are slices of one projection's output, "cache" = K and V are the filled part of
    a larger cache. kv_heads: "all", or "one" = multi-query (every query head reads the same K and V)."""
    case = dict(kind="attention", B=B, H=H, Sq=Sq, Sk=Sq if Sk is None else Sk, D=D, dtype=dtype, causal=causal, train=train,
                surface=surface, bias=bias, bias_dtype=bias_dtype, dropout=dropout, layout=layout, kv_heads=kv_heads)
    if name is not None:
        case["name"] = name
    return case


def _lion(name=None, *, model, width, layers, vocab=0, context=0, dtype="float32", momentum="bfloat16"):
    """model: "transformer" = the parameter list of a GPT-2 style decoder (embeddings, and per layer two norms, the
    attention and the feed-forward weights with their biases), "matrices" = `layers` pairs of width x 4 width matrices."""
    case = dict(kind="lion", model=model, width=width, layers=layers, vocab=vocab, context=context, dtype=dtype, momentum=momentum)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call: a short batch through an encoder, where the launch and the host's share of a call are what counts
        _attention("forward_tiny", B=2, H=4, Sq=128, D=64, dtype="float16"),
        # prefill of a GPT-2-small batch: q, k and v are slices of the projection's output, [B, S, 3, H, D]
        _attention("forward_gpt2_small", B=8, H=12, Sq=1024, D=64, dtype="bfloat16", causal=True, surface="bshd", layout="packed"),
        # the attention of a GPT-2-small training step with the dropout that model is trained with
        _attention("train_gpt2_small_dropout", B=8, H=12, Sq=1024, D=64, dtype="bfloat16", causal=True, train=True,
                   surface="bshd", dropout=0.1),
        # prefill of long documents, the benchmark's headline shape
        _attention("forward_long_causal", B=2, H=16, Sq=8192, D=128, dtype="bfloat16", causal=True),
        # training on long documents: forward and backward of the same shape
        _attention("train_long_causal", B=2, H=16, Sq=8192, D=128, dtype="bfloat16", causal=True, train=True),
        # a large encoder batch: no mask, fp16
        _attention("forward_encoder_fp16", B=16, H=32, Sq=2048, D=128, dtype="float16"),
        # twelve heads per GPU of a tensor-parallel model, a padding mask as bias and dropout (the reference's own benchmark)
        _attention("train_padding_dropout", B=1, H=12, Sq=4096, D=128, dtype="bfloat16", train=True, surface="bshd",
                   bias="key", bias_dtype="bfloat16", dropout=0.1),
        # training with a relative position bias per head (the reference's own test size)
        _attention("train_position_bias", B=1, H=12, Sq=3072, D=128, dtype="bfloat16", causal=True, train=True, surface="bshd",
                   bias="matrix", bias_dtype="bfloat16"),
        # generation: one new token per sequence against the filled part of a K/V cache
        _attention("decode_cache", B=4, H=32, Sq=1, Sk=4001, D=128, dtype="bfloat16", layout="cache"),
        # training of a decoder that attends to an encoder's output, lengths and head_dim off the tile sizes
        _attention("train_cross_ragged", B=4, H=16, Sq=777, Sk=1250, D=80, dtype="bfloat16", train=True),
        # optimizer step of GPT-2-small: 148 tensors from 768 to 38.6e6 elements
        _lion("lion_gpt2_small", model="transformer", width=768, layers=12, vocab=50257, context=1024),
        # optimizer step over 1.3e9 parameters in 78 large matrices
        _lion("lion_large", model="matrices", width=2048, layers=39),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A sequence length: half of them multiples of 128, as batches are padded to, the others as they come."""
    n = _log_int(rng, lo, hi)
    return max(128, (n + 64) // 128 * 128) if rng.random() < 0.5 and n >= 128 else n


def _fit(rng, make, heads, limit, most):
    """make(B, H) with a number of heads and a batch size up to `most` that keep the call within `limit` operations."""
    H = rng.choice([h for h in heads if work(make(1, h))["flops"] <= limit])
    return make(max(1, min(_log_int(rng, 1, most), int(limit // work(make(1, H))["flops"]))), H)


def draw(rng):
    family = rng.choice(["forward_small", "forward_prefill", "forward_long", "forward_encoder", "train_short", "train_long",
                         "train_tensor_parallel", "train_position_bias", "decode", "cross", "lion_model", "lion_matrices"])
    dtype = rng.choice(["bfloat16", "bfloat16", "float16"])
    D = rng.choice([64, 128])
    if family == "forward_small":
        return _attention(B=rng.randint(1, 4), H=rng.choice([2, 4, 6, 8, 12]), Sq=_length(rng, 32, 384), D=rng.choice([32, 64, 64, 128]),
                          dtype=dtype, causal=rng.random() < 0.5, surface=rng.choice(["bhsd", "bshd"]))
    if family == "forward_prefill":
        S = _length(rng, 256, 3000)
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=D, dtype=dtype, causal=True, surface="bshd", layout="packed"),
                    [12, 16, 20, 32], MAX_FLOPS_OPTIONS, 16)
    if family == "forward_long":
        S = _length(rng, 3000, 20000)
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=128, dtype=dtype, causal=True), [8, 12, 16, 32], MAX_FLOPS, 4)
    if family == "forward_encoder":
        S = _length(rng, 197, 4096)
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=D, dtype=dtype), [12, 16, 32], MAX_FLOPS_ENCODER, 32)
    if family == "train_short":
        S, p = _length(rng, 128, 2048), rng.choice([0.0, 0.1])
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=64, dtype=dtype, causal=True, train=True, surface="bshd", dropout=p),
                    [8, 12, 16, 25], MAX_FLOPS_OPTIONS, 16)
    if family == "train_long":
        S = _length(rng, 2048, 12000)
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=128, dtype=dtype, causal=True, train=True), [8, 12, 16, 32], MAX_FLOPS, 4)
    if family == "train_tensor_parallel":
        S, p, bias, causal = _length(rng, 1024, 8192), rng.choice([0.0, 0.1, 0.17]), rng.choice(["none", "key"]), rng.random() < 0.5
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=128, dtype=dtype, causal=causal, train=True, surface="bshd", bias=bias,
                                                 bias_dtype=dtype, dropout=p), [4, 6, 12], MAX_FLOPS_OPTIONS, 2)
    if family == "train_position_bias":
        S, f32, causal = _length(rng, 512, 4096), rng.random() < 0.3, rng.random() < 0.5
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=S, D=D, dtype=dtype, causal=causal, train=True, surface="bshd", bias="matrix",
                                                 bias_dtype="float32" if f32 else dtype), [8, 12, 16], MAX_FLOPS_OPTIONS, 4)
    if family == "decode":
        return _attention(B=_log_int(rng, 1, 16), H=rng.choice([12, 16, 32]), Sq=rng.choice([1, 1, 1, 2, 4, 5, 16]),
                          Sk=_log_int(rng, 512, 16384), D=D, dtype=dtype, layout="cache", kv_heads=rng.choice(["all", "all", "one"]))
    if family == "cross":
        Sq, Sk, dim, train = _log_int(rng, 100, 2000), _log_int(rng, 100, 3000), rng.choice([32, 48, 64, 80, 96, 112, 128]), rng.random() < 0.6
        return _fit(rng, lambda B, H: _attention(B=B, H=H, Sq=Sq, Sk=Sk, D=dim, dtype=dtype, train=train), [8, 12, 16], MAX_FLOPS_OPTIONS, 8)
    kinds = rng.choice([("float32", "bfloat16"), ("float32", "bfloat16"), ("bfloat16", "bfloat16"), ("float16", "float16"), ("float32", "float32")])
    per_element = _lion_bytes(*kinds)
    if family == "lion_model":
        width = 64 * _log_int(rng, 4, 24)
        return _lion(model="transformer", width=width, layers=rng.randint(4, 24), vocab=rng.choice([32000, 50257]), context=1024,
                     dtype=kinds[0], momentum=kinds[1])
    width = 32 * _log_int(rng, 4, 64)
    most = max(1, int(MAX_LION_BYTES // (8 * width * width * per_element)))
    return _lion(model="matrices", width=width, layers=min(_log_int(rng, 1, 40), most), dtype=kinds[0], momentum=kinds[1])


# ---------------------------------------------------------------------------------------------------------------------
# what a program has in hand before the call


def _prepare_attention(case, g):
    dtype, B, H, Sq, Sk, D = DTYPES[case["dtype"]], case["B"], case["H"], case["Sq"], case["Sk"], case["D"]
    bshd = case["surface"] == "bshd"

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32).to(dtype)

    def heads(n_heads, S):
        return (B, S, n_heads, D) if bshd else (B, n_heads, S, D)

    if case["layout"] == "packed":
        qkv = randn(B, Sq, 3, H, D)                                    # [B, S, H, D] surface
        q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
    else:
        n_kv = 1 if case["kv_heads"] == "one" else H
        q = randn(*heads(H, Sq))
        capacity = (Sk // 1024 + 1) * 1024 if case["layout"] == "cache" else Sk
        k, v = randn(*heads(n_kv, capacity)), randn(*heads(n_kv, capacity))
        if capacity != Sk:
            k, v = k.narrow(1 if bshd else 2, 0, Sk), v.narrow(1 if bshd else 2, 0, Sk)
        if n_kv != H:
            k, v = k.expand(heads(H, Sk)), v.expand(heads(H, Sk))
    state = dict(case=case, q=q, k=k, v=v, bias=None, dropout_state=None, d_o=None)
    if case["bias"] == "key":
        # a padding mask: up to a quarter of every sequence's keys do not count
        bias = torch.zeros(B, 1, 1, Sk, device=DEVICE, dtype=DTYPES[case["bias_dtype"]])
        for b, n in enumerate(torch.randint(3 * Sk // 4, Sk + 1, (B,), generator=g, device=DEVICE).tolist()):
            bias[b, :, :, n:] = -10000.0
        state["bias"] = bias
    elif case["bias"] == "matrix":
        state["bias"] = torch.randn((1, H, Sq, Sk), generator=g, device=DEVICE, dtype=torch.float32).to(DTYPES[case["bias_dtype"]])
    if case["dropout"] > 0.0:
        # the state the generator is in when the step begins, as a program that recomputes its forward keeps it
        draws = torch.randint(0, 1 << 30, (2,), generator=g, device=DEVICE).tolist()
        state["dropout_state"] = (draws[0], 4 * draws[1])
    if case["train"]:
        state["q"], state["k"], state["v"] = (t.detach().requires_grad_(True) for t in (q, k, v))
        state["d_o"] = randn(*heads(H, Sq))
    return state


def _lion_shapes(case):
    n = case["width"]
    if case["model"] == "matrices":
        return [(n, 4 * n), (4 * n, n)] * case["layers"]
    layer = [(n,), (n,), (n, 3 * n), (3 * n,), (n, n), (n,), (n,), (n,), (n, 4 * n), (4 * n,), (4 * n, n), (n,)]
    return [(case["vocab"], n), (case["context"], n)] + layer * case["layers"] + [(n,), (n,)]


def _prepare_lion(case, g):
    dtype, m_dtype = DTYPES[case["dtype"]], DTYPES[case["momentum"]]

    shapes = _lion_shapes(case)
    sizes = [math.prod(s) for s in shapes]

    # Parameters, gradients and momenta are views of one buffer each, as a data-parallel trainer lays them out
    def buffer(std, dt):
        flat = torch.empty(sum(sizes), device=DEVICE, dtype=dt).normal_(0.0, std, generator=g)
        return flat, [t.view(s) for t, s in zip(flat.split(sizes), shapes)]

    flat_p, params = buffer(0.02, dtype)
    _, grads = buffer(1e-2, dtype)
    flat_m, momenta = buffer(1e-3, m_dtype)
    params = [torch.nn.Parameter(p) for p in params]
    opt = Lion(params, lr=1e-4, betas=(0.9, 0.99), weight_decay=0.1, exp_avg_dtype=m_dtype)
    for p, grad, exp_avg in zip(params, grads, momenta):      # a run in progress: gradients and momenta are there
        p.grad = grad
        opt.state[p]["exp_avg"] = exp_avg
    return dict(case=case, params=flat_p, exp_avg=flat_m, opt=opt)


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    return _prepare_attention(case, g) if case["kind"] == "attention" else _prepare_lion(case, g)


# ---------------------------------------------------------------------------------------------------------------------
# one pass


def run(state):
    case = state["case"]
    if case["kind"] == "lion":
        state["opt"].step()
        return {"params": state["params"], "exp_avg": state["exp_avg"]}
    q, k, v = state["q"], state["k"], state["v"]
    if case["surface"] == "bshd":
        o = flash_attn(q, k, v, bias=state["bias"], causal=case["causal"], dropout_p=case["dropout"], dropout_state=state["dropout_state"])
    else:
        o = multi_head_attention(q, k, v, causal=case["causal"], dropout_p=case["dropout"], dropout_state=state["dropout_state"])
    if not case["train"]:
        return o
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["d_o"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact its results are


def _lion_bytes(dtype, momentum):
    """Per element: parameter, gradient and momentum read, parameter and momentum written."""
    p, m = DTYPES[dtype].itemsize, DTYPES[momentum].itemsize
    return 3 * p + 2 * m


def work(case):
    if case["kind"] == "lion":
        n = sum(math.prod(s) for s in _lion_shapes(case))
        return {"bytes": n * _lion_bytes(case["dtype"], case["momentum"]), "flops": 8 * n}
    B, H, Sq, Sk, D = case["B"], case["H"], case["Sq"], case["Sk"], case["D"]
    m = min(Sq, Sk)
    pairs = m * (m + 1) // 2 + (Sq - m) * Sk if case["causal"] else Sq * Sk
    n_kv = 1 if case["kv_heads"] == "one" else H
    q_elems, kv_elems = B * H * Sq * D, B * n_kv * Sk * D
    bias = {"none": 0, "key": B * Sk, "matrix": H * Sq * Sk}[case["bias"]] * DTYPES[case["bias_dtype"]].itemsize
    if not case["train"]:
        # two products per (query, key) pair; q, k, v read, o written
        return {"bytes": 2 * (2 * q_elems + 2 * kv_elems) + bias, "flops": 4 * D * B * H * pairs}
    # two products forward, five backward; q, k, v, dO read, o, dq, dk, dv written
    return {"bytes": 2 * (4 * q_elems + 4 * kv_elems) + bias, "flops": 14 * D * B * H * pairs}


def tolerance(case):
    if case["kind"] == "lion":
        return "exact"
    # Four times the distance to the same expression in float64: probabilities, and in the backward their gradients, are
    # rounded to the operand type before the second products, and results are stored in it.
    # (Measured, listed and drawn cases: 1.9e-3 to 2.6e-3 in bfloat16, 2.4e-4 to 3.3e-4 in float16.)
    return {"rel": {"bfloat16": 1.0e-2, "float16": 1.3e-3}[case["dtype"]]}
