"""The work that programs built on this library give it, as timed cases.

Two public surfaces are used as programs use them: the C ABI
(``include/ember_amd.h`` through ``ember_amd.capi``) for attention, on device
buffers that the program owns and reuses, and the Python front-end
(``Tensor``, ``nn``, ``loss``, ``optim``) for everything else, whose results
the library allocates.  All work is fp32 on the null stream.

A case is a dict of plain values; ``prepare`` makes its inputs on the GPU from
the seed alone, ``run`` is one pass, ``exact`` the same results in float64 by
plain torch, ``work`` the bytes and operations that a pass cannot do without
(each input read once, each output written once).
"""

from __future__ import annotations

import math

import torch

import ember_amd as em
from ember_amd import capi, loss, nn, optim
from ember_amd import random as em_random

HEAD_DIMS = (32, 64, 128)


def listed():
    return [
        # One request of a small model: a single launch, latency and idle CUs decide.
        dict(name="attn_fwd_small", kind="attention", B=1, H=4, S=256, D=64, causal=False, layout="dense", grad=False),
        # Prefill / inference at an ordinary length, logsumexp kept.
        dict(name="attn_fwd_2048", kind="attention", B=8, H=16, S=2048, D=64, causal=True, layout="dense", grad=False),
        # The headline training shape, forward and backward.
        dict(name="attn_train_4096", kind="attention", B=4, H=32, S=4096, D=128, causal=True, layout="dense", grad=True),
        # Many short sequences (bytes, not operations, decide).
        dict(name="attn_train_short", kind="attention", B=256, H=64, S=64, D=64, causal=True, layout="dense", grad=True),
        # An encoder on a length no tile divides, reading the packed projection.
        dict(name="attn_train_ragged", kind="attention", B=3, H=10, S=777, D=128, causal=False, layout="packed", grad=True),
        # Tensor @ Tensor, the square product.
        dict(name="matmul_4096", kind="matmul", batch=1, n=4096, k=4096, m=4096),
        # Batched products of sizes that no tile divides.
        dict(name="matmul_ragged", kind="matmul", batch=12, n=197, k=333, m=250),
        # A transformer projection, forward and backward.
        dict(name="linear_train_proj", kind="linear", rows=16384, n_in=1024, n_out=3072, gelu=False),
        # LayerNorm over a block's token rows, forward and backward.
        dict(name="layernorm_train", kind="layernorm", rows=8192, features=1024),
        # The loss of a classifier head, value and gradient.
        dict(name="classifier_loss", kind="classifier", rows=8192, classes=1000),
        # One SGD step of a small classifier: many small calls.
        dict(name="mlp_step", kind="mlp", rows=64, n_in=784, hidden=128, n_out=10),
        # One Adam step of a decoder block.
        dict(name="decoder_step", kind="decoder", B=8, S=1024, d=1024, H=16),
    ]


# ---- drawn cases: the same ranges ----


def _log_int(rng, low, high):
    """An integer spread over the logarithm of [low, high]; two in five are
    rounded to a multiple of 64 where that stays in range, as real sizes often
    are, the others left as they fall."""
    x = int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))
    if rng.random() < 0.4 and x >= 48:
        x = 64 * round(x / 64)
    return min(high, max(low, x))


def draw(rng):
    kind = rng.choices(("attention", "matmul", "linear", "layernorm", "classifier", "mlp", "decoder"),
                       weights=(6, 3, 3, 1, 1, 1, 1))[0]
    if kind == "attention":
        D = rng.choice(HEAD_DIMS)
        S = _log_int(rng, 16, 4096)
        grad = rng.random() < 0.6
        # Heads in all: no more rows than 2^20 and no more products than the largest listed case.
        most = min((1 << 20) * 64 // (S * D), (1 << 37) // (S * S * D))
        heads = _log_int(rng, 1, max(1, min(8192, most)))
        H = min(heads, rng.choice((1, 4, 8, 12, 16, 32)))
        return dict(kind=kind, B=max(1, heads // H), H=H, S=S, D=D, causal=rng.random() < 0.6,
                    layout=rng.choice(("dense", "dense", "packed")), grad=grad)
    if kind == "matmul":
        batch = rng.choice((1, 1, 1, rng.randint(2, 32)))
        top = 4096 if batch == 1 else 512
        return dict(kind=kind, batch=batch, n=_log_int(rng, 16, top), k=_log_int(rng, 16, top), m=_log_int(rng, 16, top))
    if kind == "linear":
        return dict(kind=kind, rows=_log_int(rng, 16, 16384), n_in=_log_int(rng, 16, 2048), n_out=_log_int(rng, 16, 3072),
                    gelu=rng.random() < 0.4)
    if kind == "layernorm":
        return dict(kind=kind, rows=_log_int(rng, 16, 16384), features=4 * _log_int(rng, 16, 512))
    if kind == "classifier":
        return dict(kind=kind, rows=_log_int(rng, 16, 8192), classes=_log_int(rng, 10, 4096))
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 8, 512), n_in=_log_int(rng, 16, 1024), hidden=_log_int(rng, 16, 1024),
                    n_out=_log_int(rng, 4, 100))
    H = rng.choice((2, 4, 8))
    return dict(kind=kind, B=rng.randint(1, 8), S=_log_int(rng, 32, 512), d=H * rng.choice(HEAD_DIMS), H=H)


# ---- inputs ----


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _uniform(g, a, *shape):
    return (torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * 2 - 1) * a


class _Block:
    """The device buffer of an ember Tensor, for torch to view without a copy;
    the view keeps the Tensor's buffer alive."""

    def __init__(self, t):
        self.core = t._core
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": "<f4", "version": 2,
                                         "data": (t._core.data_ptr, False)}


def _as_torch(t):
    return torch.as_tensor(_Block(t), device="cuda")


def _as_ember(x):
    t = em_random.constant(0.0, tuple(x.shape))
    _as_torch(t).copy_(x)
    return t


def _inputs(case, seed):
    """The case's inputs as float32 torch tensors, by name."""
    g, c = _generator(seed), case
    kind = c["kind"]
    if kind == "attention":
        B, H, S, D = c["B"], c["H"], c["S"], c["D"]
        if c["layout"] == "packed":
            qkv, d_o = _normal(g, B, S, 3, H, D), _normal(g, B, S, H, D)
        else:
            qkv, d_o = _normal(g, 3, B, H, S, D), _normal(g, B, H, S, D)
        return dict(qkv=qkv, d_o=d_o)
    if kind == "matmul":
        return dict(a=_uniform(g, 1.0, c["batch"], c["n"], c["k"]), b=_uniform(g, 1.0, c["batch"], c["k"], c["m"]))
    if kind == "linear":
        scale = 1 / math.sqrt(c["n_in"])
        return dict(x=_normal(g, c["rows"], c["n_in"]), w=_uniform(g, scale, c["n_in"], c["n_out"]),
                    b=_uniform(g, scale, c["n_out"]), grad=_normal(g, c["rows"], c["n_out"]))
    if kind == "layernorm":
        rows, d = c["rows"], c["features"]
        return dict(x=_normal(g, rows, d) * 2 + 0.5, gamma=1 + _uniform(g, 0.2, d), beta=_uniform(g, 0.2, d),
                    grad=_normal(g, rows, d))
    if kind == "classifier":
        rows, classes = c["rows"], c["classes"]
        label = torch.randint(classes, (rows,), generator=g, device="cuda")
        return dict(logits=_normal(g, rows, classes) * 2,
                    target=torch.nn.functional.one_hot(label, classes).float())
    if kind == "mlp":
        sizes = ((c["n_in"], c["hidden"]), (c["hidden"], c["n_out"]))
        label = torch.randint(c["n_out"], (c["rows"],), generator=g, device="cuda")
        return dict(x=torch.rand((c["rows"], c["n_in"]), generator=g, device="cuda"),
                    target=torch.nn.functional.one_hot(label, c["n_out"]).float(),
                    w=[_uniform(g, 1 / math.sqrt(i), i, o) for i, o in sizes])
    rows, d = c["B"] * c["S"], c["d"]
    w = [_uniform(g, math.sqrt(6 / (i + o)), i, o) for i, o in ((d, 3 * d), (d, d), (d, 4 * d), (4 * d, d))]
    return dict(x=_normal(g, rows, d), target=_normal(g, rows, d), w=w)


# ---- attention through the C ABI, on the program's own buffers ----


def _strides(case):
    """(batch, head, row) strides of q, k, v and of o, and the views' offsets."""
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    if case["layout"] == "packed":
        return (S * 3 * H * D, D, 3 * H * D), (S * H * D, D, H * D), H * D
    return (H * S * D, S * D, D), (H * S * D, S * D, D), B * H * S * D


def _prepare_attention(case, data):
    qkv, d_o = data["qkv"], data["d_o"]
    st = dict(qkv=qkv, d_o=d_o, o=torch.empty_like(d_o), lib=capi.lib(),
              lse=torch.empty((case["B"], case["H"], case["S"]), device="cuda"))
    in_st, out_st, step = _strides(case)
    dims = (case["B"], case["H"], case["S"], case["D"], 1 / math.sqrt(case["D"]), int(case["causal"]), *in_st, *out_st)
    parts = lambda x: [x.data_ptr() + 4 * step * i for i in range(3)]  # noqa: E731
    q, k, v = parts(qkv)
    st["fwd"] = (q, k, v, st["o"].data_ptr(), st["lse"].data_ptr(), *dims)
    if case["grad"]:
        st["dqkv"] = torch.empty_like(qkv)
        st["bwd"] = (q, k, v, st["o"].data_ptr(), st["lse"].data_ptr(), d_o.data_ptr(), *parts(st["dqkv"]), *dims)
    return st


def _run_attention(st):
    status = st["lib"].attention_fwd(*st["fwd"])
    if status == 0 and "bwd" in st:
        status = st["lib"].attention_bwd(*st["bwd"])
    if status:
        capi.check(status, "attention")
    return (st["o"], st["lse"], st["dqkv"]) if "bwd" in st else (st["o"], st["lse"])


# ---- the rest through the Python front-end ----


def prepare(case, seed):
    c, kind = case, case["kind"]
    data = _inputs(case, seed)
    if kind == "attention":
        st = _prepare_attention(case, data)
    elif kind == "matmul":
        lead = (c["batch"],) if c["batch"] > 1 else ()
        st = dict(a=_as_ember(data["a"].reshape(*lead, c["n"], c["k"])), b=_as_ember(data["b"].reshape(*lead, c["k"], c["m"])))
    elif kind == "linear":
        layer = nn.Linear(c["n_in"], c["n_out"], activation="gelu" if c["gelu"] else None)
        layer.w, layer.b = _as_ember(data["w"]), _as_ember(data["b"])
        st = dict(layer=layer, x=_as_ember(data["x"]), grad=_as_ember(data["grad"]))
    elif kind == "layernorm":
        layer = nn.LayerNorm(c["features"])
        layer.gamma, layer.beta = _as_ember(data["gamma"]), _as_ember(data["beta"])
        st = dict(layer=layer, x=_as_ember(data["x"]), grad=_as_ember(data["grad"]))
    elif kind == "classifier":
        st = dict(loss=loss.CrossEntropyLoss(), logits=_as_ember(data["logits"]), target=_as_ember(data["target"]))
    elif kind == "mlp":
        layers = [nn.Linear(c["n_in"], c["hidden"]), nn.ReLU(), nn.Linear(c["hidden"], c["n_out"])]
        layers[0].w, layers[2].w = (_as_ember(w) for w in data["w"])
        model = nn.Sequential(*layers)
        st = dict(model=model, loss=loss.CrossEntropyLoss(), opt=optim.SGD(model.parameters(), lr=0.01, momentum=0.9),
                  x=_as_ember(data["x"]), target=_as_ember(data["target"]))
    else:
        block = nn.DecoderBlock(c["d"], c["H"], 4, True)
        block.w_qkv, block.w_o, block.w_1, block.w_2 = (_as_ember(w) for w in data["w"])
        st = dict(block=block, loss=loss.MSELoss(), opt=optim.Adam(block.parameters(), lr=1e-3), B=c["B"], S=c["S"],
                  x=_as_ember(data["x"]), target=_as_ember(data["target"]))
    st["kind"] = kind
    return st


def run(st):
    kind = st["kind"]
    if kind == "attention":
        return _run_attention(st)
    if kind == "matmul":
        return _as_torch(st["a"] @ st["b"])
    if kind in ("linear", "layernorm"):
        layer = st["layer"]
        y = layer(st["x"])
        dx = layer.backward(st["grad"])
        return [_as_torch(t) for t in (y, dx, *layer.gradients())]
    if kind == "classifier":
        value = st["loss"](st["logits"], st["target"])
        return value, _as_torch(st["loss"].backward())
    if kind == "mlp":
        model, crit = st["model"], st["loss"]
        y = model(st["x"])
        value = crit(y, st["target"])
        model.backward(crit.backward())
        grads = model.gradients()
        st["opt"].apply(grads)
        return value, _as_torch(y), [_as_torch(t) for t in grads]
    block, crit = st["block"], st["loss"]
    y = block(st["x"], st["B"], st["S"])
    value = crit(y, st["target"])
    dx = block.backward(crit.backward())
    grads = block.gradients()
    st["opt"].apply(grads)
    return value, _as_torch(y), _as_torch(dx), [_as_torch(t) for t in grads]


# ---- the same in float64 ----


def _attention64(q, k, v, causal):
    """O and logsumexp of float64 (heads, S, D) operands, differentiable."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        s = s.masked_fill(torch.ones(s.shape[1:], device=s.device, dtype=torch.bool).triu(1), -math.inf)
    lse = torch.logsumexp(s, -1)
    return torch.matmul(torch.exp(s - lse[..., None]), v), lse


def _exact_attention(case, data):
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    packed = case["layout"] == "packed"
    qkv = data["qkv"].permute(2, 0, 3, 1, 4) if packed else data["qkv"]
    d_o = data["d_o"].permute(0, 2, 1, 3) if packed else data["d_o"]
    qkv, d_o = qkv.reshape(3, B * H, S, D), d_o.reshape(B * H, S, D)
    o, lse, grads = torch.empty_like(d_o, dtype=torch.float64), torch.empty(B * H, S, device="cuda", dtype=torch.float64), None
    if case["grad"]:
        grads = torch.empty_like(qkv, dtype=torch.float64)
    step = max(1, (1 << 26) // (S * S))
    for i in range(0, B * H, step):
        part = [x[i:i + step].double().requires_grad_(case["grad"]) for x in qkv]
        with torch.set_grad_enabled(case["grad"]):
            oi, li = _attention64(*part, case["causal"])
        o[i:i + step], lse[i:i + step] = oi.detach(), li.detach()
        if case["grad"]:
            grads[:, i:i + step] = torch.stack(torch.autograd.grad(oi, part, d_o[i:i + step].double()))
    o, lse = o.reshape(B, H, S, D), lse.reshape(B, H, S)
    if packed:
        o = o.permute(0, 2, 1, 3).contiguous()
    if not case["grad"]:
        return o, lse
    grads = grads.reshape(3, B, H, S, D)
    return o, lse, grads.permute(1, 3, 0, 2, 4).contiguous() if packed else grads


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(0.8 * x))


def _exact_decoder(case, x, target, w):
    B, S, d, H = case["B"], case["S"], case["d"], case["H"]
    bias = [x.new_zeros(n).requires_grad_() for n in (3 * d, d, 4 * d, d)]
    norm = [(x.new_ones(d).requires_grad_(), x.new_zeros(d).requires_grad_()) for _ in range(2)]
    layer_norm = torch.nn.functional.layer_norm
    h = layer_norm(x, (d,), *norm[0], 1e-5)
    qkv = (h @ w[0] + bias[0]).reshape(B, S, 3, H, d // H).permute(2, 0, 3, 1, 4).reshape(3, B * H, S, d // H)
    o = _attention64(*qkv, True)[0].reshape(B, H, S, d // H).permute(0, 2, 1, 3).reshape(B * S, d)
    x2 = x + o @ w[1] + bias[1]
    u = layer_norm(x2, (d,), *norm[1], 1e-5) @ w[2] + bias[2]
    y = x2 + _gelu64(u) @ w[3] + bias[3]
    value = (y - target).square().mean()
    params = [*norm[0], w[0], bias[0], w[1], bias[1], *norm[1], w[2], bias[2], w[3], bias[3]]
    dx, *grads = torch.autograd.grad(value, [x, *params])
    return value.detach(), y.detach(), dx, grads


def exact(case, seed):
    c, kind = case, case["kind"]
    data = _inputs(case, seed)
    if kind == "attention":
        return _exact_attention(case, data)
    wide = {k: [x.double().requires_grad_() for x in v] if isinstance(v, list) else v.double() for k, v in data.items()}
    if kind == "matmul":
        y = torch.matmul(wide["a"], wide["b"])
        return y if c["batch"] > 1 else y[0]
    if kind == "classifier":
        logits = wide["logits"].requires_grad_()
        value = -(wide["target"] * torch.log_softmax(logits, -1)).sum() / c["rows"]
        return value.item(), torch.autograd.grad(value, logits)[0]
    if kind == "mlp":
        w = wide["w"]
        bias = [x.new_zeros(x.shape[1]).requires_grad_() for x in w]
        y = torch.relu(wide["x"] @ w[0] + bias[0]) @ w[1] + bias[1]
        value = -(wide["target"] * torch.log_softmax(y, -1)).sum() / c["rows"]
        return value.item(), y.detach(), list(torch.autograd.grad(value, (w[0], bias[0], w[1], bias[1])))
    x = wide["x"].requires_grad_()
    if kind == "decoder":
        value, y, dx, grads = _exact_decoder(case, x, wide["target"], wide["w"])
        return value.item(), y, dx, grads
    if kind == "linear":
        params = [wide["w"].requires_grad_(), wide["b"].requires_grad_()]
        y = x @ params[0] + params[1]
        y = _gelu64(y) if c["gelu"] else y
    else:
        params = [wide["gamma"].requires_grad_(), wide["beta"].requires_grad_()]
        y = torch.nn.functional.layer_norm(x, (c["features"],), *params, 1e-5)
    return [y.detach(), *torch.autograd.grad(y, [x, *params], wide["grad"])]


# ---- what a pass cannot do without ----


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        n, rows = c["B"] * c["H"] * c["S"] * c["D"], c["B"] * c["H"] * c["S"]
        flops = 4 * n * c["S"] * (0.5 if c["causal"] else 1)
        if not c["grad"]:
            return dict(bytes=16 * n + 4 * rows, flops=flops)
        return dict(bytes=32 * n + 4 * rows, flops=3.5 * flops)  # q, k, v, dO in; O, dQ, dK, dV out
    if kind == "matmul":
        n, k, m = c["n"], c["k"], c["m"]
        return dict(bytes=4 * c["batch"] * (n * k + k * m + n * m), flops=2 * c["batch"] * n * k * m)
    if kind == "linear":
        r, i, o = c["rows"], c["n_in"], c["n_out"]
        return dict(bytes=4 * (2 * r * i + 2 * r * o + 2 * i * o + 2 * o), flops=6 * r * i * o)
    if kind == "layernorm":
        n, d = c["rows"] * c["features"], c["features"]
        return dict(bytes=4 * (4 * n + 4 * d), flops=20 * n)
    if kind == "classifier":
        n = c["rows"] * c["classes"]
        return dict(bytes=4 * 3 * n, flops=10 * n)
    if kind == "mlp":
        r, i, h, o = c["rows"], c["n_in"], c["hidden"], c["n_out"]
        params = i * h + h + h * o + o
        return dict(bytes=4 * (r * i + 2 * r * o + 6 * params), flops=4 * r * i * h + 6 * r * h * o)
    rows, d = c["B"] * c["S"], c["d"]
    params = 12 * d * d + 13 * d
    return dict(bytes=4 * (4 * rows * d + 8 * params),
                flops=6 * rows * 12 * d * d + 3.5 * 2 * rows * c["S"] * d)


def tolerance(case):
    """Against float64 the outputs measure 5e-8 to 1.3e-6 over these ranges (the
    largest: gradients and products whose sums have 4096 terms and more), so
    two correct 32-bit implementations differ by up to about 2.5e-6."""
    return dict(rel=1e-5)
