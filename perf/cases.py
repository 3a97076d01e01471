"""The performance cases: what programs written on irontensor_amd have it do, through its public
entry points, from one token's projection to a whole training step.

`listed()` names the fixed cases, `draw(rng)` gives another one of the same ranges. A case's `kind`
says which entry point it goes through:

  matmul     gemm(out=...): a projection, a weight product or a batch of products, any layout, in
             FP32 or BF16 (FP32 accumulation), with an optional bias
  linear     linear + linear_backward (FP32): a layer's forward, input gradient and weight gradient
  attention  flash_attention_bshd (FP32, head_dim up to 128): inference
  attn_train flash_attention_forward_bhsd + flash_attention_backward (head_dim 64, FP32 or BF16)
  block      GemmStep: one transformer layer and the LM head, every contraction forward and
             backward, as one graph replay
  train      TrainStep: a complete FP32 training step (embedding .. Lion), as one graph replay

Inputs are N(0, 1) activations and upstream gradients, N(0, 0.02) weights and uniform tokens, made on
the GPU by torch from the seed alone.
"""
import math

import torch

import irontensor_amd as it
from irontensor_amd.step import GemmStep, ModelShape
from irontensor_amd.train import TrainStep

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}
_IT = {"f32": it.Precision.FP32, "bf16": it.Precision.BF16}


# ---------------------------------------------------------------- device tensors as torch sees them

class _Shared:
    """A device tensor's memory for torch (shares the buffer and keeps it alive)."""

    def __init__(self, t):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape()), "typestr": "<i2" if t.is_bf16() else "<f4",
                                         "data": (t.ptr, False), "strides": None, "version": 2}


def _view(t):
    v = torch.as_tensor(_Shared(t), device="cuda")
    return v.view(torch.bfloat16) if t.is_bf16() else v


def _filled(values, dtype="f32"):
    t = it.Tensor.empty(list(values.shape), _IT[dtype])
    _view(t).copy_(values)
    return t


class _Inputs:
    """Seeded N(0, std) tensors on the GPU, the same ones in the same order for one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, shape, std=1.0, dtype="f32"):
        return (torch.randn(shape, generator=self.g, device="cuda") * std).to(_TORCH[dtype])

    def tokens(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.g, device="cuda")


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # One token's Q|K|V projection of the 256-wide model: greedy decoding, the smallest call.
        {"name": "qkv_decode_f32", "kind": "matmul", "batch": 1, "m": 1, "n": 768, "k": 256, "ta": False, "tb": True,
         "dtype": "f32", "bias": False},
        # The same projection over a training batch of 16 x 256 tokens.
        {"name": "qkv_f32", "kind": "matmul", "batch": 1, "m": 4096, "n": 768, "k": 256, "ta": False, "tb": True,
         "dtype": "f32", "bias": False},
        # A few tokens against a large weight: decoding, bound by reading the weight.
        {"name": "decode_bf16", "kind": "matmul", "batch": 1, "m": 4, "n": 11008, "k": 4096, "ta": False, "tb": True,
         "dtype": "bf16", "bias": False},
        # The large square product of the GEMM sweep.
        {"name": "square_4096_bf16", "kind": "matmul", "batch": 1, "m": 4096, "n": 4096, "k": 4096, "ta": False,
         "tb": False, "dtype": "bf16", "bias": False},
        # Sizes no tile divides: a user's own model.
        {"name": "ragged_bf16", "kind": "matmul", "batch": 1, "m": 1999, "n": 3001, "k": 1237, "ta": False, "tb": True,
         "dtype": "bf16", "bias": True},
        # A small odd-sized layer with bias, forward and backward.
        {"name": "linear_ragged_f32", "kind": "linear", "rows": 1000, "n_in": 300, "n_out": 701, "bias": True,
         "weight": "f32"},
        # The FP32 LM head over a training batch, forward and backward.
        {"name": "lm_head_f32", "kind": "linear", "rows": 4096, "n_in": 256, "n_out": 16384, "bias": False,
         "weight": "f32"},
        # FP32 inference with 128-wide heads over a ragged prompt.
        {"name": "attention_d128_f32", "kind": "attention", "batch": 2, "heads": 8, "seq": 777, "dim": 128,
         "causal": True},
        # FP32 attention of a training batch: the 256-wide model's shape.
        {"name": "attn_train_f32", "kind": "attn_train", "batch": 16, "heads": 4, "seq": 256, "dtype": "f32",
         "causal": True},
        # BF16 attention at the 1024-token shape.
        {"name": "attn_train_bf16", "kind": "attn_train", "batch": 16, "heads": 8, "seq": 1024, "dtype": "bf16",
         "causal": True},
        # One layer and the LM head of the medium BF16 model, with gate|up biases.
        {"name": "block_medium_bf16", "kind": "block", "hidden": 1024, "ffn": 2816, "vocab": 32768, "batch": 8,
         "seq": 1024, "dtype": "bf16"},
        # The complete FP32 training step of the 4-layer, 256-wide model.
        {"name": "train_step_f32", "kind": "train", "layers": 4, "hidden": 256, "ffn": 688, "vocab": 16384,
         "batch": 16, "seq": 256},
    ]


_MOST = 2.2e12  # operations of one drawn case: below the largest listed one


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """Log-uniform; half of them multiples of 16 (model widths), half anything."""
    v = _log(rng, lo, hi)
    return max(16, v // 16 * 16) if rng.random() < 0.5 and hi >= 16 else v


def draw(rng):
    while True:
        kind = rng.choice(["matmul", "matmul", "matmul", "linear", "linear", "attention", "attn_train", "attn_train",
                           "block", "train"])
        if kind == "matmul":
            batch = 1 if rng.random() < 0.8 else _log(rng, 2, 64)
            layout = rng.choice([(False, False), (False, True), (True, False)])
            c = {"kind": kind, "batch": batch, "m": _size(rng, 1, 8192), "n": _size(rng, 16, 16384),
                 "k": _size(rng, 16, 11008), "ta": layout[0], "tb": layout[1], "dtype": rng.choice(["f32", "bf16"]),
                 "bias": rng.random() < 0.3}
            if c["dtype"] == "f32" and _flops(c) > 3e11:
                continue
        elif kind == "linear":
            c = {"kind": kind, "rows": _size(rng, 16, 8192), "n_in": _size(rng, 32, 4096),
                 "n_out": _size(rng, 32, 16384), "bias": rng.random() < 0.5,
                 "weight": "bf16" if rng.random() < 0.2 else "f32"}
            if _flops(c) > 4e11:
                continue
        elif kind == "attention":
            c = {"kind": kind, "batch": _log(rng, 1, 16), "heads": _log(rng, 1, 16), "seq": _size(rng, 16, 2048),
                 "dim": rng.choice([32, 64, 128]), "causal": rng.random() < 0.8}
            if c["batch"] * c["heads"] * c["seq"] ** 2 > 1.4e8:
                continue
        elif kind == "attn_train":
            c = {"kind": kind, "batch": _log(rng, 1, 16), "heads": _log(rng, 1, 16), "seq": _size(rng, 16, 4096),
                 "dtype": rng.choice(["f32", "bf16"]), "causal": rng.random() < 0.8}
            if c["batch"] * c["heads"] * c["seq"] ** 2 > 1.4e8:
                continue
        elif kind == "block":
            heads = _log(rng, 2, 16)
            c = {"kind": kind, "hidden": 64 * heads, "ffn": 16 * _log(rng, 8, 176), "vocab": _size(rng, 1000, 32768),
                 "batch": _log(rng, 1, 8), "seq": _size(rng, 64, 1024), "dtype": rng.choice(["f32", "bf16"])}
            if c["dtype"] == "f32" and _flops(c) > 3e11:
                continue
        else:
            heads = rng.choice([2, 4, 4, 8])
            c = {"kind": kind, "layers": rng.randint(1, 4), "hidden": 64 * heads, "ffn": 8 * _log(rng, 32, 172),
                 "vocab": _size(rng, 1000, 16384), "batch": _log(rng, 1, 16), "seq": _size(rng, 32, 512)}
            if _flops(c) > 2.5e11:
                continue
        if _flops(c) <= _MOST:
            return c


# ---------------------------------------------------------------- inputs

def _matmul_inputs(c, seed):
    r = _Inputs(seed)
    lead = [] if c["batch"] == 1 else [c["batch"]]
    a = r.normal(lead + ([c["k"], c["m"]] if c["ta"] else [c["m"], c["k"]]), 1.0, c["dtype"])
    b = r.normal(lead + ([c["n"], c["k"]] if c["tb"] else [c["k"], c["n"]]), 0.02, c["dtype"])
    return a, b, r.normal([c["n"]], 0.02) if c["bias"] else None


def _linear_inputs(c, seed):
    r = _Inputs(seed)
    return (r.normal([c["rows"], c["n_in"]]), r.normal([c["n_out"], c["n_in"]], 0.02, c["weight"]),
            r.normal([c["n_out"]], 0.02) if c["bias"] else None, r.normal([c["rows"], c["n_out"]]))


def _attention_inputs(c, seed):
    r = _Inputs(seed)
    return [r.normal([c["batch"], c["seq"], c["heads"], c["dim"]]) for _ in range(3)]


def _attn_train_inputs(c, seed):
    r = _Inputs(seed)
    return [r.normal([c["batch"], c["heads"], c["seq"], 64], 1.0, c["dtype"]) for _ in range(4)]


def _block_inputs(c, seed):
    """By the GemmStep's names; activations and upstream gradients N(0, 1), weights N(0, 0.02)."""
    r = _Inputs(seed)
    t, h, f, v, d = c["batch"] * c["seq"], c["hidden"], c["ffn"], c["vocab"], c["dtype"]
    act = {"X": [t, h], "X2": [t, h], "Hf": [t, h], "dlogits": [t, v], "dZ": [t, h], "dGU": [t, 2 * f], "dY": [t, h],
           "dO": [t, h]}
    weights = {"Wqkv": [3 * h, h], "Wo": [h, h], "Wgu": [2 * f, h], "Wd": [h, f], "E": [v, h]}
    got = {n: r.normal(s, 1.0, d) for n, s in act.items()}
    got.update({n: r.normal(s, 0.02, d) for n, s in weights.items()})
    got["bgu"] = r.normal([2 * f], 0.02)
    return got


def _train_inputs(c, seed):
    """Parameters in the TrainStep's order, then the token ids and the next-token targets."""
    r = _Inputs(seed)
    h, f, v = c["hidden"], c["ffn"], c["vocab"]
    params = [r.normal([v, h], 0.02), 1.0 + r.normal([h], 0.1), r.normal([v, h], 0.02)]
    for _ in range(c["layers"]):
        params += [1.0 + r.normal([h], 0.1), 1.0 + r.normal([h], 0.1), r.normal([3 * h, h], 0.02),
                   r.normal([h, h], 0.02), r.normal([2 * f, h], 0.02), r.normal([h, f], 0.02)]
    stream = r.tokens(c["batch"] * (c["seq"] + 1), v).view(c["batch"], c["seq"] + 1)
    return params, stream[:, :-1].reshape(-1), stream[:, 1:].reshape(-1)


# ---------------------------------------------------------------- prepare and run

#: A GemmStep's results that one pass writes.
_BLOCK_OUT = ("QKV", "O", "Y", "G", "U", "Hh", "Z", "logits", "dE", "dHf", "dHh", "dX2", "dOp", "dQKV", "dX", "dWd",
              "dWgu", "dWo", "dWqkv")


def _one(v):
    """A per-layer list's only tensor, or the tensor."""
    return v[0] if isinstance(v, list) else v


def prepare(case, seed):
    c = case
    torch.cuda.synchronize()  # torch fills device memory that the library's stream may have used before
    s = {"kind": c["kind"]}
    if c["kind"] == "matmul":
        a, b, bias = _matmul_inputs(c, seed)
        s.update(a=_filled(a, c["dtype"]), b=_filled(b, c["dtype"]), ta=c["ta"], tb=c["tb"])
        s["bias"] = None if bias is None else _filled(bias)
        lead = [] if c["batch"] == 1 else [c["batch"]]
        s["out"] = it.Tensor.empty(lead + [c["m"], c["n"]], _IT[c["dtype"]])
        s["result"] = _view(s["out"])
    elif c["kind"] == "linear":
        x, w, bias, dy = _linear_inputs(c, seed)
        s.update(x=_filled(x), w=_filled(w, c["weight"]), dy=_filled(dy), bias=None if bias is None else _filled(bias))
    elif c["kind"] == "attention":
        s.update(zip("qkv", map(_filled, _attention_inputs(c, seed))), causal=c["causal"])
    elif c["kind"] == "attn_train":
        s.update(zip(("q", "k", "v", "do"), (_filled(t, c["dtype"]) for t in _attn_train_inputs(c, seed))),
                 causal=c["causal"], out=_IT[c["dtype"]])
    elif c["kind"] == "block":
        shape = ModelShape("block", 1, c["hidden"], c["hidden"] // 64, 64, c["ffn"], c["vocab"], c["batch"], c["seq"])
        step = GemmStep(shape, precision=_IT[c["dtype"]], ffn_bias=True)
        step.ctx.sync()
        for name, value in _block_inputs(c, seed).items():
            _view(_one(getattr(step, name))).copy_(value)
        torch.cuda.synchronize()
        step.enqueue()
        step.capture()
        s.update(step=step, result={n: _view(_one(getattr(step, n))) for n in _BLOCK_OUT})
    else:
        shape = ModelShape("train", c["layers"], c["hidden"], c["hidden"] // 64, 64, c["ffn"], c["vocab"], c["batch"],
                           c["seq"])
        step = TrainStep(shape)
        params, ids, targets = _train_inputs(c, seed)
        step.set_batch(ids.cpu().numpy(), targets.cpu().numpy())
        step.enqueue()  # sizes the library's workspaces
        step.capture()
        step.ctx.sync()
        for t, value in zip(step.params, params):  # the run's starting point
            _view(t).copy_(value)
        for t in step.momentum:
            _view(t).zero_()
        s.update(step=step, result={"loss": _view(step.loss), "losses": _view(step.losses),
                                    "norm_clip": _view(step.norm_clip), "grads": [_view(t) for t in step.grads]})
    torch.cuda.synchronize()
    return s


def run(state):
    s = state
    if s["kind"] == "matmul":
        it.gemm(s["a"], s["b"], trans_a=s["ta"], trans_b=s["tb"], bias=s["bias"], out=s["out"])
        return s["result"]
    if s["kind"] == "linear":
        y = it.linear(s["x"], s["w"], s["bias"])
        dx, dw = it.linear_backward(s["dy"], s["x"], s["w"])
        return [_view(t) for t in (y, dx, dw)]
    if s["kind"] == "attention":
        return _view(it.flash_attention_bshd(s["q"], s["k"], s["v"], s["causal"]))
    if s["kind"] == "attn_train":
        o, lse = it.flash_attention_forward_bhsd(s["q"], s["k"], s["v"], s["causal"], out_precision=s["out"])
        grads = it.flash_attention_backward(s["do"], s["q"], s["k"], s["v"], s["causal"], o=o, lse=lse,
                                            out_precision=s["out"])
        return [_view(t) for t in (o, lse) + tuple(grads)]
    if s["kind"] == "block":
        s["step"].replay()
        return s["result"]
    s["step"].step()
    return s["result"]


# ---------------------------------------------------------------- what a pass cannot do without

def _pairs(c):
    """Query-key pairs of an attention call."""
    q = c["seq"]
    return c["batch"] * c["heads"] * (q * (q + 1) / 2 if c.get("causal", True) else q * q)


def _flops(c):
    if c["kind"] == "matmul":
        return 2.0 * c["batch"] * c["m"] * c["n"] * c["k"]
    if c["kind"] == "linear":
        return 6.0 * c["rows"] * c["n_in"] * c["n_out"]
    if c["kind"] == "attention":
        return 4.0 * _pairs(c) * c["dim"]
    if c["kind"] == "attn_train":
        return 14.0 * _pairs(c) * 64
    t, h, layers = c["batch"] * c["seq"], c["hidden"], c.get("layers", 1)
    attn = 14.0 * _pairs(dict(c, heads=h // 64)) * 64
    return layers * (6.0 * t * h * (4 * h + 3 * c["ffn"]) + attn) + 6.0 * t * h * c["vocab"]


def work(case):
    c = case
    e = 2 if c.get("dtype") == "bf16" else 4
    if c["kind"] == "matmul":
        n = c["batch"] * (c["m"] * c["k"] + c["k"] * c["n"] + c["m"] * c["n"])
        b = e * n + (4 * c["n"] if c["bias"] else 0)
    elif c["kind"] == "linear":
        b = (4 * (2 * c["rows"] * (c["n_in"] + c["n_out"]) + c["n_in"] * c["n_out"])
             + (2 if c["weight"] == "bf16" else 4) * c["n_in"] * c["n_out"])
    elif c["kind"] == "attention":
        b = 16 * c["batch"] * c["seq"] * c["heads"] * c["dim"]
    elif c["kind"] == "attn_train":
        b = c["batch"] * c["heads"] * c["seq"] * (8 * e * 64 + 4)
    elif c["kind"] == "block":
        t, h, f, v = c["batch"] * c["seq"], c["hidden"], c["ffn"], c["vocab"]
        weights = 4 * h * h + 3 * h * f + h * v
        read = e * (t * (6 * h + 2 * f + v) + weights)
        b = read + e * t * (3 * h + 3 * h + 3 * f + v + 3 * h) + 4 * (weights + t * (4 * h + f))
    else:
        h, f, v = c["hidden"], c["ffn"], c["vocab"]
        params = 2 * h * v + h + c["layers"] * (4 * h * h + 3 * h * f + 2 * h)
        b = 4 * 5 * params + 12 * c["batch"] * c["seq"]  # weights and momentum read and written, gradients written
    return {"bytes": float(b), "flops": float(_flops(c))}


def tolerance(case):
    """Largest relative error (2-norm) another correct implementation of the same precision shows:
    about four times what the results are off their 64-bit values. FP32 sums measured 3e-7 to 1.2e-6
    (longest sums: 11008 terms); BF16 results 1.7e-3 for one rounding of the output and 3.2e-3 through
    attention and its projection. A training step's gradients measured 1.3e-6, and on a second step
    the weights whose update changed sign (Lion steps by a fixed amount) add about 3e-5."""
    if case["kind"] == "train":
        return {"rel": 1e-4}
    return {"rel": 1e-2} if case.get("dtype") == "bf16" else {"rel": 1e-5}


# ---------------------------------------------------------------- the same in 64 bits

def _softmax(s, causal):
    if causal:
        n = s.shape[-1]
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    return torch.softmax(s, -1), torch.logsumexp(s, -1)


def _attend(q, k, v, causal):
    """[.., seq, dim] -> (output, log-sum-exp, probabilities)."""
    p, lse = _softmax(torch.matmul(q, k.transpose(-1, -2)) / math.sqrt(q.shape[-1]), causal)
    return torch.matmul(p, v), lse, p


def _attend_backward(do, q, k, v, o, p):
    dv = torch.matmul(p.transpose(-1, -2), do)
    ds = p * (torch.matmul(do, v.transpose(-1, -2)) - (do * o).sum(-1, keepdim=True))
    scale = 1.0 / math.sqrt(q.shape[-1])
    return torch.matmul(ds, k) * scale, torch.matmul(ds.transpose(-1, -2), q) * scale, dv


def _heads(x, batch, seq, heads):
    """[tokens, heads * dim] -> [batch, heads, seq, dim]."""
    return x.view(batch, seq, heads, -1).transpose(1, 2)


def _tokens(x):
    """[batch, heads, seq, dim] -> [tokens, heads * dim]."""
    b, h, s, d = x.shape
    return x.transpose(1, 2).reshape(b * s, h * d)


def _exact_block(c, seed):
    i = {n: t.double() for n, t in _block_inputs(c, seed).items()}
    h, f, heads = c["hidden"], c["ffn"], c["hidden"] // 64
    o = {"QKV": i["X"] @ i["Wqkv"].T}
    q, k, v = (_heads(t, c["batch"], c["seq"], heads) for t in o["QKV"].split(h, 1))
    att, _, p = _attend(q, k, v, True)
    o["O"] = _tokens(att)
    o["Y"] = o["O"] @ i["Wo"].T
    o["G"], o["U"] = (i["X2"] @ i["Wgu"].T + i["bgu"]).split(f, 1)
    o["Hh"] = torch.nn.functional.silu(o["G"]) * o["U"]
    o["Z"] = o["Hh"] @ i["Wd"].T
    o["logits"] = i["Hf"] @ i["E"].T
    o["dE"], o["dHf"] = i["dlogits"].T @ i["Hf"], i["dlogits"] @ i["E"]
    o["dHh"], o["dWd"] = i["dZ"] @ i["Wd"], i["dZ"].T @ o["Hh"]
    o["dX2"], o["dWgu"] = i["dGU"] @ i["Wgu"], i["dGU"].T @ i["X2"]
    o["dOp"], o["dWo"] = i["dY"] @ i["Wo"], i["dY"].T @ o["O"]
    do = _heads(i["dO"], c["batch"], c["seq"], heads)
    o["dQKV"] = torch.cat([_tokens(t) for t in _attend_backward(do, q, k, v, att, p)], 1)
    o["dX"], o["dWqkv"] = o["dQKV"] @ i["Wqkv"], o["dQKV"].T @ i["X"]
    return {n: o[n] for n in _BLOCK_OUT}


def _rms(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * gamma


def _rope(x):
    """Rotates the pairs (2i, 2i + 1) of [batch, heads, seq, dim] by position * 10000^(-2i / dim)."""
    _, _, s, d = x.shape
    freq = 10000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    angle = torch.arange(s, dtype=torch.float64, device=x.device)[:, None] * freq
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], -1).flatten(-2)


def _exact_train(c, seed):
    params, ids, targets = _train_inputs(c, seed)
    p = [t.double().requires_grad_() for t in params]
    b, s, h, f = c["batch"], c["seq"], c["hidden"], c["ffn"]
    x = p[0][ids]
    for l in range(c["layers"]):
        attn_norm, ffn_norm, wqkv, wo, wgu, wd = p[3 + 6 * l: 9 + 6 * l]
        q, k, v = (_heads(t, b, s, h // 64) for t in (_rms(x, attn_norm) @ wqkv.T).split(h, 1))
        x = x + _tokens(_attend(_rope(q), _rope(k), v, True)[0]) @ wo.T
        gate, up = (_rms(x, ffn_norm) @ wgu.T).split(f, 1)
        x = x + (torch.nn.functional.silu(gate) * up) @ wd.T
    losses = torch.nn.functional.cross_entropy(_rms(x, p[1]) @ p[2].T, targets, reduction="none")
    loss = losses.mean()
    grads = torch.autograd.grad(loss, p)
    norm = torch.sqrt(sum((g * g).sum() for g in grads))
    clip = torch.clamp(1.0 / norm, max=1.0)
    return {"loss": loss.detach().view(1), "losses": losses.detach(), "norm_clip": torch.stack([norm, clip]),
            "grads": list(grads)}


def exact(case, seed):
    c = case
    if c["kind"] == "matmul":
        a, b, bias = (None if t is None else t.double() for t in _matmul_inputs(c, seed))
        y = torch.matmul(a.transpose(-1, -2) if c["ta"] else a, b.transpose(-1, -2) if c["tb"] else b)
        return y if bias is None else y + bias
    if c["kind"] == "linear":
        x, w, bias, dy = (None if t is None else t.double() for t in _linear_inputs(c, seed))
        y = x @ w.T
        return [y if bias is None else y + bias, dy @ w, dy.T @ x]
    if c["kind"] == "attention":
        q, k, v = (t.double().transpose(1, 2) for t in _attention_inputs(c, seed))
        return _attend(q, k, v, c["causal"])[0].transpose(1, 2).contiguous()
    if c["kind"] == "attn_train":
        q, k, v, do = (t.double() for t in _attn_train_inputs(c, seed))
        o, lse, p = _attend(q, k, v, c["causal"])
        return [o, lse.reshape(-1, c["seq"])] + list(_attend_backward(do, q, k, v, o, p))
    return _exact_block(c, seed) if c["kind"] == "block" else _exact_train(c, seed)
