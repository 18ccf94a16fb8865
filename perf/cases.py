"""Cases for timing the attention path end to end through its public entry points.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (inputs, a layer, a decode cache) on the GPU from a seed,
``run`` makes one pass, ``exact`` computes the same outputs in float64 with
plain torch, ``work`` counts the bytes and operations the pass cannot do
without and ``tolerance`` says how far two correct implementations at the same
precision may lie apart.  ``draw`` makes further cases of the same ranges.

Paths:

* ``gla_forward``, ``gla_train``: ``kernels.gla`` on ``[B, H, L, .]`` operands,
  without and with gradients;
* ``swa_train``: ``kernels.swa`` with its gradients;
* ``layer_train``, ``layer_prefill``, ``layer_step``: ``LizardAttention``
  training pass, prompt pass with its decode cache, and one decode step.
"""
import math
import types

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from lizard_reproduction_amd import kernels
from lizard_reproduction_amd.layer import LizardAttention

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
ROPE_THETA = 500000.0
ROPE_ROWS = 32768     # positions a decoding program keeps RoPE rows for
CHUNK = 64            # tokens per chunk of the chunked GLA algorithm (work())
TINY = torch.finfo(torch.float32).tiny


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _gla(path, batch, heads, length, features, dim, head_gate, dtype="bf16"):
    return dict(path=path, batch=batch, heads=heads, length=length, features=features, dim=dim,
                head_gate=head_gate, dtype=dtype)


def _swa(batch, heads, length, dim, window, sinks=4, dtype="bf16"):
    return dict(path="swa_train", batch=batch, heads=heads, length=length, dim=dim,
                window=window, sinks=sinks, dtype=dtype)


def _layer(path, batch, length, hidden, heads, kv_heads, feature_dim, window, dtype="bf16"):
    return dict(path=path, batch=batch, length=length, hidden=hidden, heads=heads,
                kv_heads=kv_heads, feature_dim=feature_dim, window=window, dtype=dtype)


def listed():
    return [
        # the smallest call a program makes: one short sequence, evaluation
        dict(_gla("gla_forward", 1, 4, 256, 64, 64, False), name="gla_forward_short"),
        # batched evaluation at head_dim 128 with a gate per head
        dict(_gla("gla_forward", 16, 32, 2048, 128, 128, True), name="gla_forward_batch"),
        # training on one sequence, head_dim 64: little work per launch
        dict(_gla("gla_train", 1, 32, 2048, 64, 64, False), name="gla_train_one"),
        # training on a full batch, head_dim 128: the largest operator call
        dict(_gla("gla_train", 16, 32, 2048, 128, 128, True), name="gla_train_batch"),
        # training on one long document: few (b, h) rows, long walks
        dict(_gla("gla_train", 1, 32, 16384, 128, 128, True), name="gla_train_long"),
        # ragged sizes from fp32 tensors: head_dim 96, nothing a power of two
        dict(_gla("gla_train", 3, 12, 1777, 96, 96, False, "fp32"), name="gla_train_ragged"),
        # sliding window, one sequence, narrow window
        dict(_swa(1, 32, 2048, 64, 64), name="swa_train_one"),
        # sliding window at the layer's default width, head_dim 128
        dict(_swa(4, 32, 4096, 128, 128), name="swa_train_wide"),
        # one attention layer of a small grouped-query model, training step
        dict(_layer("layer_train", 4, 4096, 2048, 32, 8, 128, 64), name="layer_train"),
        # the same at head_dim 128 with the layer's default options
        dict(_layer("layer_train", 1, 4096, 4096, 32, 8, 128, 128), name="layer_train_hd128"),
        # serving: a prompt of odd length into a decode cache
        dict(_layer("layer_prefill", 2, 3001, 2048, 32, 8, 128, 64), name="layer_prefill"),
        # serving: one token for each of a few sequences
        dict(_layer("layer_step", 4, 500, 2048, 32, 8, 128, 64), name="layer_step"),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(["gla_forward", "gla_train", "gla_train", "swa_train", "swa_train",
                       "layer_train", "layer_prefill", "layer_step"])
    dtype = "fp32" if rng.random() < 0.2 else "bf16"
    if path.startswith("gla"):
        heads = rng.choice([4, 8, 12, 16, 24, 32])
        batch = rng.choice([1, 1, 2, 3, 4, 8, 16])
        # at most the (batch, head, token) rows of the largest listed call
        length = _spread(rng, 64, min(16384, 1048576 // (batch * heads)))
        features = rng.choice([32, 64, 64, 96, 128, 128])
        dim = features if rng.random() < 0.7 else rng.choice([32, 64, 96, 128])
        return _gla(path, batch, heads, length, features, dim, rng.random() < 0.5, dtype)
    if path == "swa_train":
        heads = rng.choice([4, 8, 12, 16, 24, 32])
        batch = rng.choice([1, 1, 2, 3, 4])
        length = _spread(rng, 64, min(8192, 524288 // (batch * heads)))
        return _swa(batch, heads, length, rng.choice([32, 64, 64, 96, 128, 128]),
                    rng.choice([16, 32, 64, 64, 100, 128, 128, 256]), rng.choice([1, 4, 4, 8]),
                    dtype)
    # layers: (hidden, heads, kv heads) of head_dim 64 and 128, grouped and not
    hidden, heads, kv = rng.choice([(1024, 16, 16), (1024, 16, 4), (2048, 32, 8), (2048, 16, 4),
                                    (2048, 16, 16)])
    feature_dim = rng.choice([32, 64, 64, 128])
    window = rng.choice([32, 64, 128])
    if path == "layer_train":
        batch = rng.choice([1, 1, 2, 4])
        length = _spread(rng, 128, 8192 // batch)
    else:
        batch = _spread(rng, 1, 16)
        length = _spread(rng, 64, 8192 // batch)
        # decoding takes F = 2 feature_dim <= 128 at head_dim 128
        if hidden // heads == 128:
            feature_dim = min(feature_dim, 64)
    return _layer(path, batch, length, hidden, heads, kv, feature_dim, window, dtype)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _gla_inputs(case, seed):
    """Hedgehog features (the two softmaxes of a row, as the layer makes
    them), values, gate logs and the output's gradient."""
    g, dtype = _generator(seed), DTYPES[case["dtype"]]
    b, h, n, f, d = (case[k] for k in ("batch", "heads", "length", "features", "dim"))

    def features():
        x = _randn(g, b, h, n, f // 2)
        return torch.cat([x.softmax(-1), (-x).softmax(-1)], -1).to(dtype)
    fq, fk = features(), features()
    v = _randn(g, b, h, n, d).to(dtype)
    gate = 2 + 1.5 * _randn(g, b, h, n) if case["head_gate"] else 3 + _randn(g, b, n)
    dy = _randn(g, b, h, n, d).bfloat16()
    return (fq, fk, v, F.logsigmoid(gate)), dy


def _rope_tables(rows, dim, dtype):
    """RoPE cos and sin, [rows, dim]."""
    inv = 1.0 / ROPE_THETA ** (torch.arange(0, dim, 2, device="cuda", dtype=torch.float64) / dim)
    angle = torch.outer(torch.arange(rows, device="cuda", dtype=torch.float64), inv)
    angle = torch.cat([angle, angle], -1)
    return angle.cos().to(dtype), angle.sin().to(dtype)


def _rotate(x):
    half = x.shape[-1] // 2
    return torch.cat([-x[..., half:], x[..., :half]], -1)


def _swa_inputs(case, seed):
    g, dtype = _generator(seed), DTYPES[case["dtype"]]
    shape = tuple(case[k] for k in ("batch", "heads", "length", "dim"))
    cos, sin = _rope_tables(case["length"], case["dim"], torch.float32)
    q, k, v = (_randn(g, *shape) for _ in range(3))
    q, k = (t * cos + _rotate(t) * sin for t in (q, k))
    meta = _randn(g, case["sinks"])
    return (q.to(dtype), k.to(dtype), v.to(dtype), meta), _randn(g, *shape).bfloat16()


def _weights(case, g, dtype):
    """Layer parameters: projections of a width-preserving scale, feature maps
    a few times past their initialisation, a gate that mostly remembers."""
    hidden, heads, kv, f = (case[k] for k in ("hidden", "heads", "kv_heads", "feature_dim"))
    hd = hidden // heads
    shapes = {"q_proj.weight": (hidden, hidden), "k_proj.weight": (kv * hd, hidden),
              "v_proj.weight": (kv * hd, hidden), "o_proj.weight": (hidden, hidden),
              "phi_q.weight": (f, hd), "phi_k.weight": (f, hd), "W_gamma.weight": (1, hidden)}
    w = {n: (_randn(g, *s) * (0.1 if n.startswith("phi") else hidden ** -0.5)).to(dtype)
         for n, s in shapes.items()}
    w["meta_tokens"] = (0.5 * _randn(g, 4)).to(dtype)
    w["alpha_blend"] = torch.ones((), device="cuda", dtype=dtype)
    return w


def _layer_inputs(case, seed):
    """(layer parameters, hidden states, RoPE tables, the output's gradient,
    the next token's hidden state)."""
    g, dtype = _generator(seed), DTYPES[case["dtype"]]
    b, n, hidden = (case[k] for k in ("batch", "length", "hidden"))
    w = _weights(case, g, dtype)
    # a direction shared by the tokens, as in trained hidden states; it keeps
    # the gate open
    x = _randn(g, b, n + 1, hidden)
    x = (x + 3.0 * F.normalize(w["W_gamma.weight"].float(), dim=-1)).to(dtype)
    rope = _rope_tables(ROPE_ROWS if case["path"] == "layer_step" else n,
                        hidden // case["heads"], dtype)
    x, token = x[:, :n].contiguous(), x[:, n:].contiguous()
    dy = None
    if case["path"] == "layer_train":
        # in part noise, in part along what the token's own value adds to the
        # output, as a loss's gradient is: on noise alone the sums over all
        # tokens (alpha, the sinks) would cancel to nothing
        kv = case["kv_heads"]
        own = F.linear(x, w["v_proj.weight"]).view(b, n, kv, -1)
        own = F.linear(own.repeat_interleave(case["heads"] // kv, 2).flatten(2),
                       w["o_proj.weight"])
        dy = (_randn(g, b, n, hidden) + 0.5 * own.float()).to(dtype)
    return w, x, rope, dy, token


def _layer_of(case, w):
    config = types.SimpleNamespace(hidden_size=case["hidden"], num_attention_heads=case["heads"],
                                   num_key_value_heads=case["kv_heads"])
    with torch.device("meta"):
        layer = LizardAttention(config, 0, window=case["window"], num_meta=4,
                                feature_dim=case["feature_dim"])
    layer.load_state_dict({n: t.clone() for n, t in w.items()}, assign=True)
    return layer.requires_grad_(case["path"] == "layer_train")


def prepare(case, seed):
    path = case["path"]
    if path.startswith("layer"):
        w, x, (cos, sin), dy, token = _layer_inputs(case, seed)
        layer = _layer_of(case, w)
        state = dict(path=path, layer=layer, x=x, cos=cos, sin=sin, dy=dy, token=token)
        if path == "layer_train":
            x.requires_grad_()
            state["leaves"] = [x] + [p for _, p in sorted(layer.named_parameters())]
        if path == "layer_step":
            n = case["length"]
            state["cache"] = layer.prefill(x, (cos[:n], sin[:n]))[1]
        return state
    inputs, dy = (_gla_inputs if path.startswith("gla") else _swa_inputs)(case, seed)
    if path.endswith("train"):
        inputs = tuple(t.requires_grad_() for t in inputs)
    return dict(path=path, inputs=inputs, dy=dy, window=case.get("window"))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    path = state["path"]
    if path == "gla_forward":
        with torch.no_grad():
            return kernels.gla(*state["inputs"])
    if path == "gla_train":
        y = kernels.gla(*state["inputs"])
        return (y,) + torch.autograd.grad(y, state["inputs"], state["dy"])
    if path == "swa_train":
        y = kernels.swa(*state["inputs"], state["window"])
        return (y,) + torch.autograd.grad(y, state["inputs"], state["dy"])
    layer, rope = state["layer"], (state["cos"], state["sin"])
    if path == "layer_train":
        y, _ = layer(state["x"], rope)
        return (y,) + torch.autograd.grad(y, state["leaves"], state["dy"])
    if path == "layer_prefill":
        y, cache = layer.prefill(state["x"], rope)
    else:
        cache = state["cache"]
        at = cache.pos % ROPE_ROWS
        y = layer.step(state["token"], (rope[0][at:at + 1], rope[1][at:at + 1]), cache)
    return y, cache.state, cache.k, cache.v


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------

def _dense_gla(fq, fk, v, lg):
    """fq, fk [H, L, F], v [H, L, D], lg [H or 1, L]: the defining sums."""
    n = fq.shape[1]
    decay = lg.cumsum(-1)
    decay = decay[:, :, None] - decay[:, None, :]
    causal = torch.ones(n, n, dtype=torch.bool, device=fq.device).tril()
    w = (fq @ fk.transpose(1, 2)) * decay.masked_fill(~causal, -math.inf).exp()
    return (w @ v) / w.sum(-1, keepdim=True).clamp_min(TINY)


def _dense_swa(q, k, v, meta, window):
    """q, k, v [H, L, d]: softmax over the window and the sinks."""
    h, n, d = q.shape
    at = torch.arange(n, device=q.device)
    ahead = at[:, None] - at[None, :]
    s = (q @ k.transpose(1, 2)) / math.sqrt(d)
    s = s.masked_fill((ahead < 0) | (ahead >= window), -math.inf)
    s = torch.cat([meta.expand(h, n, meta.numel()), s], -1)
    return s.softmax(-1)[..., meta.numel():] @ v


def _slices(function, heads, length):
    """function over head slices that fit, recomputed in the backward."""
    step = max(1, min(heads, 2 ** 29 // (length * length)))

    def sliced(*operands):
        parts = []
        for lo in range(0, heads, step):
            part = [t[lo:lo + step] if t.dim() > 1 and t.shape[0] == heads else t
                    for t in operands]
            parts.append(checkpoint(function, *part, use_reentrant=False))
        return torch.cat(parts)
    return sliced


def _wide(t):
    return t.detach().double().requires_grad_(t.requires_grad)


def _exact_gla(case, seed):
    inputs, dy = _gla_inputs(case, seed)
    train = case["path"] == "gla_train"
    wide = [t.double().requires_grad_(train) for t in inputs]
    run_slices = _slices(_dense_gla, case["heads"], case["length"])
    y, grads = [], [[] for _ in wide]
    for i in range(case["batch"]):
        one = [t[i].detach().requires_grad_(train) for t in wide]
        gate = one[3] if case["head_gate"] else one[3][None].expand(case["heads"], -1)
        out = run_slices(one[0], one[1], one[2], gate)
        y.append(out.detach())
        if train:
            for into, grad in zip(grads, torch.autograd.grad(out, one, dy[i].double())):
                into.append(grad)
    return (torch.stack(y),) + tuple(torch.stack(g) for g in grads) if train else torch.stack(y)


def _exact_swa(case, seed):
    inputs, dy = _swa_inputs(case, seed)
    run_slices = _slices(lambda q, k, v, m: _dense_swa(q, k, v, m, case["window"]),
                         case["heads"], case["length"])
    meta = inputs[3].double().requires_grad_()
    y, grads, dmeta = [], [[], [], []], torch.zeros_like(meta)
    for i in range(case["batch"]):
        one = [t[i].double().requires_grad_() for t in inputs[:3]]
        out = run_slices(*one, meta)
        y.append(out.detach())
        *rest, dm = torch.autograd.grad(out, one + [meta], dy[i].double())
        for into, grad in zip(grads, rest):
            into.append(grad)
        dmeta = dmeta + dm
    return (torch.stack(y),) + tuple(torch.stack(g) for g in grads) + (dmeta,)


def _exact_layer(case, seed):
    weights, x, (cos, sin), dy, token = _layer_inputs(case, seed)
    path, heads, kv = case["path"], case["heads"], case["kv_heads"]
    train, step = path == "layer_train", path == "layer_step"
    w = {n: t.double().requires_grad_(train) for n, t in weights.items()}
    x = (torch.cat([x, token], 1) if step else x).double().requires_grad_(train)
    b, n, hidden = x.shape
    hd, group = hidden // heads, heads // kv
    cos, sin = cos[:n].double(), sin[:n].double()

    def split(t, count):
        return t.view(n, count, hd).transpose(0, 1)

    def hedgehog(t, phi):
        p = t @ phi.T
        return torch.cat([p.softmax(-1), (-p).softmax(-1)], -1)

    def repeat(t):
        return t.repeat_interleave(group, 0)

    gla = _slices(_dense_gla, heads, n)
    swa = _slices(lambda q, k, v, m: _dense_swa(q, k, v, m, case["window"]), heads, n)
    rows, states, keys, values = [], [], [], []
    for i in range(b):
        q, k, v = (split(x[i] @ w[name + ".weight"].T, count) for name, count in
                   (("q_proj", heads), ("k_proj", kv), ("v_proj", kv)))
        lg = F.logsigmoid(x[i] @ w["W_gamma.weight"][0])
        fq, fk = hedgehog(q, w["phi_q.weight"]), hedgehog(k, w["phi_k.weight"])
        qr, kr = (t * cos + _rotate(t) * sin for t in (q, k))
        y = gla(fq, repeat(fk), repeat(v), lg.expand(heads, n))
        y = y + w["alpha_blend"] * swa(qr, repeat(kr), repeat(v), w["meta_tokens"])
        rows.append(y.transpose(0, 1).reshape(n, hidden) @ w["o_proj.weight"].T)
        if not train:
            g = lg.cumsum(-1)
            left = fk * (g[-1] - g).exp()[None, :, None]
            s, z = left.transpose(1, 2) @ v, left.sum(1)
            states.append(repeat(torch.cat([s.flatten(1), z], -1)))
            keys.append(_ring(kr, case["window"]))
            values.append(_ring(v, case["window"]))
    out = torch.stack(rows)
    if train:
        leaves = [x] + [w[name] for name in sorted(w)]
        return (out.detach(),) + torch.autograd.grad(out, leaves, dy.double())
    return (out[:, -1:] if step else out, torch.stack(states), torch.stack(keys),
            torch.stack(values))


def _ring(t, window):
    """[heads, n, hd] -> the last ``window`` rows, position p in slot p % window."""
    heads, n, hd = t.shape
    ring = t.new_zeros(heads, window, hd)
    at = torch.arange(max(0, n - window), n, device=t.device)
    ring[:, at % window] = t[:, at]
    return ring


def exact(case, seed):
    if case["path"].startswith("gla"):
        return _exact_gla(case, seed)
    if case["path"] == "swa_train":
        return _exact_swa(case, seed)
    with torch.set_grad_enabled(case["path"] == "layer_train"):
        return _exact_layer(case, seed)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _bytes_of(case):
    return 4 if case["dtype"] == "fp32" else 2


def _gla_work(b, h, n, f, d, size, train, gate_bytes):
    rows = b * h * n
    flops = rows * (4 * f * d + 2 * CHUNK * (f + d))
    moved = rows * (size * (2 * f + d) + 2 * d) + gate_bytes
    if train:
        flops = rows * (12 * f * d + 8 * CHUNK * f + 6 * CHUNK * d)
        # the gradient of y in, the gradients of the operands out
        moved += rows * (2 * d + size * (2 * f + d)) + gate_bytes
    return moved, flops


def _swa_work(b, h, n, d, window, size):
    keys = sum(min(i + 1, window) for i in range(n)) / n
    rows = b * h * n
    return rows * (size * 3 * d + 2 * d + 2 * d + size * 3 * d), 14 * d * keys * rows


def work(case):
    path, b, n, heads = case["path"], case["batch"], case["length"], case["heads"]
    size = _bytes_of(case)
    if path.startswith("gla"):
        gates = 4 * b * n * (heads if case["head_gate"] else 1)
        moved, flops = _gla_work(b, heads, n, case["features"], case["dim"], size,
                                 path == "gla_train", gates)
        return {"bytes": moved, "flops": flops}
    if path == "swa_train":
        moved, flops = _swa_work(b, heads, n, case["dim"], case["window"], size)
        return {"bytes": moved, "flops": flops}
    hidden, kv, f = case["hidden"], case["kv_heads"], case["feature_dim"]
    hd = hidden // heads
    weights = 2 * hidden * hidden + 2 * hidden * kv * hd + 2 * f * hd
    state = 4 * b * heads * (2 * f * hd + 2 * f)
    ring = 2 * 2 * b * kv * case["window"] * hd
    if path == "layer_step":
        return {"bytes": size * (weights + 2 * b * hidden) + 2 * state + ring,
                "flops": 2 * b * weights + b * heads * 4 * (2 * f * hd + case["window"] * hd)}
    tokens = b * n
    flops = 2 * tokens * (weights - 2 * f * hd) + 2 * tokens * (heads + kv) * f * hd
    gla = tokens * heads * (4 * 2 * f * hd + 2 * CHUNK * (2 * f + hd))
    swa = 4 * hd * min(n, case["window"]) * tokens * heads
    if path == "layer_prefill":
        return {"bytes": size * (weights + 2 * tokens * hidden) + state + ring,
                "flops": flops + gla + swa}
    return {"bytes": size * (2 * weights + 4 * tokens * hidden),
            "flops": 3 * flops + 3 * gla + 3.5 * swa}


# ---------------------------------------------------------------------------
# how far two correct implementations may lie apart
# ---------------------------------------------------------------------------

def tolerance(case):
    """About four times the distance from ``exact`` that bf16 operands and
    results leave: outputs 2e-3, gradients 2e-3 to 5e-3 (5e-3 through a whole
    layer), the gate's gradient, a suffix sum over the sequence, up to 1.1e-2 at
    16384 tokens; single values reach 0.04 of a tensor's root mean square, in
    the gradients of the features 0.13."""
    path = case["path"]
    if path == "gla_forward":
        return {"rel": 0.01, "max": 0.2}
    if path == "gla_train":
        return {"rel": 0.03 if case["length"] > 8192 else 0.02, "max": 0.5}
    if path == "layer_train":
        return {"rel": 0.02, "max": 0.2}
    return {"rel": 0.016, "max": 0.2}
