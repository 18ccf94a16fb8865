"""The C++ autograd nodes and decode step (csrc/torch_ops.cpp) against the Python
ones they stand in for: the same bits over the forms the operators accept, and
the same behaviour under the features that act on an autograd node.  The products
of few rows, summed in another order than torch's, within a tolerance."""
import types

import pytest
import torch
import torch.nn.functional as F

from lizard_reproduction_amd import _ops, kernels
from lizard_reproduction_amd import layer as hip_layer
from lizard_reproduction_amd.layer import LizardAttention
from tests.helpers import max_rel

pytestmark = pytest.mark.gpu


def _through_python(monkeypatch, fn):
    with monkeypatch.context() as m:
        m.setattr(_ops, "plain", lambda: False)
        return fn()


def _step(op, tensors, requires):
    leaves = [t.detach().requires_grad_(r) for t, r in zip(tensors, requires)]
    y = op(*leaves)
    got = [y.detach()]
    if any(requires):
        g = torch.Generator(device="cuda").manual_seed(3)
        y.backward(torch.randn(y.shape, device="cuda", generator=g).to(y.dtype))
        got += [t.grad for t in leaves]
    return got


def _forms(t, form):
    """The same values in another dtype or layout."""
    if form == "strided":
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    return t.to({"bf16": torch.bfloat16, "fp32": torch.float32, "fp16": torch.float16}[form])


FORMS = [("bf16",) * 3, ("fp32",) * 3, ("bf16", "fp32", "fp16"), ("strided", "bf16", "strided")]


@pytest.mark.parametrize("forms", FORMS)
@pytest.mark.parametrize("requires", [(True,) * 4, (False,) * 4, (False, True, False, True)])
@pytest.mark.parametrize("shape, features, dim, per_head", [
    ((1, 2, 1), 16, 16, False), ((2, 3, 77), 24, 20, True), ((1, 2, 130), 256, 128, False),
    ((1, 2, 0), 16, 16, True)])
def test_gla_node_gives_the_python_nodes_bits(monkeypatch, forms, requires, shape, features, dim,
                                              per_head):
    g = torch.Generator(device="cuda").manual_seed(1)
    fq, fk = (torch.rand(*shape, features, device="cuda", generator=g) for _ in range(2))
    v = torch.randn(*shape, dim, device="cuda", generator=g)
    lg = F.logsigmoid(torch.randn(shape if per_head else (shape[0], shape[2]), device="cuda",
                                  generator=g))
    tensors = [_forms(t, f) for t, f in zip((fq, fk, v), forms)] + [lg]
    ours = _step(kernels.gla, tensors, requires)
    theirs = _through_python(monkeypatch, lambda: _step(kernels.gla, tensors, requires))
    for a, b in zip(ours, theirs):
        assert (a is None) == (b is None)
        assert a is None or (a.dtype == b.dtype and torch.equal(a, b))


@pytest.mark.parametrize("forms", FORMS)
@pytest.mark.parametrize("requires", [(True,) * 4, (False,) * 4, (True, False, False, False)])
@pytest.mark.parametrize("shape, window, sinks", [((1, 2, 1, 16), 4, 2), ((2, 3, 77, 64), 16, 0),
                                                  ((1, 2, 150, 128), 100, 4)])
def test_swa_node_gives_the_python_nodes_bits(monkeypatch, forms, requires, shape, window, sinks):
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(shape, device="cuda", generator=g) for _ in range(3))
    meta = torch.randn(sinks, device="cuda", generator=g)
    tensors = [_forms(t, f) for t, f in zip((q, k, v), forms)] + [meta]

    def op(*a):
        return kernels.swa(*a, window)
    ours = _step(op, tensors, requires)
    theirs = _through_python(monkeypatch, lambda: _step(op, tensors, requires))
    for a, b in zip(ours, theirs):
        assert (a is None) == (b is None)
        assert a is None or (a.dtype == b.dtype and torch.equal(a, b))


def _gla_leaves():
    g = torch.Generator(device="cuda").manual_seed(1)
    fq, fk = (torch.rand(1, 2, 70, 16, device="cuda", generator=g).bfloat16().requires_grad_()
              for _ in range(2))
    v = torch.randn(1, 2, 70, 16, device="cuda", generator=g).bfloat16().requires_grad_()
    return fq, fk, v, F.logsigmoid(torch.randn(1, 70, device="cuda", generator=g)).requires_grad_()


def test_saved_tensor_hooks_see_the_saved_operands():
    leaves, packed = _gla_leaves(), []

    def pack(t):
        packed.append(tuple(t.shape))
        return t.cpu()
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        y = kernels.gla(*leaves)
    plain = kernels.gla(*leaves)
    dy = torch.ones_like(y)
    assert packed == [tuple(t.shape) for t in leaves]
    for a, b in zip(torch.autograd.grad(y, leaves, dy), torch.autograd.grad(plain, leaves, dy)):
        assert torch.equal(a, b)


def test_changed_operands_second_backward_and_transforms_are_refused():
    fq, fk, v, lg = _gla_leaves()
    y = kernels.gla(fq, fk, v, lg)
    with torch.no_grad():
        fk.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()
    y = kernels.gla(fq, fk, v, lg)
    y.sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
    # gradients of gradients have no graph
    y = kernels.gla(fq, fk, v, lg)
    dv, = torch.autograd.grad(y.float().sum(), v, create_graph=True)
    assert not dv.requires_grad or dv.grad_fn is None
    with pytest.raises(RuntimeError):
        torch.func.vmap(kernels.gla)(*(t.detach()[None] for t in (fq, fk, v, lg)))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: kernels.gla(fq, fk, t, lg).float().sum())(v.detach())
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):
        kernels.gla(fq, fk, torch.autograd.forward_ad.make_dual(v, torch.ones_like(v)), lg)


@pytest.mark.parametrize("heads, kv, dim, dtype, rope_batched, window, prompt", [
    (4, 2, 64, torch.bfloat16, False, 16, 40), (4, 4, 64, torch.float32, True, 64, 10),
    (2, 1, 64, torch.bfloat16, True, 5, 0), (4, 2, 128, torch.bfloat16, False, 16, 40),
    (2, 2, 32, torch.float32, False, 7, 3)])
def test_native_layer_step_equals_the_step_by_operators(monkeypatch, heads, kv, dim, dtype,
                                                        rope_batched, window, prompt):
    """Prompt (none, shorter and longer than the window), then steps through the
    ring's wrap: outputs, state and caches bit for bit, the projections formed by
    the modules on both sides."""
    torch.manual_seed(heads)
    monkeypatch.setattr(LizardAttention, "_step_rows", lambda *a: False)
    native = []
    step_native = LizardAttention._step_native
    monkeypatch.setattr(LizardAttention, "_step_native",
                        lambda *a: native.append(step_native(*a)) or native[-1])
    cfg = types.SimpleNamespace(hidden_size=dim * heads, num_attention_heads=heads,
                                num_key_value_heads=kv)
    layer = LizardAttention(cfg, 0, window=window, feature_dim=32).to("cuda", dtype)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0, 0.2)
    b, steps = 3, 9
    x = torch.randn(b, prompt + steps, dim * heads, device="cuda").to(dtype)
    angle = torch.rand(prompt + steps, dim, device="cuda") * 6
    cos, sin = angle.cos().to(dtype), angle.sin().to(dtype)

    def tables(lo, hi):
        c, s = cos[lo:hi], sin[lo:hi]
        return (c.expand(b, -1, -1), s.expand(b, -1, -1)) if rope_batched else (c, s)

    def run():
        if prompt:
            with torch.no_grad():
                y, cache = layer.prefill(x[:, :prompt], tables(0, prompt))
            outs = [y]
        else:
            cache, outs = layer.new_cache(b), []
        for t in range(prompt, prompt + steps):
            outs.append(layer.step(x[:, t:t + 1], tables(t, t + 1), cache))
        return outs + [cache.state, cache.k, cache.v]
    ours = run()
    theirs = _through_python(monkeypatch, run)
    assert native == [True] * steps + [False] * steps
    for a, c in zip(ours, theirs):
        assert torch.equal(a, c)


@pytest.mark.parametrize("rows, cols, sizes", [
    (1, 8, [1]), (16, 64, [16, 17, 15, 1]), (3, 72, [33]), (5, 2048, [48, 16, 16, 1]),
    (16, 2056, [100, 7]), (2, 4104, [16]), (7, 136, [512, 128, 128, 1])])
def test_rows_linear_matches_the_product(rows, cols, sizes):
    """Edges of the 16-row tiles, of the 64-column steps and of the waves' shares
    of them (a share holds 4 steps of 64 columns in flight, 8 waves apart)."""
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(rows, 1, cols, device="cuda", generator=g).bfloat16()
    w = [torch.randn(n, cols, device="cuda", generator=g).bfloat16() for n in sizes]
    wide = [i % 2 == 1 for i in range(len(w))]
    for y, m, f32 in zip(_ops.load().rows_linear(x, w, wide), w, wide):
        exact = x.double() @ m.double().T
        assert y.dtype == (torch.float32 if f32 else torch.bfloat16) and y.shape == exact.shape
        assert torch.equal(y, y.bfloat16().to(y.dtype))
        # half a bf16 unit, and fp32 sums of `cols` products of N(0, 1) values
        bound = 2.0 ** -8 * exact.abs() + 2.0 ** -22 * cols
        assert ((y.double() - exact).abs() <= bound).all()


def _decode_layer(batch=3, heads=4):
    torch.manual_seed(5)
    cfg = types.SimpleNamespace(hidden_size=256, num_attention_heads=heads,
                                num_key_value_heads=heads // 2)
    layer = LizardAttention(cfg, 0, window=8, feature_dim=32).to("cuda", torch.bfloat16)
    with torch.no_grad():
        for n, p in layer.named_parameters():
            p.normal_(0, 0.2 if n.startswith("phi") else 0.06)
    x = torch.randn(batch, 20, 256, device="cuda").bfloat16()
    angle = torch.rand(20, 256 // heads, device="cuda") * 6
    return layer, x, (angle.cos().bfloat16(), angle.sin().bfloat16())


def _decode(layer, x, tables):
    _, cache = layer.prefill(x[:, :10], tuple(t[:10] for t in tables))
    outs = [layer.step(x[:, t:t + 1], tuple(u[t:t + 1] for u in tables), cache)
            for t in range(10, 20)]
    return torch.cat(outs, 1), cache


@pytest.mark.parametrize("batch, heads", [(1, 4), (16, 4), (17, 4), (3, 2)])
def test_step_with_its_projections_matches_the_forward(batch, heads):
    """Sixteen sequences are the most the skinny products take; head_dim 64 and 128."""
    layer, x, tables = _decode_layer(batch, heads)
    assert layer._step_rows(x[:, :1]) == (batch <= 16)
    out, _ = _decode(layer, x, tables)
    with torch.no_grad():
        y = layer(x, tables)[0][:, 10:]
    assert max_rel(out, y) <= 2e-2   # bf16 projections, outputs and o_proj, each rounded once


def test_step_leaves_modules_that_do_more_to_their_forward():
    """Hooked, patched, replaced, autocast and half-precision projections."""
    layer, x, tables = _decode_layer()
    plain, _ = _decode(layer, x, tables)
    token = x[:, :1]
    calls = []
    handle = layer.k_proj.register_forward_hook(lambda *a: calls.append(1))
    assert not layer._step_rows(token)
    hooked, _ = _decode(layer, x, tables)
    assert len(calls) == 11   # the prompt and ten steps
    assert max_rel(hooked, plain) <= 2e-2
    handle.remove()
    assert layer._step_rows(token)
    layer.q_proj.forward = lambda t, f=layer.q_proj.forward: 2 * f(t)
    assert not layer._step_rows(token)
    del layer.q_proj.forward
    with torch.autocast("cuda", dtype=torch.float16):
        assert not layer._step_rows(token)
    o_proj = layer.o_proj
    layer.o_proj = torch.nn.Sequential(o_proj)
    assert not layer._step_rows(token)
    layer.o_proj = torch.nn.Linear(256, 256, device="cuda", dtype=torch.bfloat16)   # a bias
    assert not layer._step_rows(token)
    layer.o_proj = o_proj
    assert layer._step_rows(token) and not layer._step_rows(token.float())
    assert not layer._step_rows(x.reshape(-1)[1:257].view(1, 1, 256))   # not 16-byte aligned


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name, inputs, outputs, error", [
    ("phi_k", 64, 16, ValueError), ("k_proj", 256, 64, ValueError), ("v_proj", 256, 256, ValueError),
    ("q_proj", 256, 128, ValueError), ("q_proj", 128, 256, RuntimeError),
    ("k_proj", 128, 128, RuntimeError), ("o_proj", 128, 256, RuntimeError)])
def test_step_refuses_modules_of_other_sizes(dtype, name, inputs, outputs, error):
    """The errors of the operators' step (prologue_forward's and torch's), and the
    layer decodes on once its own module is back."""
    layer, x, tables = _decode_layer()
    layer, x, tables = layer.to(dtype), x.to(dtype), tuple(t.to(dtype) for t in tables)
    plain, _ = _decode(layer, x, tables)
    _, cache = layer.prefill(x[:, :10], tuple(t[:10] for t in tables))
    own = getattr(layer, name)
    setattr(layer, name, torch.nn.Linear(inputs, outputs, bias=False, device="cuda", dtype=dtype))
    with pytest.raises(error):
        layer.step(x[:, 10:11], tuple(t[10:11] for t in tables), cache)
    setattr(layer, name, own)
    assert torch.equal(_decode(layer, x, tables)[0], plain)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_step_takes_a_gate_logit_per_head(monkeypatch, dtype):
    """W_gamma with an output per head: the operators' step, each head decaying by
    its own gate."""
    layer, x, tables = _decode_layer()
    layer, x, tables = layer.to(dtype), x.to(dtype), tuple(t.to(dtype) for t in tables)
    layer.W_gamma = torch.nn.Linear(256, 4, bias=False, device="cuda", dtype=dtype)
    calls = []
    layer.W_gamma.register_forward_hook(lambda *a: calls.append(1))

    def run():
        cache = layer.new_cache(3)
        return torch.cat([layer.step(x[:, t:t + 1], tuple(u[t:t + 1] for u in tables), cache)
                          for t in range(9)], 1), cache.state
    y, state = run()
    assert len(calls) == 9
    for a, b in zip((y, state), _through_python(monkeypatch, run)):
        assert torch.equal(a, b)
    # the normaliser state of the keys and gates that the steps saw, 9 fp32 sums
    z = torch.zeros(3, 4, 64, device="cuda", dtype=torch.float64)
    for t in range(9):
        row = x[:, t:t + 1]
        fk = hip_layer.prologue_forward(layer.q_proj(row), layer.k_proj(row), layer.v_proj(row),
                                        layer.phi_q.weight, layer.phi_k.weight,
                                        *(u[t:t + 1] for u in tables), 4, 2)[1]
        gate = torch.sigmoid(layer.W_gamma(row).double())[:, 0, :, None]
        z = gate * z + fk[:, :, 0].double().repeat_interleave(2, 1)
    assert max_rel(kernels.split_state(state, 64, 64)[1], z) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name, shape, error", [
    ("alpha_blend", (3,), RuntimeError), ("meta_tokens", (2, 2), ValueError),
    ("meta_tokens", (), ValueError)])
def test_step_refuses_blends_and_sinks_of_other_shapes(dtype, name, shape, error):
    layer, x, tables = _decode_layer()
    layer, x, tables = layer.to(dtype), x.to(dtype), tuple(t.to(dtype) for t in tables)
    setattr(layer, name, torch.nn.Parameter(torch.ones(shape, device="cuda", dtype=dtype)))
    with pytest.raises(error):
        layer.step(x[:, :1], tuple(t[:1] for t in tables), layer.new_cache(3))


@pytest.mark.parametrize("name", ["q_proj", "k_proj", "v_proj", "W_gamma", "o_proj"])
def test_step_runs_replaced_modules(name):
    layer, x, tables = _decode_layer()
    plain, _ = _decode(layer, x, tables)
    setattr(layer, name, torch.nn.Sequential(getattr(layer, name)))
    assert max_rel(_decode(layer, x, tables)[0], plain) <= 2e-2   # the products rounded apart
