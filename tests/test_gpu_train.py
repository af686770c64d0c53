"""The training batch's fused autograd Functions against the torch formulas
they stand for.  Forward values and the gradients that flow on are the same
bit for bit, but where a sum has another order: the norm weights' gradients, and
k's and v's over four query heads per KV head, agree to one bf16 rounding (half
an ulp of 8 significant bits, 2^-8)."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def T(pkg):
    return importlib.import_module(pkg.__name__ + ".train_ops")


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def _both(fused, formula, inputs, seed=3):
    res = []
    for f in (fused, formula):
        leaves = [t.detach().clone().requires_grad_() for t in inputs]
        y = f(*leaves)
        g = torch.Generator(device=y.device).manual_seed(seed)
        y.backward(torch.randn(y.shape, generator=g, device=y.device).bfloat16())
        res.append([y] + [t.grad for t in leaves])
    return res


# One row; rows that leave lane groups idle; the narrowest row, one whose
# chunks do not divide a workgroup, one of several passes per workgroup.
@pytest.mark.parametrize("shape", [(1, 1024), (2, 389, 1024), (3, 24), (1500, 8), (7, 2056), (5, 4096)])
def test_rms_norm(T, gpu, shape):
    g = torch.Generator(device=gpu).manual_seed(shape[0])
    x = torch.randn(shape, generator=g, device=gpu).bfloat16()
    w = torch.rand(shape[-1], generator=g, device=gpu).bfloat16() + 0.5
    a, b = _both(lambda x, w: T.RmsNorm.apply(x, w, 1e-6), lambda x, w: T.rms_norm_formula(x, w, 1e-6),
                 (x, w))
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and _rel(a[2], b[2]) < 2 ** -8


@pytest.mark.parametrize("shape", [(1, 16), (3, 5, 48), (2, 389, 6144)])
def test_silu_mul(T, gpu, shape):
    gu = (torch.randn(shape, device=gpu) * 4).bfloat16()
    gu[..., 0], gu[..., 1] = 200.0, -200.0  # saturated gates
    a, b = _both(T.SiluMul.apply, T.silu_mul_formula, (gu,))
    assert all(torch.equal(p, q) for p, q in zip(a, b))


# Token counts around the transposing tile and the softmax's chunk (64), not a
# multiple of 4, around the fused softmax's longest row (1,024); one token; query heads per KV head 1, 2 and 4.
@pytest.mark.parametrize("b,t", [(1, 1), (2, 33), (1, 64), (3, 65), (1, 130), (2, 700), (1, 1024),
                                 (1, 1025), (1, 1152)])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (4, 2), (8, 2)])
def test_attention(pkg, T, gpu, b, t, hq, hkv):
    g = torch.Generator(device=gpu).manual_seed(b * t)
    qkv = torch.randn(b, t, (hq + 2 * hkv) * 128, generator=g, device=gpu).bfloat16()
    qw, kw = (torch.rand(128, generator=g, device=gpu).bfloat16() + 0.5 for _ in range(2))
    cache = pkg.qwen3_naive.get_rope(128, 2048, 1e6).cos_sin_cache.to(gpu)

    def formula(qkv, qw, kw):
        return T.attention_formula(qkv, lambda x: T.rms_norm_formula(x, qw, 1e-6),
                                   lambda x: T.rms_norm_formula(x, kw, 1e-6), cache, hq, hkv, 0.09)

    a, ref = _both(lambda *z: T.QkvAttention.apply(*z, cache, hq, hkv, 1e-6, 0.09), formula, (qkv, qw, kw))
    assert torch.equal(a[0], ref[0])
    if hq // hkv <= 2:
        assert torch.equal(a[1], ref[1])
    else:  # four heads' k gradients are added in another order, then rounded
        assert _rel(a[1], ref[1]) < 2 ** -8
    if t > 1:  # one token: the scores have no gradient
        assert _rel(a[2], ref[2]) < 2 ** -8 and _rel(a[3], ref[3]) < 2 ** -8
    else:
        assert not a[2].any() and not ref[2].any()


def test_layer_routes(pkg, T, gpu):
    """The layer takes the fused Functions, unless a norm is hooked or a second
    derivative needs torch ops; same values."""
    torch.manual_seed(0)
    layer = pkg.Qwen3DecoderLayer(pkg.Qwen3Config(
        hidden_size=128, num_attention_heads=2, num_key_value_heads=1, intermediate_size=256,
        num_hidden_layers=1, max_position_embeddings=64)).to(gpu).bfloat16()
    x = torch.randn(2, 33, 128, device=gpu).bfloat16().requires_grad_()
    res, seen = [], []
    for hook in (False, True):
        h = layer.self_attn.q_norm.register_forward_hook(lambda *_: seen.append(1)) if hook else None
        layer.zero_grad()
        x.grad = None
        y = layer(x)
        y.float().square().mean().backward()
        res.append([y.detach(), x.grad])
        if h:
            h.remove()
    assert seen and all(torch.equal(a, b) for a, b in zip(*res))
    # A gradient that is differentiated again: through the formulas.  x's second
    # gradient is the sum of two, here each rounded to bf16 (2^-8) before it.
    out = []
    for f in (lambda: T.RmsNorm.apply(x, layer.input_layernorm.weight, 1e-6),
              lambda: T.rms_norm_formula(x, layer.input_layernorm.weight, 1e-6)):
        g, = torch.autograd.grad(f().float().pow(3).sum(), x, create_graph=True)
        out.append(torch.autograd.grad(g.float().square().sum(), x)[0])
    assert out[0].abs().max() > 0 and _rel(*out) < 2 ** -7
    # Saved tensors that a hook packs and unpacks elsewhere.
    with torch.autograd.graph.save_on_cpu():
        y = layer(x)
    x.grad = None
    y.float().square().mean().backward()
    assert torch.equal(x.grad, res[0][1])
    with torch.no_grad():
        assert not T.norm_ok(x, layer.input_layernorm.weight)


def _layer(pkg, gpu, max_position=64):
    torch.manual_seed(0)
    return pkg.Qwen3DecoderLayer(pkg.Qwen3Config(
        hidden_size=128, num_attention_heads=2, num_key_value_heads=1, intermediate_size=256,
        num_hidden_layers=1, max_position_embeddings=max_position)).to(gpu).bfloat16()


def _grads(layer, y, x):
    y.float().square().mean().backward()
    res = [x.grad] + [p.grad for p in layer.parameters()]
    x.grad = None
    layer.zero_grad()
    return res


# Both softmax forms; the products kept by a selective checkpoint, or every op's result.
@pytest.mark.parametrize("t", [33, 1030])
@pytest.mark.parametrize("keep", ["products", "all"])
def test_selective_checkpoint(pkg, gpu, t, keep):
    from torch.utils import checkpoint as C
    layer = _layer(pkg, gpu, 2048)
    x = torch.randn(1, t, 128, device=gpu).bfloat16().requires_grad_()
    want = _grads(layer, layer(x), x)
    aten = torch.ops.aten
    policy = ([aten.mm.default, aten.bmm.default, aten.addmm.default] if keep == "products" else
              lambda ctx, op, *a, **k: C.CheckpointPolicy.MUST_SAVE)
    y = C.checkpoint(layer, x, use_reentrant=False,
                     context_fn=lambda: C.create_selective_checkpoint_contexts(policy))
    assert all(torch.equal(a, b) for a, b in zip(_grads(layer, y, x), want))


def test_shared_norm_weight_second_derivative(pkg, T, gpu):
    """One weight as both q and k norm: a differentiable gradient counts each use once."""
    g = torch.Generator(device=gpu).manual_seed(7)
    qkv = torch.randn(1, 20, 4 * 128, generator=g, device=gpu).bfloat16()
    w = torch.rand(128, generator=g, device=gpu).bfloat16() + 0.5
    cache = pkg.qwen3_naive.get_rope(128, 64, 1e6).cos_sin_cache.to(gpu)

    def norm(x):
        return T.rms_norm_formula(x, w, 1e-6)

    out = []
    for f in (lambda: T.QkvAttention.apply(qkv, w, w, cache, 2, 1, 1e-6, 0.09),
              lambda: T.attention_formula(qkv, norm, norm, cache, 2, 1, 0.09)):
        qkv, w = qkv.detach().requires_grad_(), w.detach().requires_grad_()
        first = torch.autograd.grad(f().float().pow(3).sum(), (qkv, w), create_graph=True)
        second = torch.autograd.grad(first[0].float().square().sum(), (qkv, w))
        out.append([*first, *second])
    # Two uses' gradients are each rounded to bf16 before they are added (2^-8), and
    # with them the terms of the second derivative.
    assert all(_rel(a, b) < 2 ** -6 for a, b in zip(*out))


def _functions(pkg, T, gpu):
    """(fused, formula, inputs) of the three Functions, small."""
    g = torch.Generator(device=gpu).manual_seed(11)
    x, gu, qkv = (torch.randn(1, 5, n, generator=g, device=gpu).bfloat16() for n in (64, 32, 512))
    w, qw, kw = (torch.rand(n, generator=g, device=gpu).bfloat16() + 0.5 for n in (64, 128, 128))
    cache = pkg.qwen3_naive.get_rope(128, 64, 1e6).cos_sin_cache.to(gpu)
    return [(lambda x, w: T.RmsNorm.apply(x, w, 1e-6), lambda x, w: T.rms_norm_formula(x, w, 1e-6), (x, w)),
            (T.SiluMul.apply, T.silu_mul_formula, (gu,)),
            (lambda *z: T.QkvAttention.apply(*z, cache, 2, 1, 1e-6, 0.09),
             lambda z, a, b: T.attention_formula(z, lambda t: T.rms_norm_formula(t, a, 1e-6),
                                                 lambda t: T.rms_norm_formula(t, b, 1e-6), cache, 2, 1, 0.09),
             (qkv, qw, kw))]


def test_forward_mode_over_a_backward(pkg, T, gpu):
    from torch.autograd import forward_ad as fwAD
    for fused, formula, inputs in _functions(pkg, T, gpu):
        out = []
        for f in (fused, formula):
            leaves = [t.detach().clone().requires_grad_() for t in inputs]
            y = f(*leaves)
            with fwAD.dual_level():
                tangent = torch.linspace(-1, 1, y.numel(), device=gpu).view_as(y).bfloat16()
                dy = fwAD.make_dual(torch.ones_like(y), tangent)
                if len(inputs) == 1:  # torch has no forward mode over silu's gradient
                    with pytest.raises(NotImplementedError):
                        torch.autograd.grad(y, leaves, dy)
                    continue
                got = [fwAD.unpack_dual(g) for g in torch.autograd.grad(y, leaves, dy)]
                assert all(g.tangent is not None for g in got)
                out.append([t.clone() for g in got for t in (g.primal, g.tangent)])
        assert all(torch.equal(a, b) for a, b in zip(*out))


def test_checkpoint_recomputed_under_forward_mode(pkg, gpu):
    """The recomputation of a checkpointed layer saves what its forward did."""
    from torch.autograd import forward_ad as fwAD
    from torch.utils.checkpoint import checkpoint
    layer = _layer(pkg, gpu)
    x = torch.randn(1, 9, 128, device=gpu).bfloat16().requires_grad_()
    want = _grads(layer, layer(x), x)
    y = checkpoint(layer, x, use_reentrant=False)
    with fwAD.dual_level():
        assert all(torch.equal(a, b) for a, b in zip(_grads(layer, y, x), want))


@pytest.mark.parametrize("vmap", ["is_grads_batched", "func"])
def test_batched_gradients(pkg, T, gpu, vmap):
    """A batch of output gradients in one backward gives what one at a time gives."""
    for fused, _, inputs in _functions(pkg, T, gpu):
        leaves = [t.detach().clone().requires_grad_() for t in inputs]
        y = fused(*leaves)
        dys = torch.linspace(-2, 2, 3 * y.numel(), device=gpu).view(3, *y.shape).bfloat16()
        want = [torch.autograd.grad(y, leaves, d, retain_graph=True) for d in dys]
        if vmap == "func":
            got = torch.vmap(lambda d: torch.autograd.grad(y, leaves, d, retain_graph=True))(dys)
        else:
            got = torch.autograd.grad(y, leaves, dys, is_grads_batched=True)
        # Sums over rows in another order, and batched products: one bf16 rounding.
        for i, g in enumerate(got):
            assert _rel(g, torch.stack([w[i] for w in want])) < 2 ** -8


def test_vectorized_jacobian(pkg, gpu):
    layer = _layer(pkg, gpu)
    x = torch.randn(1, 2, 128, device=gpu).bfloat16()
    for p in layer.parameters():
        p.requires_grad_(False)
    a, b = (torch.autograd.functional.jacobian(layer, x, vectorize=v) for v in (True, False))
    assert _rel(a, b) < 2 ** -7


def test_saved_tensors_in_another_layout(pkg, T, gpu):
    """Hooks may give saved tensors back with other strides."""
    def spread(t):
        buf = torch.zeros((*t.shape, 2), dtype=t.dtype, device=t.device)
        buf[..., 0] = t.detach()
        return buf[..., 0]

    for fused, _, inputs in _functions(pkg, T, gpu):
        res = []
        for hooked in (False, True):
            leaves = [t.detach().clone().requires_grad_() for t in inputs]
            if hooked:
                with torch.autograd.graph.saved_tensors_hooks(spread, lambda t: t):
                    y = fused(*leaves)
            else:
                y = fused(*leaves)
            res.append(torch.autograd.grad(y, leaves, torch.linspace(-1, 1, y.numel(), device=gpu).view_as(y).bfloat16()))
        assert all(torch.equal(a, b) for a, b in zip(*res))


# One chunk, several, and the unfused softmax; a value of q, k or v in the
# middle of the rows, upstream gradients of zero before it.
@pytest.mark.parametrize("t", [5, 150, 1030])
@pytest.mark.parametrize("where", [3, 259, 391])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_attention_nonfinite(pkg, T, gpu, t, where, value):
    g = torch.Generator(device=gpu).manual_seed(t)
    qkv = torch.randn(1, t, 512, generator=g, device=gpu).bfloat16()
    qkv[0, t // 2, where] = value
    qw, kw = (torch.rand(128, generator=g, device=gpu).bfloat16() + 0.5 for _ in range(2))
    cache = pkg.qwen3_naive.get_rope(128, 2048, 1e6).cos_sin_cache.to(gpu)
    dy = torch.randn(1, t, 256, generator=g, device=gpu).bfloat16()
    dy[:, :t // 2] = 0
    out = []
    for f in (lambda *z: T.QkvAttention.apply(*z, cache, 2, 1, 1e-6, 0.09),
              lambda z, a, b: T.attention_formula(z, lambda x: T.rms_norm_formula(x, a, 1e-6),
                                                  lambda x: T.rms_norm_formula(x, b, 1e-6), cache, 2, 1, 0.09)):
        leaves = [a.clone().requires_grad_() for a in (qkv, qw, kw)]
        y = f(*leaves)
        y.backward(dy)
        out.append([y] + [a.grad for a in leaves])
    assert not out[1][0].isfinite().all()
    for a, b in zip(out[0][:2], out[1][:2]):
        torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)
    for a, b in zip(out[0][2:], out[1][2:]):
        assert torch.equal(a.isnan(), b.isnan())


def test_rows_nonfinite(pkg, T, gpu):
    for fused, formula, inputs in _functions(pkg, T, gpu)[:2]:
        x = inputs[0].clone()
        for i, value in enumerate((float("inf"), float("-inf"), float("nan"))):
            x[0, i, 3] = x[0, i, 20] = value
        a, b = _both(fused, formula, (x, *inputs[1:]))
        for p, q in zip(a[:2], b[:2]):
            torch.testing.assert_close(p, q, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("part", ["norm", "attention"])
def test_inputs_written_between_forward_and_backward(pkg, gpu, part):
    """A residual stream updated in place, weights stepped and a projection's
    output kept by a hook and written to: the gradients are the forward's."""
    layer = _layer(pkg, gpu)
    attn, norm = layer.self_attn, layer.input_layernorm
    x = torch.randn(1, 9, 128, device=gpu).bfloat16().requires_grad_()
    kept, res = [], []
    cache = attn._cos_sin(gpu)
    for write in (False, True):
        h = x * 1
        hook = attn.qkv_proj.register_forward_hook(lambda m, i, o: kept.append(o)) if write else None
        y = norm(h) if part == "norm" else attn(h)
        if write:
            with torch.no_grad():
                written = [h, norm.weight] if part == "norm" else [attn.q_norm.weight, attn.k_norm.weight,
                                                                    cache, *kept]
                before = [t.clone() for t in written]
                for t in written:
                    t.add_(1)
            hook.remove()
        res.append(_grads(layer, y, x))
        if write:
            with torch.no_grad():
                for t, b in zip(written, before):
                    t.copy_(b)
    assert part == "norm" or kept
    for a, b in zip(*res):
        assert a is b is None or torch.equal(a, b)


@pytest.mark.parametrize("written", [False, True])
def test_second_derivative_after_a_weight_was_written(pkg, T, gpu, written):
    for fused, formula, inputs in _functions(pkg, T, gpu)[::2]:
        out = []
        for f in (fused, formula):
            leaves = [t.detach().clone().requires_grad_() for t in inputs]
            y = f(*leaves)
            if written:
                with torch.no_grad():
                    for w in leaves[1:]:
                        w.add_(1)
            first = torch.autograd.grad(y.float().square().sum(), leaves, create_graph=True)
            second = torch.autograd.grad(sum(g.float().square().sum() for g in first), leaves)
            out.append([*first, *second])
        # Partial gradients are each rounded to bf16 before they are added (2^-8),
        # at both levels.
        assert all(_rel(a, b) < 2 ** -6 for a, b in zip(*out))


def test_traced_layer_holds_its_ops(pkg, gpu):
    """A graph recorded from the layer and its gradient computes them for other inputs."""
    from torch.fx.experimental.proxy_tensor import make_fx
    layer = _layer(pkg, gpu)

    def step(x):
        x = x.detach().requires_grad_()
        y = layer(x)
        return y, torch.autograd.grad(y.float().square().sum(), x)[0]

    a, b = (torch.randn(1, 9, 128, device=gpu).bfloat16() for _ in range(2))
    graph = make_fx(step)(a)
    for got, want in zip(graph(b), step(b)):
        assert _rel(got, want) < 2 ** -7


# Five to eight chunks of the fused softmax (its form for 257 to 512 tokens).
@pytest.mark.parametrize("t", [257, 389, 512])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (4, 2), (8, 2)])
def test_attention_eight_chunks(pkg, T, gpu, t, hq, hkv):
    test_attention(pkg, T, gpu, 2, t, hq, hkv)


def test_layer_on_a_side_stream(pkg, gpu):
    """Forward and backward on another stream than the default one."""
    layer = _layer(pkg, gpu)
    x = torch.randn(2, 33, 128, device=gpu).bfloat16().requires_grad_()
    want = _grads(layer, layer(x), x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = _grads(layer, layer(x), x)
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_backward_under_autocast(pkg, T, gpu):
    """Autocast around the backward alone changes nothing."""
    for fused, _, inputs in _functions(pkg, T, gpu):
        out = []
        for on in (False, True):
            leaves = [t.detach().clone().requires_grad_() for t in inputs]
            y = fused(*leaves)
            with torch.autocast("cuda", dtype=torch.bfloat16, enabled=on):
                out.append(torch.autograd.grad(y, leaves, torch.ones_like(y)))
        assert all(torch.equal(a, b) for a, b in zip(*out))


def test_function_transforms(pkg, gpu):
    """torch.func's grad and vmap run on torch ops."""
    layer = _layer(pkg, gpu)
    x = torch.randn(1, 9, 128, device=gpu).bfloat16()
    leaf = x.clone().requires_grad_()
    want = _grads(layer, layer(leaf), leaf)[0]
    # The products run in other forms there: flipped bf16 roundings along the layer's steps.
    assert _rel(torch.func.grad(lambda z: layer(z).float().square().mean())(x), want) < 0.02
    norm = layer.input_layernorm
    assert torch.equal(torch.func.vmap(norm)(x[0]), norm(leaf)[0])


def test_norm_weight_made_in_inference_mode(pkg, gpu):
    """Such a weight cannot be saved for a backward; the formula saves a copy."""
    norm = pkg.qwen3_naive.RMSNorm(128).to(gpu).bfloat16()
    x = torch.randn(3, 128, device=gpu).bfloat16().requires_grad_()
    norm.requires_grad_(False)
    want = torch.autograd.grad(norm(x).float().square().sum(), x)[0]
    with torch.inference_mode():
        norm.weight = torch.nn.Parameter(norm.weight.clone(), requires_grad=False)
    assert torch.equal(torch.autograd.grad(norm(x).float().square().sum(), x)[0], want)


def test_second_derivative_rounds_where_the_formula_does(pkg, T, gpu):
    """Both parts of a norm's second derivative meet in fp32, as the formula's do:
    the same bits."""
    for fused, formula, inputs in _functions(pkg, T, gpu)[:1]:
        out = []
        for f in (fused, formula):
            leaves = [t.detach().clone().requires_grad_() for t in inputs]
            first = torch.autograd.grad(f(*leaves).float().pow(3).sum(), leaves, create_graph=True)
            second = torch.autograd.grad(sum(g.float().square().sum() for g in first), leaves)
            out.append([*first, *second])
        assert all(torch.equal(a, b) for a, b in zip(*out))


def test_projection_output_kept_by_its_own_forward(pkg, gpu):
    """A forward set on the projection may keep what it returned and write to it."""
    layer = _layer(pkg, gpu)
    x = torch.randn(1, 9, 128, device=gpu).bfloat16().requires_grad_()
    want = _grads(layer, layer(x), x)
    proj, kept = layer.self_attn.qkv_proj, []
    own = proj.forward
    proj.forward = lambda z: kept.append(own(z)) or kept[-1]
    y = layer(x)
    with torch.no_grad():
        kept[0].zero_()
    assert all(torch.equal(a, b) for a, b in zip(_grads(layer, y, x), want))
