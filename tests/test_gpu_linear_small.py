"""Decode projections of at most 16 rows (qmi_linear_small) against fp32 torch
products, and the decode layer whose norms run inside them against its modules.

Tolerances: one bf16 rounding of an fp32 sum (8 significant bits: half an ulp
is at most 2^-8 of the value; SwiGLU rounds g, u and the result); the
norm's rows may differ from add_rms_norm's by flipped roundings (another order
of the sum of squares), as may SwiGLU's g and u."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


# The fewest and most rows and those around one per wave; a grid of one
# workgroup (which writes every row of the residual sum) and larger ones.
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("n", [16, 48, 4096])
@pytest.mark.parametrize("k", [1024, 2048, 3072, 4096])
@pytest.mark.parametrize("swiglu", [False, True])
def test_linear_small(pkg, gpu, m, n, k, swiglu):
    K = pkg.kernels
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=gpu).bfloat16()
    r = torch.randn(m, k + 8, generator=g, device=gpu).bfloat16()[:, :k]
    w = (torch.randn((2 * n if swiglu else n), k, generator=g, device=gpu) * 0.05).bfloat16()
    nw = torch.rand(k, generator=g, device=gpu).bfloat16() + 0.5

    def ref(rows):
        y = rows.float() @ w.float().T
        if swiglu:
            gate, up = y.bfloat16().float().chunk(2, -1)
            y = torch.nn.functional.silu(gate) * up
        return y

    tol = 2 ** -7 if swiglu else 2 ** -8
    y, s = K.linear_small(x, w, swiglu)
    assert s is None and y.shape == (m, n) and _rel(y, ref(x)) < tol
    y, s = K.linear_small(x, w, swiglu, nw, 1e-6)
    assert s is None and _rel(y, ref(K.rms_norm(x, nw, 1e-6))) < 2 * tol
    y, s = K.linear_small(x, w, swiglu, nw, 1e-6, r)
    h, total = K.add_rms_norm(x, r, nw, 1e-6)
    assert torch.equal(s, total) and _rel(y, ref(h)) < 2 * tol


# Eight weight rows per workgroup: the fewest columns that take them, and a count
# past whole multiples of the chip.  Each element by itself: one rounding (2^-8)
# after k terms summed in fp32, here and in the reference (2^-23 k of the terms'
# magnitudes); with the norm, rows whose elements may have rounded the other way
# (2^-8 of a term each, 2^-8 of their root sum of squares on average, 8 times that
# over all elements).
@pytest.mark.parametrize("m", [1, 9, 16])
@pytest.mark.parametrize("n", [2048, 3088])
@pytest.mark.parametrize("k", [1024, 2048, 3072, 4096])
def test_linear_small_eight_rows(pkg, gpu, m, n, k):
    K = pkg.kernels
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=gpu).bfloat16()
    r = torch.randn(m, k, generator=g, device=gpu).bfloat16()
    w = (torch.randn(n, k, generator=g, device=gpu) * 0.05).bfloat16()
    nw = torch.rand(k, generator=g, device=gpu).bfloat16() + 0.5
    for rows, args in ((x, ()), (K.rms_norm(x, nw, 1e-6), (nw, 1e-6)),
                       (K.add_rms_norm(x, r, nw, 1e-6)[0], (nw, 1e-6, r))):
        want = rows.float() @ w.float().T
        bound = 2 ** -8 * want.abs() + 2 ** -23 * k * (rows.float().abs() @ w.float().abs().T)
        if args:
            bound = bound + 2 ** -5 * (rows.float().square() @ w.float().square().T).sqrt()
        assert bool(((K.linear_small(x, w, False, *args)[0].float() - want).abs() <= bound).all())


def test_linear_small_refuses(pkg, gpu):
    K = pkg.kernels
    x = torch.zeros(17, 1024, device=gpu).bfloat16()
    w = torch.zeros(32, 1024, device=gpu).bfloat16()
    for a, b, sw in ((x, w, False), (x[:4], w[:24], False), (x[:4, :512], w[:, :512], False),
                     (x[:4], w[:12], True)):
        with pytest.raises(ValueError):
            K.linear_small(a, b, sw)


@pytest.mark.parametrize("batch", [1, 16, 17])
@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("fused_qkv", [False, True])
def test_decode_layer_matches_modules(pkg, gpu, batch, first, fused_qkv):
    torch.manual_seed(0)
    cfg = pkg.Qwen3Config(hidden_size=1024, num_attention_heads=8, num_key_value_heads=4,
                          intermediate_size=2048, num_hidden_layers=1, max_position_embeddings=1024)
    layer = pkg.Qwen3DecoderLayer(cfg).to(gpu).bfloat16()
    layer.self_attn.decode_fused_qkv = fused_qkv
    with torch.no_grad():
        for name, p in layer.named_parameters():
            p.uniform_(0.8, 1.2) if "norm" in name else p.normal_(0, 0.03)
    kv = [torch.randn(batch * 2, 256, 4, 128, device=gpu).bfloat16() for _ in range(2)]
    ctx = (torch.arange(batch, dtype=torch.int32, device=gpu) * 29) % 500
    bt = torch.arange(batch * 2, dtype=torch.int32, device=gpu).view(batch, 2)
    x = torch.randn(batch, 1024, device=gpu).bfloat16()
    r = None if first else torch.randn(batch, 1024, device=gpu).bfloat16()
    res = []
    for hook in (False, True):
        layer.self_attn.k_cache, layer.self_attn.v_cache = kv[0].clone(), kv[1].clone()
        seen = []
        h = (layer.input_layernorm.register_forward_hook(lambda *_: seen.append(1)) if hook else None)
        with torch.no_grad():
            assert layer._norms_in_projections(x, r) == (batch <= 16 and not hook)
            y, s = layer.forward_decode(x, ctx.long(), ctx, bt, None, r)
        res.append([t.dense() if isinstance(t, pkg.kernels.RowParts) else t
                    for t in (y, s, layer.self_attn.k_cache, layer.self_attn.v_cache)])
        if h:
            h.remove()
            assert seen
    for a, b in zip(*res):
        assert a.shape == b.shape and _rel(a, b) < 0.02
    layer.self_attn.k_cache, layer.self_attn.v_cache = kv
    assert not layer._norms_in_projections(x, r)  # weights tracked by autograd


def test_replaced_projection_gets_rows(pkg, gpu, monkeypatch):
    """A program's own _project_store, on the class or one module, is called with
    the normed rows, as a tensor."""
    torch.manual_seed(0)
    cfg = pkg.Qwen3Config(hidden_size=1024, num_attention_heads=8, num_key_value_heads=4,
                          intermediate_size=2048, num_hidden_layers=1, max_position_embeddings=1024)
    layer = pkg.Qwen3DecoderLayer(cfg).to(gpu).bfloat16()
    attn = layer.self_attn
    attn.decode_fused_qkv = False
    attn.k_cache, attn.v_cache = (torch.zeros(2, 256, 4, 128, device=gpu).bfloat16() for _ in range(2))
    ctx = torch.zeros(2, dtype=torch.int32, device=gpu)
    bt = torch.arange(2, dtype=torch.int32, device=gpu).view(2, 1)
    x = torch.randn(2, 1024, device=gpu).bfloat16()
    own, seen = pkg.qwen3_naive.Qwen3Attention._project_store, []

    def wrapped(self, rows, *args, **kwargs):
        seen.append(type(rows))
        return own(self, rows, *args, **kwargs)

    with torch.no_grad():
        for target, name in ((pkg.qwen3_naive.Qwen3Attention, wrapped),
                             (attn, lambda *a, **k: wrapped(attn, *a, **k))):
            with monkeypatch.context() as mp:
                mp.setattr(target, "_project_store", name)
                layer.forward_decode(x, ctx.long(), ctx, bt)
    assert seen == [torch.Tensor] * 2
