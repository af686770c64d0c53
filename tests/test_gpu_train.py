"""Training-batch kernels (attention, QK-norm + RoPE, forward and backward)
against the same formulas in fp64 on the same bf16 inputs.

Bounds: a correctly rounded bf16 result is within 2^-9 of the exact value
element by element, so its relative 2-norm error is at most 2^-9; the fp32
sums and the hi + lo split of the fp32 factors (2^-17 per term) add far less,
for which 1e-4 is allowed.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = 2.0 ** -9 + 1e-4


def _rel(got, ref):
    return ((got.double() - ref).norm() / ref.norm().clamp_min(1e-300)).item()


def _core(q, k, v, batch, scale):
    """fp64 causal attention of [N, heads, 128] rows."""
    n, hq, d = q.shape
    q, k, v = (t.view(batch, n // batch, -1, d).transpose(1, 2) for t in (q, k, v))
    rep = hq // k.shape[1]
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = q @ k.transpose(-1, -2) * scale
    mask = torch.ones(s.shape[-2:], dtype=torch.bool, device=q.device).triu(1)
    return (torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ v).transpose(1, 2).reshape(n, hq, d)


# One token, tile edges and remainders, every group size, and batches large
# enough for 32 rows per wave in the forward / dQ (512 blocks of 128 queries)
# and the dK / dV kernel (512 blocks of 128 keys).
@pytest.mark.parametrize("batch,t,hq,hkv", [
    (1, 1, 16, 8), (2, 63, 16, 8), (1, 64, 4, 4), (3, 65, 8, 2), (2, 129, 6, 2), (1, 389, 16, 8),
    (16, 200, 16, 8), (32, 193, 16, 8), (64, 64, 8, 8)])
def test_train_attention(pkg, gpu, batch, t, hq, hkv):
    g = torch.Generator(device=gpu).manual_seed(batch * 1000 + t)
    n, d, scale = batch * t, 128, 128 ** -0.5
    q = torch.randn(n, hq, d, generator=g, device=gpu).mul(2).bfloat16()
    k = torch.randn(n, hkv, d, generator=g, device=gpu).mul(2).bfloat16()
    qkv = torch.randn(n, (hq + 2 * hkv) * d, generator=g, device=gpu).bfloat16()
    v = qkv[:, (hq + hkv) * d:].view(n, hkv, d)
    do = torch.randn(n, hq, d, generator=g, device=gpu).bfloat16()
    out, out32, stats = pkg.kernels.train_attention(q, k, v, batch, scale, True)
    dv = torch.full_like(qkv, 7.0)
    dq, dk = pkg.kernels.train_attention_backward(q, k, v, batch, scale, out32, stats, do,
                                                  dv[:, (hq + hkv) * d:])
    ref_in = [x.double().requires_grad_() for x in (q, k, v)]
    ref = _core(*ref_in, batch, scale)
    ref.backward(do.double())
    assert _rel(out32, ref) < 2e-5
    assert _rel(out, ref) < BF16
    for name, got, want in (("dq", dq, ref_in[0].grad), ("dk", dk, ref_in[1].grad),
                            ("dv", dv[:, (hq + hkv) * d:].view(n, hkv, d), ref_in[2].grad)):
        # One token: dS is exactly zero in fp64 and rounding noise in fp32.
        assert _rel(got, want) < BF16 or (t == 1 and name != "dv" and got.abs().max() < 1e-4), name
    assert bool((dv[:, :(hq + hkv) * d] == 7.0).all())
    no_grad, none32, _ = pkg.kernels.train_attention(q, k, v, batch, scale, False)
    assert none32 is None and torch.equal(no_grad, out)


@pytest.mark.parametrize("batch,t,hq,hkv", [(1, 1, 16, 8), (3, 37, 8, 2), (2, 389, 16, 8), (1, 5, 1, 1)])
def test_qk_norm_rope_backward(pkg, gpu, batch, t, hq, hkv):
    g = torch.Generator(device=gpu).manual_seed(t)
    n, d, eps = batch * t, 128, 1e-6
    qkv = torch.randn(n, (hq + 2 * hkv) * d, generator=g, device=gpu).bfloat16()
    qw, kw = ((torch.rand(d, generator=g, device=gpu) * 0.4 + 0.8).bfloat16() for _ in range(2))
    dq = torch.randn(n, hq, d, generator=g, device=gpu).bfloat16()
    dk = torch.randn(n, hkv, d, generator=g, device=gpu).bfloat16()
    cache = pkg.RotaryEmbedding(d, 512, 1e6).cos_sin_cache.to(gpu)
    q, k = pkg.kernels.qk_norm_rope_seq(qkv, qw, kw, t, cache, hq, hkv, eps)
    pos = torch.arange(t, device=gpu).repeat(batch)
    q2, k2 = pkg.kernels.qk_norm_rope(qkv, qw, kw, pos, cache, hq, hkv, eps)
    assert torch.equal(q, q2) and torch.equal(k, k2)
    dqkv = torch.zeros_like(qkv)
    dqw, dkw = pkg.kernels.qk_norm_rope_backward(dq, dk, qkv, qw, kw, t, cache, eps, dqkv)
    x, a, b = (z.double().requires_grad_() for z in (qkv, qw, kw))
    c, s = cache[pos][:, None, :64].double(), cache[pos][:, None, 64:].double()

    def rot(y, w):
        y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + eps) * w
        return torch.cat((y[..., :64] * c - y[..., 64:] * s, y[..., 64:] * c + y[..., :64] * s), -1)

    xh = x.view(n, -1, d)
    torch.autograd.backward([rot(xh[:, :hq], a), rot(xh[:, hq:hq + hkv], b)],
                            [dq.double(), dk.double()])
    for got, want in ((dqkv, x.grad), (dqw, a.grad), (dkw, b.grad)):
        assert _rel(got, want) < BF16


def _attn(pkg, gpu, seed=0):
    torch.manual_seed(seed)
    a = pkg.Qwen3Attention(pkg.Qwen3Config(hidden_size=256, num_attention_heads=4,
                                           num_key_value_heads=2, max_position_embeddings=512))
    with torch.no_grad():
        for name, p in a.named_parameters():
            p.uniform_(0.8, 1.2) if "norm" in name else p.normal_(0, 0.06)
    return a.to(gpu).bfloat16()


def test_attention_module_matches_formula(pkg, gpu):
    """The module through the kernels and, with a hook on q_norm (which the
    kernels would pass by), through the torch formula: same values, same
    gradients, up to the bf16 roundings in between."""
    T = pkg.qwen3_naive.T
    a = _attn(pkg, gpu)
    x = torch.randn(2, 70, 256, device=gpu).bfloat16().requires_grad_()
    dy = torch.randn(2, 70, 256, device=gpu).bfloat16()
    seen, calls, real = [], [], T.QkvAttention.apply
    T.QkvAttention.apply = lambda *args: (calls.append(1), real(*args))[1]
    try:
        res = []
        for hook in (False, True):
            h = a.q_norm.register_forward_hook(lambda *_: seen.append(1)) if hook else None
            a.zero_grad()
            x.grad = None
            y = a(x)
            y.backward(dy)
            res.append([y.detach(), x.grad] + [p.grad for p in a.parameters()])
            if h:
                h.remove()
    finally:
        T.QkvAttention.apply = real
    assert len(calls) == 1 and len(seen) == 1
    for got, want in zip(*res):
        assert _rel(got, want.double()) < 0.02


def test_attention_second_derivative(pkg, gpu):
    """create_graph: a gradient penalty through the attention differentiates the formula."""
    T = pkg.qwen3_naive.T
    a = _attn(pkg, gpu)
    cache = a._cos_sin(torch.device(gpu))
    qkv = torch.randn(1, 9, 8 * 128, device=gpu).bfloat16().requires_grad_()
    args = (cache, 4, 2, a.eps, a.scale)
    res = []
    for fused in (True, False):
        if fused:
            o = T.QkvAttention.apply(qkv, a.q_norm.weight, a.k_norm.weight, *args)
        else:
            o = T.attention_formula(qkv, a.q_norm, a.k_norm, cache, 4, 2, a.scale)
        g, = torch.autograd.grad(o.float().sum(), qkv, create_graph=True)
        gg, = torch.autograd.grad(g.float().square().sum(), qkv)
        res.append(gg)
    assert res[0].abs().max() > 0 and _rel(res[0], res[1].double()) < 0.05
