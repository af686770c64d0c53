"""Prefill projections (qmi_linear_tiles) and the prefill layer as one library
call (qmi_prefill_layer) against fp32 torch products and the layer's modules.

Tolerances: a projection rounds an fp32 sum once to bf16 (8 significant bits:
half an ulp is at most 2^-8 of the value); the SwiGLU form rounds g, u and the
result.  Two layers that differ in the order of their
fp32 sums differ by flipped roundings along six bf16 steps."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


# Row counts around the tile heights 64, 128 and 256; column counts around the
# tile widths, the narrowest, and one that no form divides; the shortest sums.
@pytest.mark.parametrize("m", [1, 63, 64, 65, 129, 256, 257, 777, 2048])
@pytest.mark.parametrize("n,k", [(16, 64), (208, 128), (1024, 2048), (4096, 192)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_linear_tiles(pkg, gpu, m, n, k, swiglu):
    g = torch.Generator(device=gpu).manual_seed(m + n)
    x = torch.randn(m, k, generator=g, device=gpu).bfloat16()
    w = (torch.randn((2 * n if swiglu else n), k, generator=g, device=gpu) * 0.05).bfloat16()
    y = torch.full((m + 1, n), 7.0, device=gpu).bfloat16()
    st = pkg._lib.lib().qmi_linear_tiles(x.data_ptr(), k, w.data_ptr(), k, m, n, k, int(swiglu),
                                         y.data_ptr(), n, pkg._lib.stream_handle(x.device))
    assert st == 0
    want = x.float() @ w.float().T
    if swiglu:
        gate, up = want.bfloat16().float().chunk(2, -1)
        want = torch.nn.functional.silu(gate) * up
    assert _rel(y[:m], want) < (2 ** -7 if swiglu else 2 ** -8)
    assert bool((y[m] == 7).all())  # nothing past the last row
    assert torch.equal(y[:m], pkg.kernels.linear_tiles(x, w, swiglu))


# The two 192-column forms (ring of three and of two chunks) with partial last
# tiles both ways, at K of fewer chunks than the ring, as many and more; each
# element by itself: one rounding (2^-8 of it) after k terms summed in fp32, in
# the product and its reference (2^-23 k of the terms' magnitudes), and for SwiGLU
# the roundings of gate (silu changes by at most 1 + |g| times its relative
# error), up and the result.
@pytest.mark.parametrize("m", [1000, 1999])
@pytest.mark.parametrize("n,swiglu", [(6128, False), (3056, True)])
@pytest.mark.parametrize("k", [64, 128, 192, 1024])
def test_linear_tiles_wide_forms(pkg, gpu, m, n, swiglu, k):
    g = torch.Generator(device=gpu).manual_seed(m + k)
    x = torch.randn(m, k, generator=g, device=gpu).bfloat16()
    w = (torch.randn((2 * n if swiglu else n), k, generator=g, device=gpu) * 0.05).bfloat16()
    y = torch.full((m + 1, n), 7.0, device=gpu).bfloat16()
    st = pkg._lib.lib().qmi_linear_tiles(x.data_ptr(), k, w.data_ptr(), k, m, n, k, int(swiglu),
                                         y.data_ptr(), n, pkg._lib.stream_handle(x.device))
    assert st == 0
    want = x.float() @ w.float().T
    slack = 2 ** -23 * k * (x.float().abs() @ w.float().abs().T)
    bound = 2 ** -8 * want.abs() + slack
    if swiglu:
        gate, up = want.chunk(2, -1)
        sg, su = slack.chunk(2, -1)
        silu = torch.nn.functional.silu(gate)
        want = silu * up
        bound = 2 ** -8 * want.abs() * (3 + gate.abs()) + 1.1 * sg * up.abs() + su * silu.abs()
        bound = 1.02 * bound + 1e-6  # products of the errors; __expf
    assert bool(((y[:m].float() - want).abs() <= bound).all())
    assert bool((y[m] == 7).all())


def test_linear_tiles_strides(pkg, gpu):
    x = torch.randn(70, 200, device=gpu).bfloat16()[:, 8:136]
    w = torch.randn(48, 160, device=gpu).bfloat16()[:, :128]
    assert _rel(pkg.kernels.linear_tiles(x, w), x.float() @ w.float().T) < 2 ** -8
    with pytest.raises(Exception):
        pkg.kernels.linear_tiles(x[:, :96], w[:, :96])  # K % 64


def _layer(pkg, gpu, hidden=256, heads=4, kv=2, inter=384):
    torch.manual_seed(0)
    cfg = pkg.Qwen3Config(hidden_size=hidden, num_attention_heads=heads, num_key_value_heads=kv,
                          intermediate_size=inter, num_hidden_layers=1, max_position_embeddings=4096)
    layer = pkg.Qwen3DecoderLayer(cfg).to(gpu).bfloat16()
    with torch.no_grad():
        for name, p in layer.named_parameters():
            p.uniform_(0.8, 1.2) if "norm" in name else p.normal_(0, 0.05)
    return layer, cfg


def _batch(layer, cfg, gpu, lens, prefix, seed=0):
    g = torch.Generator(device=gpu).manual_seed(seed)
    width = -(-(max(lens) + prefix) // 256)
    nb = len(lens) * width
    shape = (nb, 256, cfg.num_key_value_heads, 128)
    layer.self_attn.k_cache = torch.randn(shape, generator=g, device=gpu).bfloat16()
    layer.self_attn.v_cache = torch.randn(shape, generator=g, device=gpu).bfloat16()
    bt = torch.arange(nb, dtype=torch.int32, device=gpu).flip(0).view(len(lens), width).contiguous()
    pos = torch.cat([torch.arange(prefix, prefix + n, device=gpu) for n in lens])
    seq = torch.cat([torch.full((n,), b, device=gpu) for b, n in enumerate(lens)])
    slots = (bt.long()[seq, pos // 256] * 256 + pos % 256).to(torch.int32)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    cu_q = torch.tensor(cu, dtype=torch.int32, device=gpu)
    cu_k = (cu_q + prefix * torch.arange(len(cu), device=gpu)).to(torch.int32)
    x = torch.randn(cu[-1], cfg.hidden_size, generator=g, device=gpu).bfloat16()
    r = torch.randn(cu[-1], cfg.hidden_size, generator=g, device=gpu).bfloat16()
    return (x, pos, cu_q, cu_k, max(lens), max(lens) + prefix, slots, bt), r


# One token, the row counts where a projection changes its kernel (64, 256),
# ragged prompts, a cached prefix, and more rows than one call takes (2,048).
@pytest.mark.parametrize("lens,prefix", [([1], 0), ([64], 300), ([65], 0), ([255, 1], 256),
                                         ([257], 0), ([3, 500, 98], 77), ([1024, 1024], 0),
                                         ([1500, 549], 0)])
@pytest.mark.parametrize("first", [False, True])
def test_layer_matches_modules(pkg, gpu, lens, prefix, first):
    layer, cfg = _layer(pkg, gpu)
    args, r = _batch(layer, cfg, gpu, lens, prefix)
    r = None if first else r
    kv = layer.self_attn.k_cache.clone(), layer.self_attn.v_cache.clone()
    seen, res = [], []
    for hook in (False, True):  # a hooked module takes the module path
        layer.self_attn.k_cache, layer.self_attn.v_cache = kv[0].clone(), kv[1].clone()
        h = layer.mlp.down_proj.register_forward_hook(lambda *_: seen.append(1)) if hook else None
        with torch.no_grad():
            y, s = layer.forward_prefill(*args, residual=r)
            native = layer._prefill_native(*args, r)
        assert (native is None) == (hook or sum(lens) > 2048)
        res.append((y, s, layer.self_attn.k_cache, layer.self_attn.v_cache))
        if h:
            h.remove()
    assert seen
    for a, b in zip(*res):
        assert a.shape == b.shape and _rel(a, b) < 0.02


def test_layer_routes(pkg, gpu, monkeypatch):
    """Calls the one-call form does not take run (or fail) as before."""
    layer, cfg = _layer(pkg, gpu)
    args, r = _batch(layer, cfg, gpu, [40], 0)
    with torch.no_grad():
        want = layer.forward_prefill(*args, residual=r)

        def native(*a, residual=r):
            return layer._prefill_native(*a, residual)

        def same(*a, residual=r):
            assert native(*a, residual=residual) is None
            for got, ref in zip(layer.forward_prefill(*a, residual=residual), want):
                assert _rel(got, ref) < 0.02

        assert native(*args) is not None
        wide = torch.cat((args[0], args[0]), 1)[:, :cfg.hidden_size]  # strided rows
        same(wide, *args[1:])
        same(args[0], args[1].int(), *args[2:])
        same(*args[:6], args[6].long(), args[7])
        same(*args, residual=torch.cat((r, r), 1)[:, :cfg.hidden_size])
        assert native(*args[:7], None) is None
        with monkeypatch.context() as mp:
            mp.setattr(pkg.qwen3_naive.Qwen3Attention, "forward_prefill", lambda self, h, *a: h)
            assert native(*args) is None
        with monkeypatch.context() as mp:
            mp.setattr(layer.mlp, "forward", lambda h: h)
            assert native(*args) is None
            assert layer.forward_prefill(*args, residual=r)[0].shape == args[0].shape
        layer.mlp.down_proj.bias = torch.nn.Parameter(torch.zeros(cfg.hidden_size, device=gpu).bfloat16())
        same(*args)
        layer.mlp.down_proj.bias = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            same(*args)
    assert native(*args) is None  # weights tracked by autograd


def test_layer_in_a_graph(pkg, gpu):
    layer, cfg = _layer(pkg, gpu)
    args, r = _batch(layer, cfg, gpu, [100, 30], 0)
    with torch.no_grad():
        want = layer.forward_prefill(*args, residual=r)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            layer.forward_prefill(*args, residual=r)
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = layer.forward_prefill(*args, residual=r)
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want))
            layer.forward_prefill(*args, residual=r)


def test_layer_with_a_subclass_weight(pkg, gpu):
    """A weight whose class has its own product (as a quantised one has) is used through it."""
    seen = []

    class Doubled(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            if func is torch.nn.functional.linear:
                seen.append(1)
                return func(args[0], args[1].as_subclass(torch.Tensor) * 2)
            return super().__torch_function__(func, types, args, kwargs)

    layer, cfg = _layer(pkg, gpu)
    args, r = _batch(layer, cfg, gpu, [40], 0)
    down = layer.mlp.down_proj
    with torch.no_grad():
        want, _ = layer.forward_prefill(*args, residual=r)
        down.weight = torch.nn.Parameter(down.weight.detach().as_subclass(Doubled))
        assert layer._prefill_native(*args, r) is None
        got, _ = layer.forward_prefill(*args, residual=r)
    assert seen and _rel(got, 2 * want) < 0.02


def test_layer_under_a_mode(pkg, gpu):
    """A mode sees the products; a default device is no such mode."""
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    layer, cfg = _layer(pkg, gpu)
    args, r = _batch(layer, cfg, gpu, [40], 0)
    with torch.no_grad():
        with torch.device(gpu):
            assert layer._prefill_native(*args, r) is not None
        with Watch():
            assert layer._prefill_native(*args, r) is None
        with FlopCounterMode(display=False) as counter:
            layer.forward_prefill(*args, residual=r)
    h, i, qkv = cfg.hidden_size, cfg.intermediate_size, 8 * 128
    assert counter.get_total_flops() == 2 * 40 * (h * qkv + 4 * 128 * h + 3 * h * i)


# A wide layer runs natively up to 300 rows; 4,096 columns at two row tiles take
# o_proj and down_proj without a split.
@pytest.mark.parametrize("hidden,rows", [(2560, 300), (2560, 301), (4096, 77), (4096, 128)])
def test_wide_layer(pkg, gpu, hidden, rows):
    layer, cfg = _layer(pkg, gpu, hidden=hidden, heads=8, kv=2, inter=512)
    args, r = _batch(layer, cfg, gpu, [rows], 0)
    with torch.no_grad():
        native = layer._prefill_native(*args, r)
        assert (native is not None) == (rows <= 300)
        got = layer.forward_prefill(*args, residual=r)
        h = layer.mlp.down_proj.register_forward_hook(lambda *_: None)
        want = layer.forward_prefill(*args, residual=r)
        h.remove()
    for a, b in zip(got, want):
        assert _rel(a, b) < 0.02


@pytest.mark.parametrize("heads,kv", [(2, 2), (8, 2)])
def test_layer_head_ratios(pkg, gpu, heads, kv):
    """One and four query heads per KV head, over a cached prefix."""
    layer, cfg = _layer(pkg, gpu, heads=heads, kv=kv)
    args, r = _batch(layer, cfg, gpu, [3, 200], 77)
    cache = layer.self_attn.k_cache.clone()
    with torch.no_grad():
        got = (*layer._prefill_native(*args, r), layer.self_attn.k_cache.clone())
        layer.self_attn.k_cache.copy_(cache)
        h = layer.mlp.down_proj.register_forward_hook(lambda *_: None)
        want = (*layer.forward_prefill(*args, residual=r), layer.self_attn.k_cache)
        h.remove()
    for a, b in zip(got, want):
        assert _rel(a, b) < 0.02
