"""Which decode projections run on the small-batch kernel, and which prefill steps
as one call (CPU: the rules alone)."""
import torch


def test_norms_in_projections(pkg):
    win = pkg.kernels.norms_in_projections_win
    # Measured on both sides of the rule: layers of depths (hidden, heads, MLP).
    for depths, most in (((1024, 2048, 3072), 14), ((2048, 2048, 3072), 12), ((4096, 2048, 4096), 8),
                         ((1024, 1024, 2048), 16)):
        assert all(win(rows, *depths) == (rows <= most) for rows in range(1, 20))
    assert not win(0, 1024, 2048, 3072)
    # A layer with a depth that the kernel does not have keeps its norms.
    assert not win(1, 2560, 4096, 9728) and not win(1, 2048, 2048, 6144) and not win(1, 4096, 4096, 12288)


def test_single_projections(pkg):
    win = pkg.kernels.linear_small_wins
    for k, most in ((1024, 8), (2048, 8), (3072, 2), (4096, 8), (2560, 0)):
        assert all(win(torch.empty(rows, k)) == (rows <= most) for rows in range(1, 18))


def test_prefill_layer_sizes(pkg):
    ok = pkg.kernels.prefill_layer_size_ok
    for hidden, qkv, inter, most in ((1024, 4096, 3072, 2048), (2048, 4096, 6144, 1024),
                                     (2560, 6144, 9728, 300), (4096, 6144, 12288, 300)):
        assert ok(1, hidden, qkv, inter) and ok(most, hidden, qkv, inter)
        assert not ok(most + 1, hidden, qkv, inter) and not ok(0, hidden, qkv, inter)


def test_large_steps_skip_the_module_checks(pkg, monkeypatch):
    """A step that a fused form is not for pays for no look at its modules."""
    layer = pkg.Qwen3DecoderLayer(pkg.Qwen3Config(
        hidden_size=64, num_attention_heads=2, num_key_value_heads=1, intermediate_size=64,
        num_hidden_layers=1, max_position_embeddings=64))
    layer.self_attn.k_cache = torch.zeros(1)

    def look(*_):
        raise AssertionError("modules looked at")

    monkeypatch.setattr(pkg.qwen3_naive, "_prefill_methods", look)
    monkeypatch.setattr(pkg.qwen3_naive, "_decode_methods", look)
    x = torch.empty(2049, 64)
    assert layer._prefill_native(x, *[None] * 6, x, None) is None
    assert not layer._norms_in_projections(x, None)
