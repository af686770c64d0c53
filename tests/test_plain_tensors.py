"""Which tensors the one-call prefill layer and the training Functions read
through their addresses (CPU: no kernel is launched)."""
import importlib
import types
import weakref

import pytest
import torch


class Wrapper(torch.Tensor):
    """A wrapper subclass: a shape without storage of its own."""

    @staticmethod
    def __new__(cls, t):
        return torch.Tensor._make_wrapper_subclass(cls, t.shape, dtype=t.dtype, device=t.device)

    def __init__(self, t):
        self.t = t

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise AssertionError(f"{func} needs the wrapper's own rule")


class Plain(torch.Tensor):
    pass


def test_prefill_layer_takes_plain_tensors_only(pkg):
    t = torch.zeros(4, 64, dtype=torch.bfloat16)
    ok = pkg.kernels._plain
    assert ok(t, torch.bfloat16, -1) and ok(torch.nn.Parameter(t), torch.bfloat16, -1)
    assert not ok(t.as_subclass(Plain), torch.bfloat16, -1)
    assert not ok(torch.nn.Parameter(t.as_subclass(Plain)), torch.bfloat16, -1)
    assert not ok(Wrapper(t), torch.bfloat16, -1)


def _backward(T, name):
    """Runs a Function's backward on CPU tensors; its launches are the caller's to replace."""
    b16 = torch.bfloat16
    x, w = torch.zeros(1, 5, 512, dtype=b16), torch.zeros(512, dtype=b16)
    f = torch.zeros(2, 5, 128)
    cls, saved, out, args = {
        "norm": (T._RmsNorm, (x, w, torch.zeros(1, 5, 1)), x.shape, {"eps": 1e-6}),
        "silu": (T.SiluMul, (x,), (1, 5, 256), {}),
        "attention": (T._QkvAttention, (x, w[:256].view(2, 128), torch.zeros(5, 128), torch.zeros(1, 5, 2, 1),
                                       torch.zeros(1, 5, 1, 1), f, f.transpose(1, 2).contiguous(), f,
                                       torch.zeros(2, 5, 5)), (1, 5, 256), {"args": (2, 1, 1e-6, 0.1)}),
    }[name]
    ctx = types.SimpleNamespace(saved_tensors=saved, needs_input_grad=(True,) * 3, **args)
    with torch.no_grad():
        cls.backward(ctx, torch.zeros((), dtype=b16).expand(out))


@pytest.mark.parametrize("name", ["norm", "silu", "attention"])
def test_backward_keeps_its_copies_until_the_launch(pkg, monkeypatch, name):
    """A copy made to be dense is alive when a kernel that gets its address is
    launched (freed earlier, another thread's allocation may write to it)."""
    T = importlib.import_module(pkg.__name__ + ".train_ops")
    copies, passed = {}, []

    def copy(t):
        c = t.contiguous().clone()
        copies[c.data_ptr()] = weakref.ref(c)
        return c

    def call(entry, device, *args):
        for a in args:
            if a in copies:
                assert copies[a]() is not None, f"{entry}: the copy at {a:#x} is gone"
                passed.append(a)

    monkeypatch.setattr(pkg.kernels, "_dense16", copy)
    monkeypatch.setattr(T, "_call", call)
    _backward(T, name)
    assert passed


@pytest.mark.parametrize("name", ["norm", "silu", "attention"])
def test_backward_runs_without_autocast(pkg, monkeypatch, name):
    """Autocast around a backward alone (its forward ran without) must not reach
    the fp32 products whose addresses the kernels get: in 16 bits they are half
    as long."""
    T = importlib.import_module(pkg.__name__ + ".train_ops")
    seen = []
    monkeypatch.setattr(T, "_call", lambda *_: seen.append(torch.is_autocast_enabled("cuda")))
    torch.set_autocast_enabled("cuda", True)
    try:
        _backward(T, name)
        assert torch.is_autocast_enabled("cuda")
    finally:
        torch.set_autocast_enabled("cuda", False)
    assert seen and not any(seen)


def test_launch_on_the_tensors_device(pkg, monkeypatch):
    """A training batch on another GPU than the current one is launched there."""
    T = importlib.import_module(pkg.__name__ + ".train_ops")
    current, launched = [0], []

    class Device:
        def __init__(self, device):
            self.index = device.index

        def __enter__(self):
            current.append(self.index)

        def __exit__(self, *_):
            current.pop()

    entry = types.SimpleNamespace(f=lambda *args: launched.append((current[-1], *args)) or 0)
    monkeypatch.setattr(T, "lib", lambda: entry)
    monkeypatch.setattr(T, "_current_device", lambda: current[-1])
    monkeypatch.setattr(T, "stream_handle", lambda device: 100 + device.index)
    monkeypatch.setattr(torch.cuda, "device", Device)
    T._call("f", torch.device("cuda", 0), 7)
    T._call("f", torch.device("cuda", 1), 8)
    assert launched == [(0, 7, 100), (1, 8, 101)] and current == [0]


def test_replaced_rotation_is_used(pkg, monkeypatch):
    """A program's own RoPE, set on RotaryEmbedding, is the batch forward's."""
    torch.manual_seed(0)
    attn = pkg.Qwen3DecoderLayer(pkg.Qwen3Config(
        hidden_size=64, num_attention_heads=2, num_key_value_heads=1, intermediate_size=64,
        num_hidden_layers=1, max_position_embeddings=64)).self_attn
    x, calls = torch.randn(1, 5, 64), []
    want = attn(x)

    def rotate(t, positions, cache):
        calls.append(1)
        return -t

    monkeypatch.setattr(pkg.qwen3_naive.RotaryEmbedding, "rotate", staticmethod(rotate))
    assert not torch.allclose(attn(x), want) and len(calls) == 2
