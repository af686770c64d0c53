"""Which tensors the one-call prefill layer and the training Functions may read
through their addresses (CPU: no kernel is launched)."""
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
