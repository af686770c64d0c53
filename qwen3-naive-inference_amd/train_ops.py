"""The training batch's element-wise chains as autograd Functions on fused
HIP kernels (csrc/train_rows.hip).

Each follows the torch formula beside it in both directions: the kernels
repeat its fp32 operations and bf16 roundings, and sums along a norm's row and
the products are the same torch calls on the same operands.  The softmax and
its gradient are own kernels that add in torch's order up to 1,024 columns and
torch calls above.  The values are the formula's, bit for bit, but for sums in
another fixed order: the norm weights' gradients, and from four query heads per
KV head on the sums of k's and v's gradients over those heads.  The formula
serves every call the kernels do not take, and a backward that is
differentiated itself (``create_graph=True``, forward mode) or runs on a batch
of gradients (vmap) goes through the formula.

The formulas work on fp32 copies of their inputs, so a program may write to an
input before the backward, and both parts of a second derivative meet in fp32.
So do the Functions: they save copies that the kernels leave, and each returns,
beside its result, a *link* per input: zeros of the input's shape in fp32, all
one element, which the formula of a differentiated backward adds to the saved
copy.  What flows back to the copy then reaches the same backward, with what
flows to the result, and is rounded once.
"""
from __future__ import annotations

import functools

import torch
from torch.autograd import forward_ad

from . import kernels as K
from ._lib import check, lib, stream_handle

HEAD_DIM = K.HEAD_DIM
F32, BF16 = torch.float32, torch.bfloat16
_current_device = torch._C._cuda_getDevice
_is_legacy_batch = torch._C._functorch.is_legacy_batchedtensor
_is_wrapped = torch._C._functorch.is_functorch_wrapped_tensor


def kernels_ok(*tensors: torch.Tensor) -> bool:
    """Whether the training kernels take a call on these tensors: plain bf16
    tensors of one GPU, run eagerly with a gradient wanted of the first.
    Function transforms (vmap, functional and forward-mode derivatives),
    tracing and autocast need torch ops."""
    dev = tensors[0].device
    if dev.type != "cuda" or not (torch.is_grad_enabled() and tensors[0].requires_grad):
        return False
    for t in tensors:
        if (type(t) not in (torch.Tensor, torch.nn.Parameter) or t.dtype != BF16 or t.device != dev
                or t.is_inference()):  # no version, not saved for a backward
            return False
    return not (torch.compiler.is_compiling() or torch.jit.is_tracing() or _make_fx()
                or torch.is_autocast_enabled("cuda") or any(map(_has_tangent, tensors))
                or torch._C._functorch.peek_interpreter_stack() is not None)


def _make_fx() -> bool:
    """Whether ops are being recorded into a graph that would not hold the kernels."""
    return torch._C._get_dispatch_mode(torch._C._TorchDispatchModeKey.PROXY) is not None


def _has_tangent(t: torch.Tensor) -> bool:
    return forward_ad._current_level >= 0 and forward_ad.unpack_dual(t).tangent is not None


def _formula_backward(grad, links, *saved) -> bool:
    """Whether a backward goes through the formula: it is differentiated itself
    (``create_graph=True``, forward mode over it), has what flowed back to its
    links, or its gradient is a batch (``is_grads_batched``, vmap) or another
    type, which kernels cannot read."""
    if grad is None or torch.is_grad_enabled() or any(d is not None for d in links):
        return True
    for t in (grad, *saved):
        if type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter or _has_tangent(t):
            return True
    return _is_legacy_batch(grad) or _is_wrapped(grad)


def _formula_grads(formula, copies, links, needs, grad, link_grads):
    """bf16 gradients of ``formula`` with respect to the inputs that ``copies``
    and ``links`` stand for, which autograd can differentiate again."""
    with torch.enable_grad():
        inputs = [link + copy.float() for link, copy in zip(links, copies)]
        out = formula(*inputs)
    got = [None] * len(inputs)
    if grad is not None:
        got = torch.autograd.grad(out, inputs, grad, create_graph=torch.is_grad_enabled(),
                                  allow_unused=True)
    sums = [d if g is None else g if d is None else g + d for g, d in zip(got, link_grads)]
    return tuple(g.to(BF16) if n and g is not None else None for g, n in zip(sums, needs))


def _no_autocast(backward):
    """A backward without autocast, as its forward ran: under it the products of
    fp32 tensors, which the kernels read, would come out in 16 bits."""
    @functools.wraps(backward)
    def run(ctx, *grads):
        if not torch.is_autocast_enabled("cuda"):
            return backward(ctx, *grads)
        with torch.autocast("cuda", enabled=False):
            return backward(ctx, *grads)
    return run


def _call(name, device, *args):
    """Launches on the device's current stream, also where another device is current
    (a torch op changes to its tensors' device by itself)."""
    if _current_device() != device.index:
        with torch.cuda.device(device):
            return _call(name, device, *args)
    check(getattr(lib(), name)(*args, stream_handle(device)), name)


# ---------------------------------------------------------------------------
# RMSNorm (qwen3_naive.py:156-162)
# ---------------------------------------------------------------------------
def rms_norm_formula(x, weight, eps, dtype=None):
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + eps)
            * weight.float()).to(dtype or x.dtype)


def _mean_square(x, rows, stride, heads, n, shape, x_copy=None, zero=None):
    """``x.float().pow(2).mean(-1, keepdim=True)`` of ``heads`` adjacent rows of ``n`` per row of
    ``x``; ``x_copy`` and ``zero`` get a copy of the rows and a zero."""
    sq = torch.empty(shape, dtype=F32, device=x.device)
    _call("qmi_square_rows", x.device, x.data_ptr(), rows, stride, heads, n, sq.data_ptr(),
          None if x_copy is None else x_copy.data_ptr(), None if zero is None else zero.data_ptr())
    return sq.mean(dim=-1, keepdim=True)


def _norm_grad(x, rows, stride, heads, n, shape, mean, w, eps, dy, dx):
    """Gradients of the norm: ``dx`` is written (laid out as ``x``), the weight's is returned."""
    prod = torch.empty(shape, dtype=F32, device=w.device)
    _call("qmi_norm_prod", w.device, x.data_ptr(), rows, stride, heads, n, w.data_ptr(),
          dy.data_ptr(), prod.data_ptr())
    dr = prod.sum(dim=-1, keepdim=True)
    parts = torch.empty((lib().qmi_norm_grad_parts(rows, n), n), dtype=F32, device=w.device)
    _call("qmi_norm_grad", w.device, x.data_ptr(), rows, stride, heads, n, mean.data_ptr(),
          w.data_ptr(), eps, dy.data_ptr(), dr.data_ptr(), dx.data_ptr(), parts.data_ptr())
    dw = torch.empty(n, dtype=BF16, device=w.device)
    _call("qmi_sum_rows", w.device, parts.data_ptr(), parts.shape[0], n, dw.data_ptr())
    return dw


def norm_ok(x, weight) -> bool:
    return (kernels_ok(x, weight) and x.numel() > 0 and x.numel() < 1 << 33
            and weight.shape == x.shape[-1:] and x.shape[-1] % 8 == 0 and x.shape[-1] <= 65536
            and x.is_contiguous() and x.data_ptr() % 16 == 0)


class _RmsNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, eps):
        n = x.shape[-1]
        rows = x.numel() // n
        w = K._dense16(weight)
        x_copy, y, w_copy = torch.empty_like(x), torch.empty_like(x), torch.empty_like(w)
        zero = torch.empty(1, dtype=F32, device=x.device)
        mean = _mean_square(x, rows, n, 1, n, x.shape, x_copy, zero)
        _call("qmi_norm_apply", x.device, x.data_ptr(), rows, n, n, mean.data_ptr(), w.data_ptr(),
              eps, y.data_ptr(), w_copy.data_ptr())
        links = zero.expand(x.shape), zero.expand(n)
        ctx.save_for_backward(x_copy, w_copy, mean, *links)
        ctx.set_materialize_grads(False)
        ctx.eps = eps
        return (y, *links)

    @staticmethod
    @_no_autocast
    def backward(ctx, dy, *dlinks):
        x, weight, mean, *links = ctx.saved_tensors
        need = ctx.needs_input_grad
        if _formula_backward(dy, dlinks, x, weight):
            return (*_formula_grads(lambda x, w: rms_norm_formula(x, w, ctx.eps, BF16), (x, weight),
                                    links, need, dy, dlinks), None)
        n = x.shape[-1]
        x, mean = K._dense16(x), K._dense16(mean)  # saved-tensor hooks may have laid them out anew
        dx = torch.empty_like(x)
        dw = _norm_grad(x, x.numel() // n, n, 1, n, x.shape, mean, K._dense16(weight), ctx.eps,
                        K._dense16(dy), dx)
        return dx if need[0] else None, dw if need[1] else None, None


class RmsNorm:
    """``rms_norm_formula`` as an autograd Function."""

    @staticmethod
    def apply(x, weight, eps):
        return _RmsNorm.apply(x, weight, eps)[0]


# ---------------------------------------------------------------------------
# SwiGLU (qwen3_naive.py:695-702)
# ---------------------------------------------------------------------------
def silu_mul_formula(gate_up):
    gate, up = gate_up.chunk(2, dim=-1)
    return torch.nn.functional.silu(gate) * up


def silu_mul_ok(gate_up) -> bool:
    return (kernels_ok(gate_up) and gate_up.numel() > 0 and gate_up.numel() < 1 << 33
            and gate_up.shape[-1] % 16 == 0 and gate_up.shape[-1] <= 65536
            and gate_up.is_contiguous() and gate_up.data_ptr() % 16 == 0)


class SiluMul(torch.autograd.Function):
    """``silu(gate) * up`` of a packed ``[..., 2 * inter]`` projection."""

    @staticmethod
    def forward(ctx, gate_up):
        inter = gate_up.shape[-1] // 2
        y = torch.empty((*gate_up.shape[:-1], inter), dtype=BF16, device=gate_up.device)
        _call("qmi_silu_mul_train", y.device, gate_up.data_ptr(), y.numel() // inter, inter, None,
              y.data_ptr())
        ctx.save_for_backward(gate_up)
        return y

    @staticmethod
    @_no_autocast
    def backward(ctx, dy):
        gate_up, = ctx.saved_tensors
        if _formula_backward(dy, (), gate_up):
            with torch.enable_grad():
                gate_up = gate_up.view_as(gate_up)
                y = silu_mul_formula(gate_up)
            return torch.autograd.grad(y, gate_up, dy, create_graph=torch.is_grad_enabled())[0]
        gate_up, dy = K._dense16(gate_up), K._dense16(dy)
        dgu = torch.empty_like(gate_up)
        inter = gate_up.shape[-1] // 2
        _call("qmi_silu_mul_train", dy.device, gate_up.data_ptr(), dy.numel() // inter, inter,
              dy.data_ptr(), dgu.data_ptr())
        return dgu


# ---------------------------------------------------------------------------
# Attention of a training batch (qwen3_naive.py:553-590)
# ---------------------------------------------------------------------------
def rotate(x: torch.Tensor, positions: torch.Tensor, cache: torch.Tensor) -> torch.Tensor:
    """Differentiable half-split rotation (fp32 math, cast back)."""
    half = x.shape[-1] // 2
    cs = cache[positions]
    while cs.dim() < x.dim():
        cs = cs.unsqueeze(-2)
    c, s = cs[..., :half], cs[..., half:]
    x1, x2 = x[..., :half].float(), x[..., half:].float()
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), dim=-1).to(x.dtype)


def attention_formula(qkv, norm_q, norm_k, cache, num_heads, num_kv_heads, scale, rotate=rotate,
                      dtype=None):
    """QK-norm, RoPE and causal attention of ``qkv [B, T, (Hq + 2 Hkv) * D]`` ->
    ``[B, T, Hq * D]``; ``norm_q`` / ``norm_k`` map ``[B, T, heads, D]``."""
    batch, seq_len, width = qkv.shape
    d = width // (num_heads + 2 * num_kv_heads)
    q, k, v = qkv.split([num_heads * d, num_kv_heads * d, num_kv_heads * d], dim=-1)
    q = norm_q(q.reshape(batch, seq_len, num_heads, d))
    k = norm_k(k.reshape(batch, seq_len, num_kv_heads, d))
    v = v.reshape(batch, seq_len, num_kv_heads, d)
    positions = torch.arange(seq_len, device=qkv.device)[None, :].expand(batch, -1)
    q = rotate(q, positions, cache)
    k = rotate(k, positions, cache)
    rep = num_heads // num_kv_heads
    # Attention core in fp32: batched bf16 products with transposed operands
    # (and their autograd) are avoided on this platform.
    qf = q.transpose(1, 2).float()
    kf = k.transpose(1, 2).float().repeat_interleave(rep, dim=1)
    vf = v.transpose(1, 2).float().repeat_interleave(rep, dim=1)
    scores = torch.matmul(qf, kf.transpose(-2, -1).contiguous()) * scale
    mask = torch.triu(torch.ones(seq_len, seq_len, device=qkv.device, dtype=torch.bool), 1)
    scores = scores.masked_fill(mask, float("-inf"))
    w = torch.softmax(scores, dim=-1)
    o = torch.matmul(w, vf).to(dtype or qkv.dtype)
    return o.transpose(1, 2).reshape(batch, seq_len, -1)


def _score_rows_ok(rows: int, t: int) -> bool:
    """Whether one launch (fewer than 2^32 lanes) covers the score rows: a wave
    of 64 lanes per row, 256 lanes above ``SOFTMAX_MAX`` columns."""
    return rows < 1 << (26 if t <= SOFTMAX_MAX else 24)


def attention_ok(qkv, q_weight, k_weight, cache, num_heads, num_kv_heads) -> bool:
    """Whether ``QkvAttention`` takes this batch."""
    return (kernels_ok(qkv, q_weight, k_weight) and qkv.dim() == 3 and qkv.numel() > 0
            and qkv.is_contiguous() and qkv.data_ptr() % 16 == 0 and num_heads % num_kv_heads == 0
            and qkv.shape[2] == (num_heads + 2 * num_kv_heads) * HEAD_DIM
            and _score_rows_ok(qkv.shape[0] * num_heads * qkv.shape[1], qkv.shape[1])
            and qkv.shape[0] <= 65535
            and q_weight.shape == k_weight.shape == (HEAD_DIM,)
            and cache.dtype == F32 and cache.device == qkv.device and cache.is_contiguous()
            and cache.data_ptr() % 16 == 0 and cache.shape[1] == HEAD_DIM
            and qkv.shape[1] <= cache.shape[0])


# Longest row of the fused causal softmax; torch's own kernel adds longer rows in
# another order.
SOFTMAX_MAX = 1024


class _QkvAttention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qkv, q_weight, k_weight, cache, hq, hkv, eps, scale):
        b, t, width = qkv.shape
        dev, d = qkv.device, HEAD_DIM
        qw, kw = K._dense16(q_weight), K._dense16(k_weight)
        zero = torch.empty(1, dtype=F32, device=dev)
        q_mean = _mean_square(qkv, b * t * hq, width, hq, d, (b, t, hq, d), None, zero)
        k_mean = _mean_square(qkv[..., hq * d:], b * t * hkv, width, hkv, d, (b, t, hkv, d))
        qf = torch.empty((b * hq, t, d), dtype=F32, device=dev)
        kt = torch.empty((b * hq, d, t), dtype=F32, device=dev)
        vf = torch.empty_like(qf)
        w_copy = torch.empty((2, d), dtype=BF16, device=dev)
        cache_copy = torch.empty((t, d), dtype=F32, device=dev)
        _call("qmi_train_qkv", dev, qkv.data_ptr(), width, b, t, hq, hkv, q_mean.data_ptr(),
              k_mean.data_ptr(), qw.data_ptr(), kw.data_ptr(), eps, cache.data_ptr(), qf.data_ptr(),
              kt.data_ptr(), vf.data_ptr(), w_copy.data_ptr(), cache_copy.data_ptr())
        scores = torch.bmm(qf, kt)
        # Kernels write to tensors of their own: a dispatch mode (selective
        # checkpointing) may keep what a torch op returned, and sees no write.
        w = torch.empty_like(scores)
        if t <= SOFTMAX_MAX:
            _call("qmi_causal_softmax", dev, scores.data_ptr(), None, b * hq * t, t, scale, w.data_ptr())
        else:
            _call("qmi_scale_mask", dev, scores.data_ptr(), b * hq * t, t, scale, float("-inf"),
                  w.data_ptr())
            w = torch.softmax(w, dim=-1)
        del scores
        o = torch.bmm(w, vf)
        out = torch.empty((b, t, hq * d), dtype=BF16, device=dev)
        _call("qmi_train_heads", dev, o.data_ptr(), out.data_ptr(), b, t, hq, 1)
        links = zero.expand(qkv.shape), zero.expand(d), zero.expand(d)
        ctx.save_for_backward(qkv, w_copy, cache_copy, q_mean, k_mean, qf, kt, vf, w, *links)
        ctx.set_materialize_grads(False)
        ctx.args = (hq, hkv, eps, scale)
        return (out, *links)

    @staticmethod
    @_no_autocast
    def backward(ctx, dout, *dlinks):
        qkv, weights, cache, q_mean, k_mean, qf, kt, vf, w, *links = ctx.saved_tensors
        hq, hkv, eps, scale = ctx.args
        need = ctx.needs_input_grad
        if _formula_backward(dout, dlinks, qkv, weights):
            def formula(qkv, q_weight, k_weight):
                return attention_formula(qkv, lambda a: rms_norm_formula(a, q_weight, eps, BF16),
                                         lambda a: rms_norm_formula(a, k_weight, eps, BF16), cache,
                                         hq, hkv, scale, dtype=BF16)
            return (*_formula_grads(formula, (qkv.detach(), *weights), links, need, dout, dlinks),
                    None, None, None, None, None)
        qkv, cache, q_mean, k_mean, w, dout = map(K._dense16, (qkv, cache, q_mean, k_mean, w, dout))
        b, t, width = qkv.shape
        dev, d = qkv.device, HEAD_DIM
        qw, kw = K._dense16(weights)
        do = torch.empty((b * hq, t, d), dtype=F32, device=dev)
        _call("qmi_train_heads", dev, do.data_ptr(), dout.data_ptr(), b, t, hq, 0)
        dw = torch.bmm(do, vf.transpose(1, 2))
        dv = torch.bmm(w.transpose(1, 2), do)
        ds = torch.empty_like(dw)
        if t <= SOFTMAX_MAX:
            _call("qmi_causal_softmax", dev, dw.data_ptr(), w.data_ptr(), b * hq * t, t, scale,
                  ds.data_ptr())
        else:
            dw = torch.ops.aten._softmax_backward_data(dw, w, -1, F32)
            _call("qmi_scale_mask", dev, dw.data_ptr(), b * hq * t, t, scale, 0.0, ds.data_ptr())
        del dw
        dq = torch.bmm(ds, kt.transpose(1, 2))
        dkt = torch.bmm(qf.transpose(1, 2), ds)
        del ds
        dqkv = torch.empty_like(qkv)
        dn_q = torch.empty((b, t, hq, d), dtype=BF16, device=dev)
        dn_k = torch.empty((b, t, hkv, d), dtype=BF16, device=dev)
        _call("qmi_train_qkv_grad", dev, b, t, hq, hkv, dq.data_ptr(), dkt.data_ptr(), dv.data_ptr(),
              cache.data_ptr(), dn_q.data_ptr(), dn_k.data_ptr(), dqkv.data_ptr())
        dqw = _norm_grad(qkv, b * t * hq, width, hq, d, dn_q.shape, q_mean, qw, eps, dn_q, dqkv)
        dkw = _norm_grad(qkv[..., hq * d:], b * t * hkv, width, hkv, d, dn_k.shape, k_mean, kw, eps,
                         dn_k, dqkv[..., hq * d:])
        return (dqkv if need[0] else None, dqw if need[1] else None, dkw if need[2] else None, None,
                None, None, None, None)


class QkvAttention:
    """``attention_formula`` with RMS norms of a packed bf16 qkv as an autograd
    Function; the backward writes one packed ``d qkv``.  ``qkv`` itself is saved:
    the program does not write to it."""

    @staticmethod
    def apply(qkv, q_weight, k_weight, cache, num_heads, num_kv_heads, eps, scale):
        return _QkvAttention.apply(qkv, q_weight, k_weight, cache, num_heads, num_kv_heads, eps,
                                   scale)[0]
