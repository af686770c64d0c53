"""Differentiable operations of the training batch on the gfx950 kernels.

Each is an autograd Function whose forward and backward are HIP kernels, with
the torch formula beside it: the formula serves every call the kernels do not
take (``kernels_ok``), and a backward that has to be differentiable itself
(``create_graph=True``) differentiates the formula.
"""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import kernels as K


def kernels_ok(*tensors: torch.Tensor) -> bool:
    """Whether the training kernels take a call on these tensors: plain bf16
    tensors of one GPU, run eagerly.  Function transforms (vmap, functional
    and forward-mode derivatives), tracing and autocast need torch ops."""
    dev = tensors[0].device
    if dev.type != "cuda":
        return False
    for t in tensors:
        if (type(t) not in (torch.Tensor, torch.nn.Parameter) or t.dtype != torch.bfloat16
                or t.device != dev):
            return False
    return not (torch.compiler.is_compiling() or torch.jit.is_tracing()
                or torch.is_autocast_enabled("cuda") or forward_ad._current_level >= 0
                or torch._C._functorch.peek_interpreter_stack() is not None)


def _formula_grads(formula, inputs, needs, grads):
    """Gradients of ``formula(*inputs)`` that autograd can differentiate again."""
    with torch.enable_grad():
        out = formula(*inputs)
    wanted = [t for t, n in zip(inputs, needs) if n]
    got = iter(torch.autograd.grad(out, wanted, grads, create_graph=True, allow_unused=True))
    return tuple(next(got) if n else None for n in needs)


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


def attention_formula(qkv, norm_q, norm_k, cache, num_heads, num_kv_heads, scale):
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
    o = torch.matmul(w, vf).to(qkv.dtype)
    return o.transpose(1, 2).reshape(batch, seq_len, -1)


def rms_norm_formula(x, weight, eps):
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(dim=-1, keepdim=True) + eps)
            * weight.float()).to(x.dtype)


class QkvAttention(torch.autograd.Function):
    """``attention_formula`` of a packed bf16 qkv: QK-norm + RoPE kernel, then
    the MFMA attention; the backward writes one packed ``d qkv``."""

    @staticmethod
    def forward(ctx, qkv, q_weight, k_weight, cache, num_heads, num_kv_heads, eps, scale):
        batch, seq_len, width = qkv.shape
        x = qkv.reshape(-1, width)
        x = K._dense16(x) if x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16 else x
        qw, kw = K._dense16(q_weight), K._dense16(k_weight)
        q, k = K.qk_norm_rope_seq(x, qw, kw, seq_len, cache, num_heads, num_kv_heads, eps)
        v = x[:, (num_heads + num_kv_heads) * K.HEAD_DIM:].view(-1, num_kv_heads, K.HEAD_DIM)
        need = any(ctx.needs_input_grad[:3])
        out, out32, stats = K.train_attention(q, k, v, batch, scale, need)
        if need:
            ctx.save_for_backward(qkv, q_weight, k_weight, cache, q, k, out32, stats)
            ctx.args = (num_heads, num_kv_heads, eps, scale)
        return out.view(batch, seq_len, num_heads * K.HEAD_DIM)

    @staticmethod
    def backward(ctx, dout):
        qkv, q_weight, k_weight, cache, q, k, out32, stats = ctx.saved_tensors
        num_heads, num_kv_heads, eps, scale = ctx.args
        if torch.is_grad_enabled():  # create_graph: the gradients are differentiated again
            def formula(qkv, q_weight, k_weight):
                return attention_formula(qkv, lambda t: rms_norm_formula(t, q_weight, eps),
                                         lambda t: rms_norm_formula(t, k_weight, eps), cache,
                                         num_heads, num_kv_heads, scale)
            return (*_formula_grads(formula, (qkv, q_weight, k_weight), ctx.needs_input_grad[:3],
                                    dout), None, None, None, None, None)
        batch, seq_len, width = qkv.shape
        x = qkv.reshape(-1, width)
        x = K._dense16(x) if x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16 else x
        qw, kw = K._dense16(q_weight), K._dense16(k_weight)
        first_v = (num_heads + num_kv_heads) * K.HEAD_DIM
        v = x[:, first_v:].view(-1, num_kv_heads, K.HEAD_DIM)
        dqkv = torch.empty((batch * seq_len, width), dtype=torch.bfloat16, device=x.device)
        dq, dk = K.train_attention_backward(
            q, k, v, batch, scale, out32, stats, K._dense16(dout.reshape(-1, dout.shape[-1])),
            dqkv[:, first_v:])
        dqw, dkw = K.qk_norm_rope_backward(dq, dk, x, qw, kw, seq_len, cache, eps, dqkv)
        need = ctx.needs_input_grad
        return (dqkv.view(batch, seq_len, width) if need[0] else None, dqw if need[1] else None,
                dkw if need[2] else None, None, None, None, None, None)


def attention_ok(qkv, q_weight, k_weight, cache, num_heads, num_kv_heads) -> bool:
    """Whether ``QkvAttention`` takes this batch."""
    return (kernels_ok(qkv, q_weight, k_weight) and qkv.dim() == 3 and qkv.numel() > 0
            and num_heads % num_kv_heads == 0 and num_heads <= 4096
            and qkv.shape[2] == (num_heads + 2 * num_kv_heads) * K.HEAD_DIM
            and q_weight.shape == k_weight.shape == (K.HEAD_DIM,)
            and cache.dtype == torch.float32 and cache.is_contiguous()
            and cache.data_ptr() % 16 == 0 and cache.shape[1] == K.HEAD_DIM
            and qkv.shape[1] <= cache.shape[0] and qkv.shape[0] <= 65535)
