"""Llama-style decoder layer whose seven linears run on the INT8 path (forward and backward):
the training step either side of the hot path, as BASELINE config 5 describes it (hidden 4096,
32 heads, MLP 14336, bf16 elsewhere).  RMSNorm, rotary embedding, causal attention (torch
SDPA) and SwiGLU stay in bf16; ``int8=False`` builds the bf16 twin used for loss/grad parity.

In the int8 layer the RMSNorms, the rotary embedding and the SwiGLU product run as one kernel each per direction
(csrc/decoder.hip), and the attention's backward as two (csrc/attention.hip); the twin, tensors those kernels do not take and calls under a tracer or a function transform go through the
torch expressions, which are also what a backward that is differentiated again is made of.
"""
import math

import torch
import torch.nn.functional as F

from . import ops
from .linear import Int8Linear, LinearGroupFunction, _one_group

__all__ = ["DecoderLayer", "rope_tables"]


def rope_tables(seq_len, head_dim, device, base=10000.0):
    # (device None: the default one of torch, left to it; the kernel counts in 32 bits)
    on = torch.device("cpu" if device is None else device)
    if (on.type == "cuda" and on.index in (None, torch._C._cuda_getDevice()) and type(base) is float and type(seq_len) is int and 0 < seq_len < 1 << 30
            and type(head_dim) is int and 0 < head_dim < 1 << 24 and _untraced()):
        return ops.rope_tables(seq_len, head_dim, on, base)
    return _rope_tables(seq_len, head_dim, device, base)


def _rope_tables(seq_len, head_dim, device, base=10000.0):
    inv = 1.0 / (base ** (torch.arange(0, head_dim, 2, device=device, dtype=torch.float32) / head_dim))
    ang = torch.outer(torch.arange(seq_len, device=device, dtype=torch.float32), inv)
    return ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)


def _rope(x, cos, sin):
    # x: [B, H, S, D]; rotate pairs (even, odd halves convention)
    d = x.shape[-1] // 2
    x1, x2 = x[..., :d], x[..., d:]
    c, s = cos[None, None], sin[None, None]
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), dim=-1)


def _rope_pair(q, k, cos, sin):
    """Both rotated, [B, S, H, D] in and out."""
    return tuple(_rope(t.transpose(1, 2), cos, sin).transpose(1, 2) for t in (q, k))


def _rmsnorm(x, weight, eps):
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)).to(x.dtype) * weight


def _swiglu(gate, up):
    return F.silu(gate) * up


def _untraced():
    """Whether this runs outside tracing and function transforms (to which a kernel launch is invisible)."""
    return not (torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0 or torch.utils._python_dispatch._get_current_dispatch_mode() is not None)


def _plain(*tensors):
    """Whether these are plain bf16 tensors on the current device, and nothing traces what is done with them."""
    return _untraced() and all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda and t.dtype == torch.bfloat16 and t.numel() > 0
               and t.device.index == torch._C._cuda_getDevice() for t in tensors)


def _kernels_take(*tensors):
    """Whether tensors can go to the elementwise kernels: plain ones that are dense and aligned."""
    return _plain(*tensors) and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in tensors)


def _rows16(t):
    """Whether the attention kernels read a [batch, heads, seq, head_dim] tensor in place: rows of bf16 at 16-byte steps, at 32-bit
    offsets from the first of a (batch, head)."""
    sb, sh, ss = ops.attention_strides(t)
    return t.stride(3) == 1 and not (sb | sh | ss) & 7 and t.data_ptr() % 16 == 0 and t.shape[3] <= ss <= 0x3fffffff // (t.shape[2] + 512)


FLASH_ATTENTION = int(torch.nn.attention.SDPBackend.FLASH_ATTENTION)


def _attention_kernels_take(q, k, v, scale):
    """Whether the backward of an attention goes to csrc/attention.hip: where torch would take its flash kernels (whose forward is kept),
    on shapes and layouts that ours take."""
    if not (torch.is_grad_enabled() and (q.requires_grad or k.requires_grad or v.requires_grad)) or torch.is_autocast_enabled("cuda"):
        return False
    return (_plain(q, k, v) and ops.attention_backward_takes(*q.shape) and all(t.shape == q.shape and _rows16(t) for t in (q, k, v))
            and torch._fused_sdp_choice(q, k, v, None, 0.0, True, scale=scale) == FLASH_ATTENTION)


def _dense(t, like, dtype=torch.bfloat16):
    """A gradient or a saved tensor as the kernels read it, on the device of `like`.  A saved tensor comes back from a hook
    (torch.autograd.graph.saved_tensors_hooks) in whatever layout, type and place that one gives it."""
    if t.get_device() != like.get_device():
        raise RuntimeError(f"expected tensors on {like.device}, got one on {t.device}")
    if t.dtype != dtype or not t.is_contiguous():
        t = t.to(dtype).contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _differentiable(expression, inputs, grads):
    """Gradients as a graph of torch operators, for a backward that will be differentiated again."""
    with torch.enable_grad():
        out = expression(*inputs)
        wanted = [t for t in inputs if t.requires_grad]
        found = iter(torch.autograd.grad(out, wanted, grads, create_graph=True))
        return tuple(next(found) if t.requires_grad else None for t in inputs)


class _RMSNormFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, eps):
        y, rstd = ops.rmsnorm(x, weight, eps)
        ctx.save_for_backward(x, weight, rstd)
        ctx.eps = eps
        return y

    @staticmethod
    def backward(ctx, dy):
        x, weight, rstd = ctx.saved_tensors
        if torch.is_grad_enabled():
            return (*_differentiable(lambda a, w: _rmsnorm(a, w, ctx.eps), (x, weight), dy), None)
        return (*ops.rmsnorm_backward(_dense(dy, dy), _dense(x, dy), _dense(weight, dy), _dense(rstd, dy, torch.float32)), None)


class _RopeFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, cos, sin):
        ctx.save_for_backward(cos, sin)
        return ops.rope(q, k, cos, sin)

    @staticmethod
    def backward(ctx, dq, dk):
        cos, sin = ctx.saved_tensors
        if torch.is_grad_enabled():
            return (*_rope_pair(dq, dk, cos, -sin), None, None)     # linear in q and k: the transposed rotation
        return (*ops.rope(*(_dense(t, dq) for t in (dq, dk, cos, sin)), backward=True), None, None)


class _SwiGLUFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gate, up):
        ctx.save_for_backward(gate, up)
        return ops.swiglu(gate, up)

    @staticmethod
    def backward(ctx, d):
        gate, up = ctx.saved_tensors
        if torch.is_grad_enabled():
            return _differentiable(_swiglu, (gate, up), d)
        return ops.swiglu_backward(*(_dense(t, d) for t in (d, gate, up)))


class _AttentionFunction(torch.autograd.Function):
    """Causal attention: torch's flash forward, and a backward with its roundings (probabilities and score gradients to bf16) in
    csrc/attention.hip.  The forward stays torch's: the int8 codes behind it spread every bit in which another one would differ."""

    @staticmethod
    def forward(ctx, q, k, v, scale):
        o, lse = torch.ops.aten._scaled_dot_product_flash_attention(q, k, v, 0.0, True, False, scale=scale)[:2]
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.scale = scale
        return o

    @staticmethod
    def backward(ctx, d_o):
        q, k, v, o, lse = ctx.saved_tensors
        if torch.is_grad_enabled():
            return (*_differentiable(lambda *t: F.scaled_dot_product_attention(*t, is_causal=True, scale=ctx.scale), (q, k, v), d_o), None)
        q, k, v, o, d_o = (t if t.dtype == torch.bfloat16 and t.device == d_o.device and _rows16(t) else _dense(t, d_o) for t in (q, k, v, o, d_o))
        return (*ops.attention_backward(d_o, q, k, v, o, _dense(lse, d_o, torch.float32), ctx.scale), None)


def _attention(q, k, v, scale):
    if _attention_kernels_take(q, k, v, scale):
        return _AttentionFunction.apply(q, k, v, scale)
    return F.scaled_dot_product_attention(q, k, v, is_causal=True, scale=scale)


def _projections(x, *layers):
    """The layers' outputs for the same x."""
    if _one_group(x, layers) and _kernels_take(x, *(m.weight for m in layers)):
        return LinearGroupFunction.apply(x, *(m.weight for m in layers))
    return tuple(m(x) for m in layers)


class RMSNorm(torch.nn.Module):
    def __init__(self, dim, eps=1e-5, device=None, fused=False):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(dim, device=device, dtype=torch.bfloat16))
        self.eps = eps
        self.fused = fused

    def forward(self, x):
        # rows that the kernels add up in the order of torch's sum over the last dim, so that results and gradients have the bits of the
        # expression (fewer than 8 rows, or longer ones, torch splits over more threads)
        dim = self.weight.numel()
        if self.fused and dim <= 4096 and dim % 256 == 0 and x.shape[-1] == dim and x.numel() >= 8 * dim and _kernels_take(x, self.weight):
            return _RMSNormFunction.apply(x, self.weight, self.eps)
        return _rmsnorm(x, self.weight, self.eps)


class DecoderLayer(torch.nn.Module):
    def __init__(self, hidden=4096, heads=32, mlp=14336, int8=True, scheme="block_channel", device=None):
        super().__init__()
        assert hidden % heads == 0
        self.hidden, self.heads, self.head_dim = hidden, heads, hidden // heads

        def lin(i, o):
            if int8:
                return Int8Linear(i, o, bias=False, scheme=scheme, device=device)
            m = torch.nn.Linear(i, o, bias=False, device=device, dtype=torch.bfloat16)
            torch.nn.init.normal_(m.weight, std=0.02)
            return m

        self.q_proj, self.k_proj, self.v_proj, self.o_proj = lin(hidden, hidden), lin(hidden, hidden), lin(hidden, hidden), lin(hidden, hidden)
        self.gate_proj, self.up_proj, self.down_proj = lin(hidden, mlp), lin(hidden, mlp), lin(mlp, hidden)
        self.int8 = int8
        self.input_norm, self.post_norm = RMSNorm(hidden, device=device, fused=int8), RMSNorm(hidden, device=device, fused=int8)

    def copy_weights_from(self, other):
        """Share initial values with another layer (int8 layer <-> bf16 twin)."""
        with torch.no_grad():
            for (_, p), (_, q) in zip(sorted(self.named_parameters()), sorted(other.named_parameters())):
                p.copy_(q)

    def forward(self, x):
        B, S, H = x.shape
        cos, sin = rope_tables(S, self.head_dim, x.device)
        h = self.input_norm(x)
        q, k, v = (t.view(B, S, self.heads, self.head_dim) for t in _projections(h, self.q_proj, self.k_proj, self.v_proj))
        rotate = _RopeFunction.apply if self.int8 and self.head_dim % 16 == 0 and _kernels_take(q, k, cos, sin) else _rope_pair
        q, k = rotate(q, k, cos, sin)
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
        scale = 1.0 / math.sqrt(self.head_dim)
        a = _attention(q, k, v, scale) if self.int8 else F.scaled_dot_product_attention(q, k, v, is_causal=True, scale=scale)
        x = x + self.o_proj(a.transpose(1, 2).reshape(B, S, H))
        h = self.post_norm(x)
        gate, up = _projections(h, self.gate_proj, self.up_proj)
        product = _SwiGLUFunction.apply if self.int8 and _kernels_take(gate, up) else _swiglu
        return x + self.down_proj(product(gate, up))
