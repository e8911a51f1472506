"""A differential-attention layer built on the fused kernel.

The reference stops at the functional operator (src/layers.py:10-26); its kernel header points to
the Differential Transformer paper (src/kernel.py:1) for the layer around it.  This module is that
layer: input projections, the re-parametrised lambda, the fused operator with its per-head RMSNorm
and (1 - lambda_init) scale, a learnable per-feature gain on the normalised heads, and the output
projection.  Attention is bidirectional unless `causal=True`; `attention_dropout` drops entries of
the two softmax maps while the module is in training mode.

  x [B, N, E]  ->  q, k [B, 2H, N, d],  v [B, H, N, 2d]      (E = 2 * H * d)
  lambda = exp(lq1 . lk1) - exp(lq2 . lk2) + lambda_init       (one scalar per layer, or one per
                                                                head with per_head_lambda=True)
  heads  = gain * MultiheadDiffAttnKernel(q1, q2, k1, k2, v, lambda, lambda_init, rms_norm=True)
  y      = out_proj(concat heads)
"""
import math

import torch
from torch import nn
from torch.autograd import forward_ad

import _native
from kernel import _DTYPES, _SUPPORTED_D, _current_stream
from layers import MultiheadDiffAttnKernel


def lambda_init_for_depth(depth: int) -> float:
    """The paper's schedule for the initial lambda of layer `depth` (0-based)."""
    return 0.8 - 0.6 * math.exp(-0.3 * depth)


class _recalled_linear(torch.autograd.Function):
    """F.linear(x, w) with its value at hand: what autograd needs of it is the graph."""

    @staticmethod
    def forward(ctx, value, x, w):
        ctx.save_for_backward(x if ctx.needs_input_grad[2] else None, w if ctx.needs_input_grad[1] else None)
        return value.view_as(value)

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        return None, None if w is None else g @ w, None if x is None else g.flatten(0, 1).t() @ x.flatten(0, 1)


class _recalled_gain(torch.autograd.Function):
    """heads * gain with its value at hand, of heads [tokens, E] that need no gradient"""

    @staticmethod
    def forward(ctx, value, heads, gain):
        ctx.save_for_backward(heads)
        ctx.width = gain.numel()
        return value.view_as(value)

    @staticmethod
    def backward(ctx, g):
        return None, None, (g * ctx.saved_tensors[0]).view(-1, ctx.width).sum(0)


class _diff_attn_layer(torch.autograd.Function):
    """The whole layer as one node: csrc/layer_host.cpp runs it.  (As single operations, B8 H8 N1024 d64 causal fp16: 39
    launches and 709 us of device time a step, of which the operator and four projections of 90 us in all are forward
    work.)  A backward that is itself differentiated goes through the single operations, so that what they can differentiate
    twice still can: the gradients of the output projection and of the gain.  Behind these is the operator, whose gradients
    are plain kernel outputs; their derivative raises."""

    @staticmethod
    def forward(ctx, x, wq, wk, wv, wo, gain, lq1, lk1, lq2, lk2, heads, causal, lambda_init):
        inputs = (x, wq, wk, wv, wo, gain, lq1, lk1, lq2, lk2)
        options = (heads, causal, lambda_init)
        need = ctx.needs_input_grad
        projections, lambdas = need[1] or need[2] or need[3], need[6] or need[7] or need[8] or need[9]
        operator = need[0] or projections or lambdas        # its gradients are wanted
        inner = operator or need[5]                         # a gradient behind the output projection is
        y, *saved = _native.layer().layer_forward(*inputs, *options, inner, need[4], _current_stream(x.device))
        if inner or need[4]:
            ctx.options = (*x.shape[:2], *options)
            # An input is saved where the single operations would save it: what no wanted gradient reads may be written in
            # place before the backward, and is not held until then.  The gain beside its own gradient alone is such a one,
            # but the kernel that forms that gradient reads it: its values, without the version that autograd would check.
            none = (None,) * 4
            ctx.save_for_backward(x if projections else None, *((wq, wk, wv) if need[0] else none[:3]),
                                  *((wo, gain if operator else gain.data) if inner else none[:2]),
                                  *((lq1, lk1, lq2, lk2) if lambdas else none), *saved)
        return y

    @staticmethod
    def backward(ctx, dy):
        saved = ctx.saved_tensors
        dev = dy.device
        wanted = _native.layer().wanted(ctx)
        if torch.is_grad_enabled():         # create_graph
            return (*_differentiable_gradients(ctx, saved, dy, wanted), None, None, None)

        def launch():
            return _native.layer().layer_backward(*saved, dy, *ctx.options, wanted, _current_stream(dev))

        if dev.index != torch._C._cuda_getDevice():
            with torch.cuda.device(dev):
                grads = launch()
        else:
            grads = launch()
        return (*grads, None, None, None)


def _differentiable_gradients(ctx, saved, dy, wanted):
    """The gradients of _diff_attn_layer as functions of dy and of its inputs."""
    B, N, heads, causal, lambda_init = ctx.options
    E, need = dy.size(-1), ctx.needs_input_grad
    *inputs, qkv, hd, hg, _, _, lam = saved
    operator = any(need[:4]) or any(need[6:])           # else the heads are constants

    def at(i, *sizes):
        """Input i.  What was not saved is not read, and its place in the graph is what counts.  An alias, at which the
        gradients are taken: hooks on the inputs run where the node's gradients arrive, and not here too."""
        t = inputs[i]
        if sizes and (t is None or i == 5 and not operator):
            t = _native.layer().input_edge(ctx, i, dy, *sizes)
        inputs[i] = None if t is None else t.view_as(t)
        return inputs[i]

    with torch.autocast("cuda", enabled=False):
        wo, gain = at(4, E, E), at(5, E // heads)
        if operator:
            x, *weights = at(0, B, N, E), at(1, E, E), at(2, E, E), at(3, E, E)
            q, k, v = (_recalled_linear.apply(value, x, w) for value, w in zip(qkv.view(B, N, 3, E).unbind(2), weights))
            q1, q2 = q.view(B, N, heads, 2, -1).transpose(1, 2).unbind(3)
            k1, k2 = k.view(B, N, heads, 2, -1).transpose(1, 2).unbind(3)
            vectors = [at(i) for i in range(6, 10)]
            if vectors[0] is not None:
                lam = _lambda(*vectors, lambda_init)
            y = MultiheadDiffAttnKernel(q1, q2, k1, k2, v.view(B, N, heads, -1).transpose(1, 2), lambda_scale=lam,
                                        lambda_init=lambda_init, rms_norm=True, causal=causal)
            y = (y * gain).transpose(1, 2)
        else:
            y = _recalled_gain.apply(hd if hg is None else hg, hd, gain) if need[5] else hg
        y = nn.functional.linear(y.reshape(B, N, E), wo)
        ids = [i for i in range(10) if wanted >> i & 1]
        grads = [None] * 10
        for i, g in zip(ids, torch.autograd.grad(y, [inputs[i] for i in ids], dy, create_graph=True)):
            grads[i] = g
    return grads


def _lambda(q1, k1, q2, k2, lambda_init):
    """[1], or [num_heads] from vectors per head"""
    return (torch.exp((q1 * k1).sum(-1)) - torch.exp((q2 * k2).sum(-1)) + lambda_init).reshape(-1)


def _plain(t):
    return type(t) is torch.Tensor or type(t) is nn.Parameter


_LINEAR_SOURCE = nn.modules.linear.__file__


def _linear_is_its_own():
    """Whether nn.Linear and F.linear are torch's: profilers and quantizers replace them for every module at once."""
    return (getattr(getattr(nn.Linear.forward, "__code__", None), "co_filename", None) == _LINEAR_SOURCE
            and nn.Linear.__call__ is nn.Module._wrapped_call_impl and nn.functional.linear is torch._C._nn.linear)


def _plain_linear(m):
    """Whether calling m is F.linear with its weight and nothing else: no bias, hooks, wrapper or override."""
    return (type(m) is nn.Linear and m.bias is None and "forward" not in m.__dict__ and m._compiled_call_impl is None
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks))


class DiffAttn(nn.Module):
    def __init__(self, embed_dim: int, num_heads: int, depth: int = 0, attention=MultiheadDiffAttnKernel,
                 causal: bool = False, per_head_lambda: bool = False, attention_dropout: float = 0.0,
                 device=None, dtype=torch.float16):
        super().__init__()
        if embed_dim % (2 * num_heads) != 0:
            raise ValueError("embed_dim must be divisible by 2 * num_heads")
        self.embed_dim = embed_dim
        self.num_heads = num_heads
        self.head_dim = embed_dim // (2 * num_heads)      # d: q/k sub-head width; a value head is 2d wide
        self.lambda_init = lambda_init_for_depth(depth)
        self.attention = attention
        self.causal = causal
        self.attention_dropout = float(attention_dropout)     # on both softmax maps, in training mode only
        kw = dict(device=device, dtype=dtype)
        self.q_proj = nn.Linear(embed_dim, embed_dim, bias=False, **kw)
        self.k_proj = nn.Linear(embed_dim, embed_dim, bias=False, **kw)
        self.v_proj = nn.Linear(embed_dim, embed_dim, bias=False, **kw)
        self.out_proj = nn.Linear(embed_dim, embed_dim, bias=False, **kw)
        # the four lambda vectors live in fp32: their products go through exp()
        lam = dict(device=device, dtype=torch.float32)
        shape = (num_heads, self.head_dim) if per_head_lambda else (self.head_dim,)
        self.lambda_q1 = nn.Parameter(torch.empty(shape, **lam).normal_(0.0, 0.1))
        self.lambda_k1 = nn.Parameter(torch.empty(shape, **lam).normal_(0.0, 0.1))
        self.lambda_q2 = nn.Parameter(torch.empty(shape, **lam).normal_(0.0, 0.1))
        self.lambda_k2 = nn.Parameter(torch.empty(shape, **lam).normal_(0.0, 0.1))
        self.head_gain = nn.Parameter(torch.ones(2 * self.head_dim, **kw))

    def lambda_scale(self) -> torch.Tensor:
        return _lambda(self.lambda_q1, self.lambda_k1, self.lambda_q2, self.lambda_k2, self.lambda_init)

    def _streams(self, p: torch.Tensor):
        """[B, N, H, 2, d] -> two [B, H, N, d] views: sub-heads 2h and 2h+1 of the q/k projections are the two softmax
        streams of head h.

        With unbind the backward writes the two gradients side by side in one pass; selecting each stream makes it two
        fills, two copies, a sum and a copy into the projection's layout (B8 H8 N1024 d64: some 55 us each for q and k).
        Views from unbind may not be written in place, which an `attention` of the caller's own is free to do."""
        if self.attention is MultiheadDiffAttnKernel:
            p1, p2 = p.unbind(3)
        else:
            p1, p2 = p.select(3, 0), p.select(3, 1)
        return p1.transpose(1, 2), p2.transpose(1, 2)

    def _fused_inputs(self, x):
        """The layer's tensors when one node may stand for all of its operations, else None.  Whatever could see or change a
        single operation goes through them one by one: a replaced or hooked projection, another `attention`, tensor
        subclasses, autocast, transforms, tracers, compilers and modes, and what the kernels do not read in place."""
        if not (_plain(x) and x.is_cuda and x.dtype in _DTYPES and x.dim() == 3 and x.numel() > 0 and self.head_dim in _SUPPORTED_D
                and self.attention is MultiheadDiffAttnKernel and not (self.training and self.attention_dropout)):
            return None
        if (torch.compiler.is_compiling() or torch._C._are_functorch_transforms_active() or torch._C._get_tracing_state() is not None
                or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack() or forward_ad._current_level >= 0
                or torch.is_autocast_enabled("cuda") or nn.modules.module._has_any_global_hook()):
            return None
        cls = type(self)
        if (cls.lambda_scale is not DiffAttn.lambda_scale or cls._streams is not DiffAttn._streams
                or "lambda_scale" in self.__dict__ or "_streams" in self.__dict__):
            return None
        projections = (self.q_proj, self.k_proj, self.v_proj, self.out_proj)
        if not (_linear_is_its_own() and all(_plain_linear(m) for m in projections)):
            return None
        E, H, d, dev = self.embed_dim, self.num_heads, self.head_dim, x.device
        if x.size(2) != E or dev.index != torch._C._cuda_getDevice() or x.size(0) * H * (x.size(1) + 127) > 1 << 28:
            return None
        lambdas = (self.lambda_q1, self.lambda_k1, self.lambda_q2, self.lambda_k2)
        shape = lambdas[0].shape
        if shape not in ((d,), (H, d)):
            return None
        inputs = (*(m.weight for m in projections), self.head_gain, *lambdas)
        shapes = ((E, E),) * 4 + ((2 * d,),) + (shape,) * 4
        dtypes = (x.dtype,) * 5 + (torch.float32,) * 4
        for t, s, dt in zip(inputs, shapes, dtypes):
            if not (_plain(t) and t.shape == s and t.dtype == dt and t.device == dev and t.is_contiguous() and t.data_ptr() % 16 == 0
                    and not t.is_neg()):
                return None
        return (x, *inputs)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        fused = self._fused_inputs(x)
        if fused is not None:
            options = (self.num_heads, self.causal, self.lambda_init)
            if torch.is_grad_enabled():
                return _diff_attn_layer.apply(*fused, *options)
            return _native.layer().layer_forward(*fused, *options, False, False, _current_stream(x.device))[0]
        B, N, E = x.shape
        H, d = self.num_heads, self.head_dim
        q1, q2 = self._streams(self.q_proj(x).view(B, N, H, 2, d))
        k1, k2 = self._streams(self.k_proj(x).view(B, N, H, 2, d))
        v = self.v_proj(x).view(B, N, H, 2 * d).transpose(1, 2)
        # lambda stays in fp32: the operator then reads it unrounded and returns its gradient in fp32, which a
        # gradient scaler's loss scale cannot push out of range
        lam = self.lambda_scale()
        # views of the projection outputs: the operator reads them through their strides and returns the
        # heads in v's [B,N,H,2d] memory layout, so neither side of it copies
        heads = self.attention(q1, q2, k1, k2, v, lambda_scale=lam, lambda_init=self.lambda_init, rms_norm=True,
                               **({"causal": True} if self.causal else {}),
                               **({"dropout_p": self.attention_dropout} if self.training and self.attention_dropout else {}))
        heads = heads * self.head_gain
        return self.out_proj(heads.transpose(1, 2).reshape(B, N, E))
