"""Autograd wiring of the MI355X differential-attention kernels.

Host-side counterpart of the reference's `_diff_attention` (src/kernel.py:461-575): same class
name, same `apply` argument order, same 9-slot gradient tuple (the optional arguments `causal`,
`dropout_p` and `dropout_seed` -- masking and dropout are features the reference lists as missing,
src/kernel.py:4 -- add a slot each).  The work itself is done by the
hand-written HIP kernels in libdiffattn.so, called by the extension module diffattn_host (csrc/host.cpp), which
also allocates the outputs; if either is missing the call raises -- there is no other path.
"""
import torch
from torch.autograd import forward_ad
from torch.autograd.function import once_differentiable
from torch.overrides import has_torch_function_unary

import _native

_SUPPORTED_D = (32, 64, 128)
_FLAG_RMS_NORM = 1      # DIFFATTN_RMS_NORM
_FLAG_CAUSAL = 2        # DIFFATTN_CAUSAL
_DTYPES = (torch.float16, torch.bfloat16)


def _check_inputs(Q1, Q2, K1, K2, V):
    names = ("q1", "q2", "k1", "k2", "v")
    for n, t in zip(names, (Q1, Q2, K1, K2, V)):
        if not torch.is_tensor(t):
            raise TypeError("%s must be a tensor" % n)
        if t.dtype not in _DTYPES:
            raise TypeError("%s must be float16 (like the reference, src/kernel.py:3-4) or bfloat16 (got %s)"
                            % (n, t.dtype))
        if t.dtype != Q1.dtype:
            raise TypeError("all inputs must have the same dtype (%s has %s, q1 has %s)" % (n, t.dtype, Q1.dtype))
        if t.dim() != 4:
            raise ValueError("%s must be [B,H,N,D] (got %d dims)" % (n, t.dim()))
    for n, t in zip(names, (Q1, Q2, K1, K2, V)):
        if not t.is_cuda:
            raise ValueError("%s must live on the GPU" % n)
        if t.device != Q1.device:
            raise ValueError("all inputs must be on the same device")
    B, H, N, D = Q1.shape
    for n, t in zip(names[1:4], (Q2, K1, K2)):
        if tuple(t.shape) != (B, H, N, D):
            raise ValueError("%s has shape %s, expected %s" % (n, tuple(t.shape), (B, H, N, D)))
    if tuple(V.shape) != (B, H, N, 2 * D):
        raise ValueError("v has shape %s, expected %s" % (tuple(V.shape), (B, H, N, 2 * D)))
    if D not in _SUPPORTED_D:
        raise ValueError("head dim %d unsupported; supported: %s" % (D, _SUPPORTED_D))
    if N < 1:
        raise ValueError("empty sequence")
    return B, H, N, D


def _in_place(t):
    """t itself when the kernels can read it through its strides, else a dense copy."""
    return t if _native.host().readable(t) else t.contiguous()


def _current_stream(dev):
    """Raw handle of torch's current stream on dev (no Stream object is built)."""
    return torch._C._cuda_getCurrentRawStream(dev.index if dev.index is not None else torch._C._cuda_getDevice())


def _lambda_tensor(lambda_scale, device, dtype=torch.float16, num_heads=1):
    """The kernels read lambda from device memory (src/kernel.py:138).  A python number is wrapped, in the
    dtype of the tensors (a superset of the reference, whose float default cannot reach its kernel).
    A tensor holds one value, like the reference's, or one per head (`num_heads` values, more than one);
    an fp32 tensor is read as fp32 and gets an fp32 gradient, anything else goes through the tensors' dtype
    like the reference's `dtype=V.dtype` (src/kernel.py:573)."""
    if torch.is_tensor(lambda_scale):
        if lambda_scale.numel() not in (1, num_heads):
            raise ValueError("lambda_scale must have exactly one element, or one per head (%d)" % num_heads)
        if lambda_scale.dtype == torch.float32:
            dtype = torch.float32
        return lambda_scale.detach().to(device=device, dtype=dtype).reshape(-1).contiguous()
    return torch.tensor([float(lambda_scale)], dtype=dtype, device=device)


def _dropout(p, seed):
    """The two dropout arguments as the extension module takes them.  Without dropout there is no seed to look at."""
    p = float(p)
    return p, int(seed) & 0xFFFFFFFFFFFFFFFF if p > 0 else 0


def _typed_like(V, out):
    """A forward's outputs with y of the type that torch.empty_like(V) has: for a tensor subclass, what its
    __torch_function__ makes of it."""
    if type(V) is not torch.Tensor and has_torch_function_unary(V):
        return (out[0].as_subclass(type(torch.empty_like(V[:0]))), *out[1:])
    return out


def _run_forward(Q1, Q2, K1, K2, V, SM_SCALE, LAMBDA_SCALE, LAMBDA_INIT, rms_norm, causal, dropout_p, dropout_seed,
                 differentiable):
    """One forward launch on the current stream.  Returns (inputs as the kernels read them: q1, q2, k1, k2, v, lambda),
    (y, u2, lse1, lse2, rinv, flags, padded length).

    The kernels work on blocks of 128 rows (like the reference's, src/kernel.py:527).  For other lengths they run on
    the next multiple of 128, redirect reads past the last real row to that row and ignore the padding keys: no tensor
    is padded or copied here; only what the library keeps for itself (u2, the row statistics, the backward's workspace)
    is sized for the padded length.  Tensors are read through their strides (the reference passes Q1's and V's to its
    kernel, src/kernel.py:487-494): a [B,N,H,d] projection output viewed as [B,H,N,d] is not copied.  The four q/k
    tensors share one set of strides, as in the reference.  What only a backward reads (src/kernel.py:505 saves its
    counterparts unconditionally) is neither allocated nor written unless `differentiable`."""
    SM_SCALE, LAMBDA_INIT = float(SM_SCALE), float(LAMBDA_INIT)
    dropout_p, dropout_seed = _dropout(dropout_p, dropout_seed)
    flags = (_FLAG_RMS_NORM if rms_norm else 0) | (_FLAG_CAUSAL if causal else 0)
    forward = _native.host().forward
    p_ok = 0.0 <= dropout_p <= 255 / 256
    if p_ok and torch.is_tensor(Q1) and Q1.is_cuda:
        dev = torch._C._cuda_getDevice()
        out = forward(Q1, Q2, K1, K2, V, LAMBDA_SCALE, SM_SCALE, LAMBDA_INIT, flags, dropout_p, dropout_seed, differentiable,
                      dev, torch._C._cuda_getCurrentRawStream(dev), False)
        if out is not None:
            return (Q1, Q2, K1, K2, V, LAMBDA_SCALE), _typed_like(V, out)
    # something about the inputs stands in the way: an error, a layout, another device, a lambda to be converted
    B, H, N, D = _check_inputs(Q1, Q2, K1, K2, V)
    if not p_ok:
        raise ValueError("dropout_p must lie in [0, 255/256] (got %r)" % dropout_p)
    q1, q2, k1, k2, v = (_in_place(t) for t in (Q1, Q2, K1, K2, V))
    if not (q1.stride() == q2.stride() == k1.stride() == k2.stride()):
        q1, q2, k1, k2 = (t.contiguous() for t in (q1, q2, k1, k2))
    dev = q1.device
    lam = _lambda_tensor(LAMBDA_SCALE, dev, Q1.dtype, H)
    with torch.cuda.device(dev):
        out = forward(q1, q2, k1, k2, v, lam, SM_SCALE, LAMBDA_INIT, flags, dropout_p, dropout_seed, differentiable,
                      q1.get_device(), _current_stream(dev), True)
    if out is None:
        raise RuntimeError("tensors of this size are out of the kernels' range")
    return (q1, q2, k1, k2, v, lam), _typed_like(V, out)


class _diff_attention(torch.autograd.Function):

    @staticmethod
    def forward(ctx, Q1, Q2, K1, K2, V, SM_SCALE, LAMBDA_SCALE, LAMBDA_INIT, rms_norm=False, causal=False,
                dropout_p=0.0, dropout_seed=0):
        differentiable = any(ctx.needs_input_grad)
        (*qkv, lam), (y, u2, lse1, lse2, rinv, flags, n_pad) = _run_forward(
            Q1, Q2, K1, K2, V, SM_SCALE, LAMBDA_SCALE, LAMBDA_INIT, rms_norm, causal, dropout_p, dropout_seed, differentiable)
        if differentiable:
            ctx.save_for_backward(*qkv, y, u2, lse1, lse2, rinv, lam)
        ctx.SM_SCALE = float(SM_SCALE)
        ctx.LAMBDA_INIT = float(LAMBDA_INIT)
        ctx.FLAGS = flags
        ctx.N_PAD = n_pad
        # the same dropout goes to the backward: the masks are a function of (seed, position) only
        ctx.DROPOUT = _dropout(dropout_p, dropout_seed)
        ctx.lambda_meta = (LAMBDA_SCALE.dtype, LAMBDA_SCALE.shape) if torch.is_tensor(LAMBDA_SCALE) else None
        return y

    @staticmethod
    @once_differentiable        # the gradients are plain kernel outputs: a second derivative raises
    def backward(ctx, dO):
        saved = ctx.saved_tensors
        dev = saved[0].device
        # only the kernels whose outputs some input asked for are launched (stage bits of the C ABI:
        # 1 row preprocess, 2 d(lambda) reduction, 4 dK/dV, 8 dQ)
        need = ctx.needs_input_grad
        want_lam = ctx.lambda_meta is not None and need[6]
        stages = (1 | (2 if want_lam else 0) | (4 if need[2] or need[3] or need[4] else 0)
                  | (8 if need[0] or need[1] else 0))

        def launch():
            return _native.host().backward(*saved, dO, ctx.SM_SCALE, ctx.LAMBDA_INIT, ctx.FLAGS, ctx.N_PAD, *ctx.DROPOUT,
                                           stages, _current_stream(dev))

        if dev.index != torch._C._cuda_getDevice():
            with torch.cuda.device(dev):
                dq1, dq2, dk1, dk2, dv, dlambda = launch()
        else:
            dq1, dq2, dk1, dk2, dv, dlambda = launch()
        if want_lam:
            dtype, shape = ctx.lambda_meta
            if dlambda.dtype != dtype or dlambda.shape != shape:
                dlambda = dlambda.to(dtype).reshape(shape)
        # one slot per forward argument: nine, or more when causal / dropout arguments were passed
        return (dq1, dq2, dk1, dk2, dv, None, dlambda) + (None,) * (len(ctx.needs_input_grad) - 7)


def diff_attention(*args):
    """`_diff_attention.apply`, without the autograd machinery where nothing can ask for it: gradients are off, and no
    transform, tracer, compiler, dispatch mode or forward-mode level is active.  (B1 H16 N77 D64 forward: about a third of
    the call's host time.)"""
    if (torch.is_grad_enabled() or torch._C._are_functorch_transforms_active() or torch._C._get_tracing_state() is not None
            or torch._C._len_torch_dispatch_stack() or forward_ad._current_level >= 0 or torch.compiler.is_compiling()):
        return _diff_attention.apply(*args)
    args += (False, False, 0.0, 0)[len(args) - 8:]
    return _run_forward(*args, False)[1][0]
