"""Shared helpers of the parity tests: seeded synthetic inputs and the tolerance metrics."""
import torch

from synthetic import make_inputs  # noqa: F401  (the benchmark draws the same tensors)

# tolerances stated by the build's target: outputs within max-abs 2e-2 of the fp32 oracle,
# gradients within 5e-2 relative to the max-norm of the oracle gradient
Y_ATOL = 2e-2
GRAD_RTOL = 5e-2


def max_abs(a, b):
    return (a.float().cpu() - b.float().cpu()).abs().max().item()


def rel_to_max(a, ref):
    ref = ref.float().cpu()
    return (a.float().cpu() - ref).abs().max().item() / max(ref.abs().max().item(), 1e-30)


def dlambda_rounding(ins, lam, lambda_init, rms_norm, **options):
    """The scale of the rounding error of d(lambda) = -sum dX * U2: the 2-norm of the terms of that sum, in fp32, times the
    unit roundoff of the inputs' type.  The terms are as many positive as negative ones, so the sum may come out near zero;
    its error is a random walk over the roundings of U2, Y, the probabilities and the scaled Q.  Measured over 25 problems of
    each type it is 1.6 of this scale as a root mean square, 4.3 at most; the tests allow 8."""
    from oracle import diff_attn_oracle as orc
    _, aux = orc.forward(*ins[:5], lam, lambda_init, rms_norm, want_aux=True, **options)
    x, dx = aux["x"], ins[5].float()
    if rms_norm:
        r = aux["rinv"][..., None]
        dx = (1 - lambda_init) * (r * dx - r ** 3 * (dx * x).mean(-1, keepdim=True) * x)
    u = 2.0 ** -12 if ins[0].dtype == torch.float16 else 2.0 ** -9
    return u * (dx * aux["u2"]).double().norm().item()


def run_kernel(q1, q2, k1, k2, v, lam_value, lambda_init, rms_norm, dy=None, device="cuda", causal=False):
    """Runs layers.MultiheadDiffAttnKernel on the GPU; returns (y, grads or None) as CPU tensors."""
    from layers import MultiheadDiffAttnKernel

    need = dy is not None
    t = [x.to(device).requires_grad_(need) for x in (q1, q2, k1, k2, v)]
    # one lambda, or a list with one per head
    lam = torch.tensor(list(lam_value) if isinstance(lam_value, (list, tuple)) else [lam_value],
                       dtype=q1.dtype, device=device, requires_grad=need)
    extra = {"causal": True} if causal else {}
    y = MultiheadDiffAttnKernel(*t, lambda_scale=lam, lambda_init=lambda_init, rms_norm=rms_norm, **extra)
    grads = None
    if need:
        y.backward(dy.to(device))
        grads = [x.grad.cpu() for x in t] + [lam.grad.cpu()]
    torch.cuda.synchronize()
    return y.detach().cpu(), grads
