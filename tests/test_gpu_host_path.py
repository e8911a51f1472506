"""The host side of a call (csrc/host.cpp and kernel.py around it): the call without autograd against the one with it, and
inputs that cannot go to the kernels as they are against their plain copies, bit for bit."""
import pytest
import torch

from util import make_inputs

pytestmark = pytest.mark.gpu


def _tensors(N=77, dtype=torch.float16):
    return [t.cuda().to(dtype) for t in make_inputs(2, 3, N, 64, seed=5)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kw", [{}, {"rms_norm": True, "causal": True}, {"dropout_p": 0.25, "dropout_seed": -3},
                                {"rms_norm": True, "causal": True, "dropout_p": 0.1, "dropout_seed": 2 ** 70 + 1}])
def test_without_gradients_the_same_bits(kw, dtype):
    from layers import MultiheadDiffAttnKernel
    ins = _tensors(dtype=dtype)[:5]
    lam = torch.tensor([0.5], device="cuda", dtype=dtype)
    want = MultiheadDiffAttnKernel(*[t.requires_grad_() for t in ins], lam, 0.8, **kw)
    assert want.requires_grad
    with torch.no_grad():
        got = MultiheadDiffAttnKernel(*ins, lam, 0.8, **kw)
    with torch.inference_mode():
        inf = MultiheadDiffAttnKernel(*ins, lam, 0.8, **kw)
    assert not got.requires_grad and torch.equal(got, want) and torch.equal(inf, want)


@pytest.mark.parametrize("grad", [False, True])
def test_inputs_that_need_converting(grad):
    from layers import MultiheadDiffAttnKernel
    ins = _tensors()
    dy = ins.pop()
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)

    def run(ins, lam):
        leaves = [t.detach().requires_grad_(grad) for t in ins]
        y = MultiheadDiffAttnKernel(*leaves, lam, 0.8, True)
        if not grad:
            return [y]
        y.backward(dy)
        return [y.detach()] + [t.grad for t in leaves]

    want = run(ins, lam)
    same = lambda got: all(torch.equal(a, b) for a, b in zip(got, want))
    for l in (0.5, lam.double(), lam.cpu(), lam.reshape(1, 1, 1), torch.full((3,), 0.5, device="cuda", dtype=torch.float16),
              torch.full((6,), 0.5, device="cuda", dtype=torch.float16)[::2]):
        assert same(run(ins, l))
    mixed = list(ins)
    mixed[1] = ins[1].transpose(1, 2).contiguous().transpose(1, 2)          # not q1's strides
    assert same(run(mixed, lam))
    odd = list(ins)
    odd[4] = torch.nn.functional.pad(ins[4], (0, 4))[..., :128]             # rows not 16-byte aligned
    odd[0] = ins[0].transpose(2, 3).contiguous().transpose(2, 3)            # columns, not rows, contiguous
    assert same(run(odd, lam))
    if grad:                                                                # the upstream gradient likewise
        for other in (dy.transpose(2, 3).contiguous().transpose(2, 3), dy.transpose(0, 1).contiguous().transpose(0, 1)):
            leaves = [t.detach().requires_grad_() for t in ins]
            MultiheadDiffAttnKernel(*leaves, lam, 0.8, True).backward(other)
            assert same([want[0]] + [t.grad for t in leaves])


@pytest.mark.parametrize("layout", ["dense", "token-major", "sliced", "long"])
def test_layouts_of_the_results(layout):
    """y and dv are written in v's layout and the q/k gradients in q1's where those are permuted dense buffers, else
    compactly in the same order of dimensions; a leaf's gradient then is the buffer the kernel wrote.  The bits are those of
    dense tensors."""
    from layers import MultiheadDiffAttnKernel
    B, H, N, D = 2, 3, 77, 64
    dense = _tensors(N)
    dy = dense.pop()
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)

    def arranged(t):
        if layout == "dense":
            return t
        C = t.shape[-1]
        rows, width = (N + 3 if layout == "long" else N), (2 * C if layout == "sliced" else C)
        buf = torch.zeros(B, rows, H, width, device="cuda", dtype=t.dtype)
        view = buf.transpose(1, 2)[:, :, :N, :C]
        view.copy_(t)
        return view

    def run(ins):
        leaves = [t.detach().requires_grad_() for t in ins]
        y = MultiheadDiffAttnKernel(*leaves, lam, 0.8, True)
        return [y.detach(), *torch.autograd.grad(y, leaves, dy)]

    want = run(dense)
    ins = [arranged(t) for t in dense]
    got = run(ins)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    strides = lambda C: (H * N * C, N * C, C, 1) if layout == "dense" else (N * H * C, C, H * C, 1)
    assert [t.stride() for t in got] == [strides(2 * D)] + [strides(D)] * 4 + [strides(2 * D)]


def test_an_upstream_gradient_of_another_type():
    """autograd hands the operator gradients of its output's type; a caller of the extension module may not."""
    import _native
    from kernel import _run_forward
    ins = _tensors()
    dy = ins.pop()
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)
    (*qkv, lam), (y, u2, lse1, lse2, rinv, flags, n_pad) = _run_forward(*ins, 0.125, lam, 0.8, True, False, 0.0, 0, True)
    stream = torch.cuda.current_stream().cuda_stream
    back = lambda g: _native.host().backward(*qkv, y, u2, lse1, lse2, rinv, lam, g, 0.125, 0.8, flags, n_pad, 0.0, 0, 15, stream)
    assert all(torch.equal(a, b) for a, b in zip(back(dy.float()), back(dy)))


def test_other_threads_run_during_a_call():
    """Two threads on streams of their own get the results of one; and a call into the extension module lets go of the
    interpreter's lock: with a switch interval that never passes, a waiting thread only runs when the calling one does."""
    import sys
    import threading
    import time

    import _native
    from layers import MultiheadDiffAttnKernel
    ins = _tensors(640)
    dy = ins.pop()
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)

    def run():
        leaves = [t.detach().requires_grad_() for t in ins]
        y = MultiheadDiffAttnKernel(*leaves, lam, 0.8, True)
        y.backward(dy)
        return [y.detach()] + [t.grad for t in leaves]

    want = run()
    torch.cuda.synchronize()
    wrong = []

    def worker():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got = run()
                stream.synchronize()
                wrong.extend(i for i, (a, b) in enumerate(zip(got, want)) if not torch.equal(a, b))

    threads = [threading.Thread(target=worker) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong

    turns, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)

    forward = _native.host().forward
    row = [t[:1, :1, :1].contiguous() for t in ins]
    dev, stream = torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream
    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    try:
        sys.setswitchinterval(1000.0)       # before the thread first waits for the lock
        thread.start()
        # the outputs are kept: freeing a tensor lets go of the lock too
        outputs, seen, deadline = [], turns[0], time.monotonic() + 10
        while turns[0] == seen and time.monotonic() < deadline and len(outputs) < 20000:
            outputs.append(forward(*row, lam, 0.125, 0.8, 1, 0.0, 0, False, dev, stream, False))
        ran = turns[0] != seen
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()
    assert ran


def test_what_was_refused_stays_refused():
    from layers import MultiheadDiffAttnKernel
    q1, q2, k1, k2, v, _ = _tensors()
    unaligned = torch.empty(v.numel() + 1, device="cuda", dtype=v.dtype)[1:].view_as(v)     # contiguous, not 16-byte aligned
    with torch.no_grad():
        for args, error in (((q1, q2, k1, k2, unaligned), RuntimeError), ((q1, q2[:, :2], k1, k2, v), ValueError), ((q1, q2, k1, k2, v[..., :64]), ValueError),
                            ((q1.float(), q2, k1, k2, v), TypeError), ((q1, q2, k1.bfloat16(), k2, v), TypeError),
                            ((q1, q2, k1, k2, v.cpu()), ValueError), ((q1[:, :, :0], q2[:, :, :0], k1[:, :, :0], k2[:, :, :0], v[:, :, :0]), ValueError),
                            ((q1[:0], q2[:0], k1[:0], k2[:0], v[:0]), RuntimeError)):
            with pytest.raises(error):
                MultiheadDiffAttnKernel(*args, 0.5)
        with pytest.raises(ValueError):
            MultiheadDiffAttnKernel(q1, q2, k1, k2, v, torch.zeros(2, device="cuda"))
        with pytest.raises(ValueError):
            MultiheadDiffAttnKernel(q1, q2, k1, k2, v, 0.5, dropout_p=1.0, dropout_seed=1)
        # a transform goes to the autograd function, which has no rule for it
        with pytest.raises(RuntimeError):
            torch.func.vmap(lambda q: MultiheadDiffAttnKernel(q, q2, k1, k2, v, 0.5))(q1[None])


def _odd(t, dim, stride):
    """t with another stride for its dimension `dim`, of size 1."""
    s = list(t.stride())
    s[dim] = stride
    return torch.empty_strided(t.shape, s, dtype=t.dtype, device=t.device).copy_(t)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("dim,B,H,N", [(0, 1, 3, 77), (1, 2, 1, 77), (2, 2, 3, 1)])
def test_strides_of_dimensions_of_size_one_do_not_matter(dim, B, H, N, grad):
    """Slices of a fused projection, or tensors with any other stride that addresses nothing: the bits of plain copies.
    (A lambda given as a number takes the call the other way into the extension module.)"""
    from layers import MultiheadDiffAttnKernel
    ins = [t.cuda() for t in make_inputs(B, H, N, 64, seed=6)]
    dy = ins.pop()
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)

    def run(ins, lam):
        leaves = [t.detach().requires_grad_(grad) for t in ins]
        y = MultiheadDiffAttnKernel(*leaves, lam, 0.8, True)
        if grad:
            y.backward(dy)
        return [y.detach()] + [t.grad for t in leaves if grad]

    want = run(ins, lam)
    wide = lambda i: _odd(ins[i], dim, 2 * ins[i].stride(dim))       # as in a fused projection of two
    for changed in ({0: wide(0)}, {1: _odd(ins[1], dim, 7)}, {2: _odd(ins[2], dim, 8)}, {3: wide(3)},
                    {0: wide(0), 1: wide(1), 3: _odd(ins[3], dim, 1 << 20)}):
        mixed = [changed.get(i, t) for i, t in enumerate(ins)]
        for l in (lam, 0.5):
            assert all(torch.equal(a, b) for a, b in zip(run(mixed, l), want)), changed.keys()


@pytest.mark.parametrize("which", [0, 4])
def test_a_refusal_says_what_is_wrong(which):
    """Strides that a copy does not change (torch calls the tensor contiguous as it is) are refused as strides, pointers as
    pointers."""
    from layers import MultiheadDiffAttnKernel
    ins = [t.cuda() for t in make_inputs(2, 3, 1, 64, seed=6)][:5]
    t = ins[which]
    for bad, message in ((_odd(t, 2, 8), "strides"), (torch.empty(t.numel() + 1, device="cuda", dtype=t.dtype)[1:].view_as(t), "16-byte aligned")):
        with pytest.raises(RuntimeError, match=message):
            MultiheadDiffAttnKernel(*ins[:which], bad, *ins[which + 1:], 0.5)


@pytest.mark.parametrize("grad", [False, True])
def test_without_dropout_the_seed_is_not_looked_at(grad):
    from kernel import _diff_attention
    ins = [t.requires_grad_(grad) for t in _tensors()[:5]]
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)
    want = _diff_attention.apply(*ins, 0.125, lam, 0.8, True)
    for seed in (None, "unused", float("nan")):
        y = _diff_attention.apply(*ins, 0.125, lam, 0.8, True, False, 0.0, seed)
        assert torch.equal(y, want)
        if grad:
            y.backward(torch.ones_like(y))


def test_scales_are_whatever_float_takes():
    import numpy as np
    from kernel import _diff_attention
    ins = _tensors()[:5]
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16)
    want = _diff_attention.apply(*ins, 0.125, lam, 0.75, True)
    for sm_scale, lambda_init in (("0.125", "0.75"), (np.float64(0.125), np.float32(0.75)), (torch.tensor(0.125), torch.tensor([0.75], device="cuda"))):
        assert torch.equal(_diff_attention.apply(*ins, sm_scale, lam, lambda_init, True), want)


class _Tagged(torch.Tensor):
    pass


class _Plain(torch.Tensor):
    """A subclass whose operations return plain tensors."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        with torch._C.DisableTorchFunctionSubclass():
            return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("lam", [0.5, None])
def test_a_subclass_of_tensor_is_the_type_of_the_output(lam, grad):
    from layers import MultiheadDiffAttnKernel
    ins = _tensors()
    dy = ins.pop()
    lam = torch.full((1,), 0.5, device="cuda", dtype=torch.float16) if lam is None else lam

    def run(ins):
        leaves = [t.detach().requires_grad_(grad) for t in ins]
        with torch.set_grad_enabled(grad):
            y = MultiheadDiffAttnKernel(*leaves, lam, 0.8, True)
        if grad:
            y.backward(dy)
        return [y] + [t.grad for t in leaves if grad]

    want = run(ins)
    for given, returned in ((_Tagged, _Tagged), (_Plain, torch.Tensor), (torch.nn.Parameter, torch.Tensor)):
        got = run(ins[:4] + [ins[4].as_subclass(given) if given is not torch.nn.Parameter else torch.nn.Parameter(ins[4], requires_grad=grad)])
        assert type(got[0]) is returned and got[0].requires_grad == grad
        assert all(torch.equal(a.as_subclass(torch.Tensor), b) for a, b in zip(got, want))
