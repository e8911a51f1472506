"""The layer as one node (modules._diff_attn_layer, csrc/layer_host.cpp): its kernels and its gradients against the same layer
taken operation by operation, and which calls it stands for."""
import copy
import weakref

import pytest
import torch

import _native
import baselines
import modules

pytestmark = pytest.mark.gpu
_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,E", [(1, 128), (63, 128), (64, 384), (65, 256), (255, 640), (1000, 384), (4129, 256), (8192, 1024)])
def test_weight_gradient(T, E, dtype):
    """Edges of a 64-token slab, one and several splits, an operand with a row stride of its own."""
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    a = torch.randn(T, 3 * E, device="cuda", generator=gen).to(dtype)[:, E:2 * E]
    b = torch.randn(T, E, device="cuda", generator=gen).to(dtype)
    got = _native.layer().weight_gradient(a, b, torch.cuda.current_stream().cuda_stream)
    want = a.double().t() @ b.double()
    # one rounding of the result, and T additions of exact products in fp32
    bound = _ULP[dtype] * want.abs() + T * 2.0 ** -23 * (a.double().abs().t() @ b.double().abs()) + 2.0 ** -24
    assert got.dtype == dtype and bool(((got.double() - want).abs() <= bound).all())


def _step(layer, x, dy):
    x = x.clone().requires_grad_(True)
    layer.zero_grad(set_to_none=True)
    y = layer(x)
    y.backward(dy)
    return dict({n: p.grad for n, p in layer.named_parameters()}, x=x.grad, y=y.detach())


def _node(layer, x):
    return type(layer(x.clone().requires_grad_(True)).grad_fn).__name__


@pytest.mark.parametrize("B,N,H,d,causal,per_head,dtype", [
    (2, 77, 1, 32, False, False, torch.float16),          # E = 64: library weight gradients
    (1, 1, 2, 32, True, True, torch.bfloat16),
    (2, 200, 3, 64, True, True, torch.float16),           # E = 384, padded sequence
    (3, 256, 4, 64, False, True, torch.bfloat16),
    (2, 130, 2, 128, False, False, torch.float16),
    (2, 2048, 8, 64, True, False, torch.float16),         # E = 1024: one weight in four splits, four in one
    (1, 130, 40, 64, True, False, torch.float16),         # E = 5120: the widest layer whose weights are packed
    (2, 48, 40, 64, True, False, torch.bfloat16),         # ... and where those of few tokens are not, forward
    (1, 130, 41, 64, False, True, torch.float16),         # E = 5248: a product for each projection
    (2, 2050, 12, 128, True, False, torch.bfloat16),      # E = 3072 and many tokens: forward only
])
def test_layer_node_matches_its_operations(B, N, H, d, causal, per_head, dtype):
    gen = torch.Generator(device="cuda").manual_seed(N)
    E = 2 * H * d
    layer = modules.DiffAttn(E, H, depth=2, causal=causal, per_head_lambda=per_head, device="cuda", dtype=dtype)
    with torch.no_grad():
        for name, p in layer.named_parameters():
            p.normal_(1.0 if name == "head_gain" else 0.0, 0.1 if "lambda" in name or name == "head_gain" else E ** -0.5, generator=gen)
    single = copy.deepcopy(layer)
    single.out_proj.register_forward_hook(lambda *a: None)          # a hook: the operations one by one
    x = torch.randn(B, N, E, device="cuda", generator=gen).to(dtype)
    dy = torch.randn(B, N, E, device="cuda", generator=gen).add_(0.25).to(dtype)
    assert _node(layer, x) == "_diff_attn_layerBackward" and _node(single, x) != "_diff_attn_layerBackward"
    got, want = _step(layer, x, dy), _step(single, x, dy)
    for name in want:
        a, b = got[name].double(), want[name].double()
        assert got[name].dtype == want[name].dtype and got[name].shape == want[name].shape and got[name].stride() == want[name].stride()
        if N == 1 and name.startswith("lambda"):
            continue            # zero but for rounding: both softmax maps of a single position are 1, and the norm takes out the factor
        # dx and the gain's gradient have up to four roundings on the one side that the other does not have; the rest differ by the
        # order of fp32 sums, d(lambda), a sum of both signs, included: everything in front of it rounds alike on both sides
        assert (a - b).norm() <= 8 * _ULP[dtype] * b.norm(), name
    again = _step(layer, x, dy)
    assert all(torch.equal(again[n], got[n]) for n in got)
    with torch.no_grad():
        assert torch.equal(layer(x), got["y"])
    # Any subset of the gradients is what the whole gives, bit for bit but for weights: how the sum over the tokens is split
    # depends on how many weights want theirs.  Two fp32 sums of the same products that round to different values round to
    # neighbours, 2 ulp of a half apart at most.
    def same(n, g):
        if not n.endswith("weight"):
            return torch.equal(g, got[n])
        return (g.double() - got[n].double()).norm() <= 2 * _ULP[dtype] * got[n].double().norm()

    for wanted in (("x",), ("q_proj.weight",), ("k_proj.weight", "head_gain"), ("v_proj.weight", "lambda_k1"), ("out_proj.weight",)):
        part = copy.deepcopy(layer).requires_grad_(False)
        for n, p in part.named_parameters():
            p.requires_grad_(n in wanted)
        xp = x.clone().requires_grad_("x" in wanted)
        part(xp).backward(dy)
        grads = dict({n: p.grad for n, p in part.named_parameters()}, x=xp.grad)
        assert all(same(n, g) if n in wanted else g is None for n, g in grads.items()), wanted


def test_which_calls_the_node_stands_for():
    node = "_diff_attn_layerBackward"
    x = torch.randn(1, 64, 128, device="cuda").half()

    def changed(change, x=x):
        layer = modules.DiffAttn(128, 1, device="cuda")
        change(layer)
        return _node(layer, x)

    assert changed(lambda l: None) == node
    assert changed(lambda l: None, x.transpose(0, 1)) == node       # any strides of x
    for change in (lambda l: setattr(l, "q_proj", torch.nn.Sequential(l.q_proj)),
                   lambda l: setattr(l, "attention", lambda *a, **k: baselines.MultiheadDiffAttn(*a, **k)),
                   lambda l: l.v_proj.register_full_backward_hook(lambda *a: None),
                   lambda l: setattr(l, "lambda_scale", lambda: torch.full((1,), 0.5, device="cuda")),
                   lambda l: torch.nn.utils.parametrizations.weight_norm(l.k_proj),
                   lambda l: setattr(l, "attention_dropout", 0.5)):
        assert changed(change) != node
    layer = modules.DiffAttn(128, 1, device="cuda")
    # under a compiler the choice itself is traced without a break, and the single operations are what it sees
    assert torch.compile(lambda t: t + (1 if layer._fused_inputs(t) is None else 2), backend="eager", fullgraph=True)(x).equal(x + 1)
    y = layer(x.requires_grad_(True))
    (g,) = torch.autograd.grad(y.float().square().sum(), x, create_graph=True)
    with pytest.raises(RuntimeError):
        g.sum().backward()      # the operator's gradients have no derivative
    # saved tensors go through hooks that return other memory
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
        y2 = layer(x)
    dy = torch.randn_like(y2)
    assert torch.equal(torch.autograd.grad(y2, x, dy)[0], torch.autograd.grad(layer(x), x, dy)[0])


def _pair(E=256, H=2, seed=0, **options):
    """A layer that goes as one node, and the same layer operation by operation (a hook sees to that)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    layer = modules.DiffAttn(E, H, device="cuda", **options)
    with torch.no_grad():
        for name, p in layer.named_parameters():
            p.normal_(1.0 if name == "head_gain" else 0.0, 0.1 if "lambda" in name or name == "head_gain" else E ** -0.5, generator=gen)
    single = copy.deepcopy(layer)
    single.out_proj.register_forward_hook(lambda *a: None)
    x = torch.randn(2, 77, E, device="cuda", generator=gen).to(layer.head_gain.dtype)
    dy = torch.randn(2, 77, E, device="cuda", generator=gen).add_(0.25).to(x.dtype)
    return layer, single, x, dy


def test_results_may_be_written_in_place():
    """A residual added to the output, dropout on it and detach_(), an output made without gradients that meets a trainable
    tensor later, and the gradient of x: none of them is a view of anything."""
    layer, single, x, dy = _pair()
    scale = torch.full((1,), 0.5, device="cuda", dtype=x.dtype, requires_grad=True)
    results = []
    for l in (layer, single):
        xg = x.clone().requires_grad_(True)
        y = l(xg)
        assert not y._is_view() and y.is_contiguous()
        y += xg
        torch.nn.functional.dropout(y, 0.0, True, inplace=True)
        (g,) = torch.autograd.grad(y, xg, dy)
        if l is layer:
            g.mul_(scale)
        else:
            g = g * scale
        with torch.no_grad():
            n = l(xg)
        n.mul_(scale)
        l(xg).detach_().add_(1.0)
        results.append((y.detach(), g.detach(), n.detach(), torch.autograd.grad(n, scale, dy)[0]))
    for a, b in zip(*results):
        assert (a.double() - b.double()).norm() <= 8 * _ULP[x.dtype] * b.double().norm()


@pytest.mark.parametrize("wanted", [("x",), ("x", "out_proj.weight"), ("out_proj.weight",), ("head_gain",), ("q_proj.weight",),
                                    ("lambda_k1",), ("k_proj.weight", "head_gain")])
def test_only_what_a_gradient_reads_is_saved(wanted):
    """Inputs that no wanted gradient reads may be written in place before the backward, as with the single operations, and
    are not held until then."""
    layer, single, x, dy = _pair()
    # what each wanted gradient reads of the inputs, by the graph of the single operations
    reads = {"x": {"q_proj.weight", "k_proj.weight", "v_proj.weight", "out_proj.weight", "head_gain"},
             "out_proj.weight": set(), "head_gain": {"out_proj.weight"},
             "q_proj.weight": {"x", "out_proj.weight", "head_gain"}, "k_proj.weight": {"x", "out_proj.weight", "head_gain"},
             "lambda_k1": {"out_proj.weight", "head_gain", "lambda_q1", "lambda_k1", "lambda_q2", "lambda_k2"}}
    read = set().union(*(reads[n] for n in wanted))
    grads = []
    for l in (layer, single):
        for n, p in l.named_parameters():
            p.requires_grad_(n in wanted)
        xg = x.clone().requires_grad_("x" in wanted) * 1.0
        y = l(xg)
        inputs = dict(l.named_parameters(), x=xg)
        with torch.no_grad():
            for n, t in inputs.items():
                if n not in read:
                    t.add_(1.0)
        grads.append(torch.autograd.grad(y, [inputs[n] for n in wanted], dy))
    for a, b in zip(*grads):
        assert (a.double() - b.double()).norm() <= 8 * _ULP[x.dtype] * b.double().norm()
    if "x" in wanted:
        xg = x.clone().requires_grad_(True) * 1.0
        held = weakref.ref(xg)
        y = layer(xg)
        del xg
        assert held() is None and y.requires_grad


def test_only_the_gradients_asked_for_are_formed(monkeypatch):
    """Of a layer that trains as a whole, grad() of some inputs and backward(inputs=...) form what they ask for and nothing
    else."""
    layer, _, x, dy = _pair()
    x.requires_grad_(True)
    inputs = [x, *(getattr(layer, n).weight for n in ("q_proj", "k_proj", "v_proj", "out_proj")), layer.head_gain,
              layer.lambda_q1, layer.lambda_k1, layer.lambda_q2, layer.lambda_k2]
    formed = []
    native = _native.layer()

    class Recorded:
        layer_forward, wanted = native.layer_forward, native.wanted

        @staticmethod
        def layer_backward(*args):
            formed.append(native.layer_backward(*args))
            return formed[-1]

    monkeypatch.setattr(_native, "layer", lambda: Recorded)
    whole = torch.autograd.grad(layer(x), inputs, dy)
    assert all(g is not None for g in formed.pop())
    for ids in ((0,), (4,), (1, 2), (5,), (0, 4), (3, 9)):
        y = layer(x)
        grads = torch.autograd.grad(y, [inputs[i] for i in ids], dy)
        for i, g in zip(ids, grads):
            assert (g.double() - whole[i].double()).norm() <= _ULP[x.dtype] * whole[i].double().norm()
        assert tuple(i for i, g in enumerate(formed.pop()) if g is not None) == ids
    layer(x).backward(dy, inputs=[inputs[3]])
    assert [i for i, g in enumerate(formed.pop()) if g is not None] == [3]
    assert [i for i, t in enumerate(inputs) if t.grad is not None] == [3]


@pytest.mark.parametrize("frozen", [(), ("q_proj.weight", "k_proj.weight", "v_proj.weight"), ("x",), ("x", "qkv", "lambda")])
@pytest.mark.parametrize("of", ["out_proj.weight", "head_gain"])
def test_second_derivatives(of, frozen):
    """A penalty on the gradient of the output projection or of the gain is differentiable by everything that it depends on,
    also by an x that nobody holds any more and by tensors of which no values were saved."""
    layer, single, x, dy = _pair(causal=True)
    results = []
    for l in (layer, single):
        params = dict(l.named_parameters())
        for n, p in params.items():
            p.requires_grad_(not any(n.startswith(f) or f == "qkv" and n[:6] in ("q_proj", "k_proj", "v_proj") for f in frozen))
        leaf = x.clone().requires_grad_("x" not in frozen)
        factor = torch.ones((), device="cuda", dtype=x.dtype, requires_grad=True)
        calls = []
        params[of].register_hook(lambda g: calls.append(1) or 2.0 * g)
        y = l(leaf * 1.0)
        (g,) = torch.autograd.grad((y * y * factor).float().sum() / 64, params[of], create_graph=True)
        assert len(calls) == 1
        (g.float().square().sum() / 1024).backward()
        results.append((y, g, factor.grad, leaf.grad, *(p.grad for p in params.values())))
    tensors = 0
    for a, b in zip(*results):
        assert (a is None) == (b is None)
        if a is not None:
            tensors += 1
            # the same operations on values that differ by their last bits
            assert (a.double() - b.double()).norm() <= 16 * _ULP[x.dtype] * b.double().norm()
    assert tensors >= 5


def test_replacements_of_the_linear_class_are_seen(monkeypatch):
    """What replaces nn.Linear.forward, nn.Linear.__call__ or F.linear for all modules at once is called for the four
    projections, as without the node."""
    layer, _, x, _ = _pair()
    calls = []

    def recorded(f):
        def call(*args):
            calls.append(1)
            return f(*args)
        return call

    with torch.no_grad():
        want = layer(x)
        for owner, name in ((torch.nn.Linear, "forward"), (torch.nn.Linear, "__call__"), (torch.nn.functional, "linear")):
            with monkeypatch.context() as m:
                m.setattr(owner, name, recorded(getattr(owner, name)), raising=True)
                got = layer(x)
            assert len(calls) == 4, name
            calls.clear()
            assert (got.double() - want.double()).norm() <= 8 * _ULP[x.dtype] * want.double().norm()


@pytest.mark.parametrize("which", ["x", "dy", "weight"])
def test_pending_negations(which):
    """A tensor with the negative bit set is stored with the other sign, which a kernel cannot see."""
    layer, single, x, dy = _pair()
    if which == "x":
        x = torch._neg_view(-x)
    elif which == "dy":
        dy = torch._neg_view(-dy)
    else:
        for l in (layer, single):
            l.k_proj.weight = torch.nn.Parameter(torch._neg_view(-l.k_proj.weight.detach()))
    grads = []
    for l in (layer, single):
        y = l(x)
        grads.append((y, *torch.autograd.grad(y, [p for p in l.parameters() if p.dtype == x.dtype], dy)))
    for a, b in zip(*grads):
        assert (a.double() - b.double()).norm() <= 8 * _ULP[x.dtype] * b.double().norm()


def _exact(layer, x, dy):
    """The layer's step in 64 bits, from its formula."""
    p = {n: t.detach().double().requires_grad_(True) for n, t in layer.named_parameters()}
    x = x.double().requires_grad_(True)
    B, N, E = x.shape
    H, d = layer.num_heads, layer.head_dim
    q, k = ((x @ p[n + "_proj.weight"].t()).view(B, N, H, 2, d).permute(3, 0, 2, 1, 4) for n in "qk")
    v = (x @ p["v_proj.weight"].t()).view(B, N, H, 2 * d).transpose(1, 2)
    mask = torch.ones(N, N, device=x.device, dtype=torch.bool).tril() if layer.causal else torch.ones(N, N, device=x.device, dtype=torch.bool)
    a = torch.softmax((q @ k.transpose(-1, -2) / d ** 0.5).masked_fill(~mask, float("-inf")), -1)
    lam = (torch.exp((p["lambda_q1"] * p["lambda_k1"]).sum(-1)) - torch.exp((p["lambda_q2"] * p["lambda_k2"]).sum(-1)) + layer.lambda_init)
    heads = a[0] @ v - lam.reshape(-1, 1, 1) * (a[1] @ v)
    heads = heads * torch.rsqrt(heads.square().mean(-1, keepdim=True) + 1e-5) * (1 - layer.lambda_init) * p["head_gain"]
    y = heads.transpose(1, 2).reshape(B, N, E) @ p["out_proj.weight"].t()
    y.backward(dy.double())
    return dict({n: t.grad for n, t in p.items()}, x=x.grad, y=y.detach())


@pytest.mark.parametrize("E,H,N,options", [
    (384, 3, 200, dict(causal=True, per_head_lambda=True)), (512, 2, 256, dict(dtype=torch.bfloat16)), (64, 1, 77, dict(causal=True)),
    (5248, 41, 130, dict(per_head_lambda=True)), (5632, 44, 32, dict(causal=True, dtype=torch.bfloat16)),
])
def test_layer_node_is_as_exact_as_its_operations(E, H, N, options):
    """Against 64 bits: no output or gradient is further off than that of the single operations, but for the chance of the
    roundings (a tenth) and what is less than a quarter of a rounding of the result."""
    layer, single, _, _ = _pair(E, H, depth=2, **options)
    gen = torch.Generator(device="cuda").manual_seed(N)
    x, dy = (torch.randn(2, N, E, device="cuda", generator=gen).add_(m).to(layer.head_gain.dtype) for m in (0.0, 0.25))
    want, got, ref = _exact(layer, x, dy), _step(layer, x, dy), _step(single, x, dy)
    off = {n: [((g[n].double() - w).norm() / w.norm()).item() for g in (got, ref)] for n, w in want.items()}
    assert not {n: o for n, o in off.items() if o[0] > 1.1 * o[1] + _ULP[x.dtype] / 4}


def test_layer_graph_replays_match_eager():
    """A training step of the layer captured: no call of it allocates outside torch's allocator, synchronises or clears
    memory with a memset, so every replay gives the eager result, with eager work and a synchronisation in between."""
    for E, H, N in ((384, 3, 200), (5632, 44, 32)):          # with packed projections and with three products
        layer, _, _, _ = _pair(E, H, causal=True)
        gen = torch.Generator(device="cuda").manual_seed(1)
        x, dy, x2 = (torch.randn(2, N, E, device="cuda", generator=gen).half() for _ in range(3))
        want = [_step(layer, t, dy) for t in (x, x2)]
        params = dict(layer.named_parameters())
        leaf = x.clone().requires_grad_(True)
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            for _ in range(2):
                torch.autograd.grad(layer(leaf), [*params.values(), leaf], dy)
            torch.cuda.synchronize()
            with torch.cuda.graph(graph, stream=stream):
                y = layer(leaf)
                grads = torch.autograd.grad(y, [*params.values(), leaf], dy)
        for i in (0, 1, 0, 1):
            with torch.no_grad():
                leaf.copy_((x, x2)[i])
            graph.replay()
            torch.cuda.synchronize()
            for n, g in zip((*params, "x"), grads):
                assert torch.equal(g, want[i][n]), n
            assert torch.equal(y, want[i]["y"])
            _ = (x[0] @ x[0].t()).float().sum().item()


def test_layer_on_streams_of_several_threads():
    """Two threads that train the same layer's values on streams of their own get what one gets on the default stream."""
    import threading
    layer, _, x, dy = _pair(512, 4, causal=True)
    want = _step(layer, x, dy)
    torch.cuda.synchronize()
    wrong = []

    def worker():
        own, stream = copy.deepcopy(layer), torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            for _ in range(20):
                got = _step(own, x, dy)
                with torch.no_grad():
                    got["again"] = own(x)
                stream.synchronize()
                wrong.extend(n for n in want if not torch.equal(got[n], want[n]))
                if not torch.equal(got["again"], want["y"]):
                    wrong.append("without gradients")

    threads = [threading.Thread(target=worker) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_a_step_needs_little_more_memory_than_its_operations():
    """The node holds what it saved until its end, where the single operations let go of theirs one by one: at the peak, in the
    operator's backward, the scaled heads, which are 1/11 of what is held then.  What it needs in passing it gives back."""
    layer, single, _, _ = _pair(1024, 8, causal=True)
    x, dy = (torch.randn(8, 1024, 1024, device="cuda").half() for _ in range(2))
    peaks = []
    for l in (layer, single):
        leaf = x.clone().requires_grad_(True)
        for _ in range(2):
            l.zero_grad(set_to_none=True)
            leaf.grad = None
            torch.cuda.synchronize()
            base = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            l(leaf).backward(dy)
            torch.cuda.synchronize()
        peaks.append(torch.cuda.max_memory_allocated() - base)
    assert peaks[0] <= 1.1 * peaks[1], peaks
