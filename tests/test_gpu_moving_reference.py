"""The forward with P*V one tile behind the exponentials (D = 32, and D = 64 in small grids without the causal mask) where the
reference of its online softmax moves: at every tile, now and then, never, and in some waves of a workgroup only, so that waves which
form a tile's probabilities a second time, waves that watch the row maxima (D = 32, from the turn of four tiles behind the first with three
moves) and waves that do neither meet at the same barriers.  The scores grow along the keys by about 3 or 20 powers of two a tile of
64 keys: the product of one feature of the queries (4) and of the keys (a whole number per tile), both exact.

The row statistics are checked by themselves, since an error of the reference cancels in y: against the logsumexp in 64 bits of the
scores of the keys with Q scaled and rounded as the kernel does.  Bound of their error, in nats: the unit roundoff u of the 16-bit
probabilities that are summed, what is lost of them below 2^-25 of the reference, and the roundings in 32 bits, each 2^-24 of at most the
largest sum S of magnitudes of a score: D + 1 in a product that starts at minus the reference (which is at most S itself), one for
each move of the reference and one for each score that it is taken from."""
import pytest
import torch

from oracle import diff_attn_oracle as orc
from test_gpu_dropout import kernel_masks, run
from util import GRAD_RTOL, Y_ATOL, make_inputs, max_abs, rel_to_max

pytestmark = pytest.mark.gpu

LN2 = 0.6931471805599453


def growing_inputs(H, N, D, growth, some, dtype):
    """q1, q2, k1, k2, v, dy; `some`: the scores of stream 1 alone grow, and in every other block of 32 rows."""
    ins = [t.to(dtype) for t in make_inputs(1, H, N, D, seed=N + growth)]
    # a tile adds 4 * step / sqrt(D) * log2(e): 3.1 and 20.4 powers of two at D = 32, 2.9 and 20.2 at D = 64
    step = {0: 0, 3: 3 if D == 32 else 4, 20: 20 if D == 32 else 28}[growth]
    if step:
        tile = (torch.arange(N) // 64).to(dtype) * step
        rows = 4.0 * (torch.arange(N) // 32 % 2 if some else torch.ones(N))
        for q, k in ((ins[0], ins[2]),) if some else ((ins[0], ins[2]), (ins[1], ins[3])):
            q[..., 0] = rows.to(dtype)
            k[..., 0] = tile
    return ins


def forward_statistics(q1, q2, k1, k2, v, causal):
    """y, lse1 and lse2 of the library's forward, as CPU tensors without padding rows."""
    import _native
    lib = _native.lib()
    B, H, N, D = q1.shape
    n_pad = -(-N // 128) * 128
    dev = [t.cuda() for t in (q1, q2, k1, k2, v)]
    lam = torch.tensor([0.5], dtype=q1.dtype, device="cuda")
    y = torch.empty_like(dev[4])
    lse = [torch.empty(B, H, n_pad, device="cuda") for _ in range(2)]
    flags = (2 if causal else 0) | (4 if q1.dtype == torch.bfloat16 else 0) | 32      # causal, bf16, n_valid rows
    _native.check(lib.diffattn_forward_padded(*[t.data_ptr() for t in dev], lam.data_ptr(), y.data_ptr(), None, lse[0].data_ptr(),
                                              lse[1].data_ptr(), None, B, H, n_pad, N, D, D ** -0.5, 0.8, flags, None, None,
                                              torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return y.cpu(), [t[..., :N].cpu() for t in lse]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("growth,some", [(0, False), (3, False), (20, False), (20, True)])
@pytest.mark.parametrize("D,causal,H,N", [
    (32, False, 2, 200), (32, False, 1, 640), (32, False, 2, 1000), (32, False, 33, 1024),       # 64-row workgroups, then 128-row ones
    (32, True, 2, 200), (32, True, 2, 1000), (32, True, 2, 1024), (32, True, 65, 600),
    (64, False, 2, 200), (64, False, 1, 640), (64, False, 2, 1000), (64, False, 3, 1024),
    (64, True, 2, 1000),
])
def test_row_statistics(D, causal, H, N, growth, some, dtype):
    print("statistics", dict(D=D, causal=causal, H=H, N=N, growth=growth, some=some, dtype=dtype), flush=True)
    q1, q2, k1, k2, v, _ = growing_inputs(H, N, D, growth, some, dtype)
    y, lse = forward_statistics(q1, q2, k1, k2, v, causal)
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    scale = torch.tensor(D ** -0.5, dtype=torch.float32) * torch.tensor(1.4426950408889634, dtype=torch.float32)
    for q, k, got in ((q1, k1, lse[0]), (q2, k2, lse[1])):
        qs = (q.float() * scale).to(dtype).double()
        for h in range(H):
            s = qs[0, h] @ k[0, h].double().T
            largest = (qs[0, h].abs() @ k[0, h].double().abs().T).max().item()
            if causal:
                s = s.masked_fill(torch.ones(N, N, dtype=torch.bool).triu(1), float("-inf"))
            want = torch.logsumexp(s * LN2, dim=-1)
            bound = u + N * 2.0 ** -25 + LN2 * 2.0 ** -24 * largest * (2 * (D + 1) + 2 * (N // 64 + 1))
            assert (got[0, h].double() - want).abs().max().item() <= bound, (h, bound)
    ref = orc.forward(q1, q2, k1, k2, v, torch.tensor([0.5], dtype=dtype), 0.8, False, causal=causal)
    assert max_abs(y, ref) <= (1 if dtype == torch.float16 else 3) * Y_ATOL


@pytest.mark.parametrize("growth,some", [(3, False), (20, False), (20, True)])
@pytest.mark.parametrize("D,causal,H,N", [
    (32, False, 2, 128), (32, False, 2, 200), (32, False, 1, 640), (32, False, 33, 512),
    (32, True, 2, 200), (32, True, 1, 1024), (32, True, 65, 512),
    (64, False, 2, 128), (64, False, 2, 200), (64, False, 1, 640), (64, False, 1, 1000),
    (64, True, 1, 640),
])
def test_dropout_where_the_reference_moves(D, causal, H, N, growth, some):
    """A move forms a tile's keep masks a second time, and its row sum, which counts the dropped probabilities too."""
    print("dropout", dict(D=D, causal=causal, H=H, N=N, growth=growth, some=some), flush=True)
    p, seed = 0.25, 77 + N
    cpu = growing_inputs(H, N, D, growth, some, torch.float16)
    n_pad = -(-N // 128) * 128
    m1, m2 = (m[:, :, :N, :N] for m in kernel_masks(1, H, n_pad, p, seed))
    y, grads = run(cpu, 0.5, 0.8, True, causal, p, seed)
    ref = orc.forward_backward(*cpu[:5], torch.tensor([0.5], dtype=torch.float16), cpu[5], 0.8, True, causal=causal,
                               keep1=m1, keep2=m2, dropout_p=p)
    assert torch.isfinite(y).all() and all(torch.isfinite(g).all() for g in grads)
    assert max_abs(y, ref[0]) <= Y_ATOL
    # The backward forms the probabilities anew, with K scaled and rounded where the forward scales and rounds Q: a logit of L
    # powers of two differs by up to 2 L u between the two, a probability by as much times ln 2.  dv is compared where that stays
    # below a fifth of its tolerance.
    logit = (4 * growth * D ** -0.5 * 1.4427 * (1 if D == 32 else 1.4)) * ((N - 1) // 64)
    if 2 * logit * 2.0 ** -12 * LN2 <= 1e-2:
        assert rel_to_max(grads[4], ref[5]) <= GRAD_RTOL, "dv"
