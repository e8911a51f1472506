"""The forward with P*V one tile behind the exponentials and row sums watched instead of row maxima (D = 32, and D = 64 in small
grids without the causal mask) at its edges: one to ten
tiles of 64 keys with an even and an odd number of turns of its ring, sequences that end inside a tile, and scores that grow along
the keys: by 0, 3 and 20 powers of two a tile at D = 32, so that the reference moves never, now and then, and at every tile, in the last case
past the range of fp16; by 0, 2 and 14 at D = 64, where few probabilities pass it.  (test_gpu_moving_reference.py has the growth of D = 32 at both,
dropout, and the row statistics by themselves, of which only those of short sequences are checked here, through dv.)  The growth is the product of one feature of the queries (4) and of the keys (a whole number per tile), both
exact; what rounding it meets is common to the keys of a tile, and keys of other tiles differ by far more.  So the tolerances
are those of any other input: 2e-2 of y and 5e-2 of a gradient's maximum in fp16, 6e-2 and 8e-2 in bf16."""
import pytest
import torch

from oracle import diff_attn_oracle as orc
from util import GRAD_RTOL, Y_ATOL, make_inputs, max_abs, rel_to_max, run_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("growth", [0, 3, 20])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("H,N", [(2, 1), (2, 64), (2, 77), (3, 128), (2, 200), (2, 384), (1, 640), (160, 256), (300, 77)])
def test_forward_of_narrow_heads(H, N, D, growth, causal, dtype):
    q1, q2, k1, k2, v, dy = (t.to(dtype) for t in make_inputs(1, H, N, D, seed=N + growth))
    if growth:
        tile = (torch.arange(N) // 64).to(dtype) * growth
        for q, k in ((q1, k1), (q2, k2)):
            q[..., 0] = 4
            k[..., 0] = tile
    y, grads = run_kernel(q1, q2, k1, k2, v, 0.5, 0.8, True, dy, causal=causal)
    ref = orc.forward_backward(q1, q2, k1, k2, v, torch.tensor([0.5], dtype=dtype), dy, 0.8, True, causal=causal)
    wide = 1 if dtype == torch.float16 else 3
    assert torch.isfinite(y).all() and all(torch.isfinite(g).all() for g in grads)
    assert max_abs(y, ref[0]) <= wide * Y_ATOL
    # The backward forms the probabilities anew from the forward's statistics, with the keys scaled and rounded where the forward
    # scales and rounds the queries: a logit of L powers of two differs by up to 2 L u between the two, a probability by as much
    # times ln 2.  Where that stays below a fifth of the tolerance, dv tells whether the statistics are right.
    unit = 2.0 ** -12 if dtype == torch.float16 else 2.0 ** -9
    logit = growth * ((N - 1) // 64) * 4 * D ** -0.5 * 1.4427
    if 2 * logit * unit * 0.6931 > 1e-2:
        return
    assert rel_to_max(grads[4], ref[5]) <= (GRAD_RTOL if dtype == torch.float16 else 8e-2), "dv"
