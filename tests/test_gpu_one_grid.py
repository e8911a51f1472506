"""Backwards whose dK/dV and dQ blocks share one grid (csrc/dispatch.hpp, bwd_one_grid), and the ones just past the line where they
become two launches again, against the fp32 oracle: every head dim, masks, ragged lengths, one block to two rounds of
blocks, and calls that ask for one kind of gradient only."""
import pytest
import torch

from oracle import diff_attn_oracle as orc
from test_gpu_full_grids import check
from util import GRAD_RTOL, Y_ATOL, make_inputs, max_abs, rel_to_max, run_kernel

pytestmark = pytest.mark.gpu

NAMES = ("dq1", "dq2", "dk1", "dk2", "dv", "dlambda")


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,H,N,causal", [
    (1, 1, 128, False),        # one block of each kind
    (1, 1, 1, True),           # a single row
    (1, 3, 384, True),         # an odd number of blocks per unit, half a turn of the rings first
    (2, 5, 640, False),
    (1, 2, 1000, True),        # ragged
    (1, 257, 128, False),      # one block more than there are CUs
    (2, 65, 250, False),       # ragged, a second round
    (4, 72, 256, True),
    (1, 289, 256, True),
    (2, 128, 256, False),      # 512 and 514 blocks: either side of the line at D <= 64
    (1, 257, 256, False),
])
def test_gradients_match_the_oracle(B, H, N, causal, D):
    q1, q2, k1, k2, v, dy = make_inputs(B, H, N, D, seed=1000 + N + D)
    y, grads = run_kernel(q1, q2, k1, k2, v, 0.5, 0.8, True, dy, causal=causal)
    ref = orc.forward_backward(q1, q2, k1, k2, v, torch.tensor([0.5], dtype=torch.float16), dy, 0.8, True, causal=causal)
    assert max_abs(y, ref[0]) <= Y_ATOL
    # the smallest problems have gradients that are exactly or almost zero (a single key): an absolute floor of one
    # 16-bit rounding of the terms they are summed from
    for name, g, r in zip(NAMES, grads, ref[1:]):
        assert rel_to_max(g, r) <= GRAD_RTOL or max_abs(g, r) <= 2e-3, name


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("H,N", [
    (216, 256), (217, 256),    # 432 and 434 blocks of two to a unit
    (144, 512), (145, 512),    # 576 and 580 of four
    (384, 128), (385, 128),    # single ones (at D = 64 always one grid)
])
def test_either_side_of_the_causal_lines(H, N, D):
    ins = make_inputs(1, H, N, D, seed=1500 + N + D)
    y, grads = run_kernel(*ins[:5], 0.5, 0.8, True, ins[5], causal=True)
    check(ins, True, y, grads, causal=True)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("N", [256, 384])
def test_one_kind_of_gradient_only(N, D):
    """Asked for the gradients of q (or of k and v) alone, the grid holds blocks of one kind: the same bits as in a full
    backward."""
    from layers import MultiheadDiffAttnKernel
    ins = [t.cuda() for t in make_inputs(1, 4, N, D, seed=N)]
    dy = ins.pop()

    def run(grad_of):
        leaves = [t.clone().requires_grad_(i in grad_of) for i, t in enumerate(ins)]
        lam = torch.tensor([0.4], dtype=torch.float16, device="cuda", requires_grad=True)
        MultiheadDiffAttnKernel(*leaves, lam, 0.8, True).backward(dy)
        return [t.grad for t in leaves] + [lam.grad]

    full = run({0, 1, 2, 3, 4})
    for part in ({0, 1}, {2, 3, 4}):
        got = run(part)
        assert torch.equal(got[5], full[5])
        for i in range(5):
            assert torch.equal(got[i], full[i]) if i in part else got[i] is None
