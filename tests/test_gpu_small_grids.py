"""The forward in 64-row workgroups and on either side of the lines where 128-row ones take over (csrc/dispatch.hpp,
fwd_64_rows), against the fp32 oracle: with 64-key tiles, under the causal mask, every other workgroup has an odd number
of key tiles to see and one more that is masked throughout; lengths end in every part of the last two blocks.  The gradients check the saved row statistics."""
import pytest
import torch

from oracle import diff_attn_oracle as orc
from test_gpu_dropout import kernel_masks, run
from util import GRAD_RTOL, Y_ATOL, make_inputs, max_abs, rel_to_max, run_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,H,N,causal", [
    (1, 1, 64, True),          # the second block has no real row
    (1, 3, 65, True),          # one real row in it
    (1, 3, 65, False),
    (2, 2, 63, False),         # the last tile has no real key
    (1, 2, 128, True),         # one visible tile, and two
    (2, 3, 256, True),         # half a turn of the ring, a turn, and every masked tile in between
    (1, 2, 640, True),
    (1, 2, 577, True),
    (2, 2, 577, False),
    (1, 5, 1000, True),        # several turns without a test
    (1, 5, 1000, False),
    (1, 128, 128, True),       # either side of the lines between the two
    (1, 129, 128, True),
    (1, 192, 128, True),
    (1, 193, 128, True),
    (1, 256, 128, True),
    (1, 257, 128, True),
    (1, 21, 1024, True),
    (1, 22, 1024, True),
    (1, 28, 1000, True),
    (1, 29, 1000, True),
    (1, 16, 2048, True),
    (1, 64, 255, False),
    (1, 129, 100, False),
    (1, 128, 128, False),
    (1, 129, 128, False),
    (1, 85, 300, False),
])
def test_masked_forward_matches_the_oracle(B, H, N, causal, D):
    q1, q2, k1, k2, v, dy = make_inputs(B, H, N, D, seed=4000 + N + D)
    y, grads = run_kernel(q1, q2, k1, k2, v, 0.5, 0.8, True, dy, causal=causal)
    ref = orc.forward_backward(q1, q2, k1, k2, v, torch.tensor([0.5], dtype=torch.float16), dy, 0.8, True, causal=causal)
    assert max_abs(y, ref[0]) <= Y_ATOL
    # Single-key rows have gradients that are exactly zero, up to the rounding of their terms; d(lambda) adds up such a sum
    # for each of them, B*H under the causal mask, of either sign.
    floor = dict(dlambda=2e-3 * (B * H) ** 0.5)
    for name, g, r in zip(("dq1", "dq2", "dk1", "dk2", "dv", "dlambda"), grads, ref[1:]):
        assert rel_to_max(g, r) <= GRAD_RTOL or max_abs(g, r) <= floor.get(name, 2e-3), name


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("B,H,N,causal", [
    (1, 3, 128, True),
    (1, 3, 640, False),
    (1, 2, 577, True),
    (2, 2, 577, False),
    (1, 128, 128, False),      # either side of the lines
    (1, 129, 128, False),
    (1, 192, 128, True),
    (1, 257, 65, True),
])
def test_dropout_forward_matches_the_oracle(B, H, N, causal, D):
    seed, p = 77 + N, 0.125
    cpu = make_inputs(B, H, N, D, seed=5000 + N + D)
    m1, m2 = (m[:, :, :N, :N] for m in kernel_masks(B, H, -(-N // 128) * 128, p, seed))
    # without the norm: a row whose few keys are all dropped in one map would be a norm of rounding errors
    y, _ = run(cpu, 0.5, 0.8, False, causal, p, seed)
    ref = orc.forward_backward(*cpu[:5], torch.tensor([0.5], dtype=torch.float16), cpu[5], 0.8, False, causal=causal, keep1=m1, keep2=m2,
                               dropout_p=p)
    assert max_abs(y, ref[0]) <= Y_ATOL
