"""The D = 128 forward with a mask in 128-row workgroups (csrc/dispatch.hpp, fwd_64_rows: always from 256 of them on), against the fp32
oracle: one block to several turns of the ring in front of the masked tail, and lengths that end in every part of the
last block.  The gradients check the saved row statistics."""
import pytest
import torch

from oracle import diff_attn_oracle as orc
from test_gpu_bf16 import BF16_GRAD_RTOL, BF16_Y_ATOL
from util import GRAD_RTOL, Y_ATOL, dlambda_rounding, make_inputs, max_abs, rel_to_max, run_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,N,causal", [
    (1, 256, 128, True),       # the tail alone
    (2, 128, 1, True),         # a single real row
    (4, 32, 256, True),
    (4, 32, 129, True),        # one real row in the last block
    (4, 32, 129, False),
    (2, 64, 255, False),
    (2, 43, 384, True),
    (3, 29, 289, False),       # the last block holds one tile and one row
    (3, 11, 1000, True),       # several turns without a test, then two with
    (3, 11, 1000, False),
    (3, 11, 900, False),       # a last tile without a real key
])
def test_masked_forward_matches_the_oracle(B, H, N, causal, dtype):
    assert B * H * (-(-N // 128)) >= 256
    fp16 = dtype == torch.float16
    y_atol, grad_rtol = (Y_ATOL, GRAD_RTOL) if fp16 else (BF16_Y_ATOL, BF16_GRAD_RTOL)
    q1, q2, k1, k2, v, dy = (t.to(dtype) for t in make_inputs(B, H, N, 128, seed=3000 + N))
    y, grads = run_kernel(q1, q2, k1, k2, v, 0.5, 0.8, True, dy, causal=causal)
    ref = orc.forward_backward(q1, q2, k1, k2, v, torch.tensor([0.5], dtype=dtype), dy, 0.8, True, causal=causal)
    assert max_abs(y, ref[0]) <= y_atol
    # Single-key rows have gradients that are exactly zero, up to the rounding of their terms: for dX, about 0.4 in each of
    # 256 features, 0.4 * 2^-12 * sqrt(256) = 1.6e-3 of a row's sum.  d(lambda) adds up such a sum for every row, B*H of
    # them single-key ones under the causal mask, of either sign.  bf16 rounds eight times as coarsely.
    tiny = 2e-3 if fp16 else 1.6e-2
    floor = dict(dlambda=tiny * (B * H) ** 0.5 if fp16 else
                 8 * dlambda_rounding((q1, q2, k1, k2, v, dy), torch.tensor([0.5]), 0.8, True, causal=causal))
    for name, g, r in zip(("dq1", "dq2", "dk1", "dk2", "dv", "dlambda"), grads, ref[1:]):
        assert rel_to_max(g, r) <= grad_rtol or max_abs(g, r) <= floor.get(name, tiny), name
