"""What large calls run, on grids just large enough for it, against the fp32 oracle: at D <= 64 the 128-row forward and the
separate dK/dV and dQ launches, the latter in 256-row workgroups, each with several turns of the ring in front of its mask;
the backwards with dropout.  In both types: the kernels are compiled, and their registers allocated, for each."""
import pytest
import torch

from oracle import diff_attn_oracle as orc
from test_gpu_bf16 import BF16_GRAD_RTOL, BF16_Y_ATOL
from test_gpu_dropout import kernel_masks, run
from util import GRAD_RTOL, Y_ATOL, dlambda_rounding, make_inputs, max_abs, rel_to_max, run_kernel

pytestmark = pytest.mark.gpu

DTYPES = {torch.float16: (Y_ATOL, GRAD_RTOL), torch.bfloat16: (BF16_Y_ATOL, BF16_GRAD_RTOL)}


def blocks(B, H, N):
    return B * H * (-(-N // 128))


def check(ins, rms_norm, y, grads, **options):
    y_atol, grad_rtol = DTYPES[ins[0].dtype]
    lam = torch.tensor([0.5])
    ref = orc.forward_backward(*ins[:5], lam, ins[5], 0.8, rms_norm, **options)
    assert y.dtype == ins[0].dtype and max_abs(y, ref[0]) <= y_atol
    for name, g, r in zip(("dq1", "dq2", "dk1", "dk2", "dv"), grads, ref[1:]):
        assert rel_to_max(g, r) <= grad_rtol, name
    assert max_abs(grads[5], ref[6]) <= 8 * dlambda_rounding(ins, lam, 0.8, rms_norm, **options)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("B,H,N,causal", [
    (1, 64, 1024, False),
    (1, 64, 1000, False),      # the last tile holds 40 keys
    (1, 64, 897, False),       # the last tile of the real length holds one key, the one behind it none
    (2, 40, 1024, True),
    (2, 40, 1000, True),
    (2, 40, 961, True),        # one real row in the last tile
])
def test_separate_launches_match_the_oracle(B, H, N, causal, D, dtype):
    # past the lines of bwd_one_grid (576 causal blocks; 512 others are two whole rounds of either launch), on 256-row blocks,
    # and with them past every line of the 64-row forward
    assert (blocks(B, H, N) > 576 if causal else blocks(B, H, N) == 512) and -(-N // 128) % 2 == 0
    ins = [t.to(dtype) for t in make_inputs(B, H, N, D, seed=6000 + N + D)]
    y, grads = run_kernel(*ins[:5], 0.5, 0.8, True, ins[5], causal=causal)
    check(ins, True, y, grads, causal=causal)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("B,H,N,D,causal", [
    (2, 20, 1024, 32, False),
    (2, 20, 1000, 32, True),
    (2, 20, 1024, 64, False),
    (2, 20, 1000, 64, False),
    (2, 20, 1024, 64, True),
    (2, 20, 897, 64, True),
    (1, 6, 1024, 128, False),      # (always 64-row forward and 128-row dQ workgroups)
    (1, 6, 1000, 128, True),
])
def test_dropout_matches_the_oracle(B, H, N, D, causal, dtype):
    assert D == 128 or (blocks(B, H, N) > 256 and -(-N // 128) % 2 == 0)      # 128-row forward, 256-row dQ workgroups
    seed, p = 99 + N, 0.125
    cpu = [t.to(dtype) for t in make_inputs(B, H, N, D, seed=7000 + N + D)]
    m1, m2 = (m[:, :, :N, :N] for m in kernel_masks(B, H, -(-N // 128) * 128, p, seed))
    # without the norm: a row whose few keys are all dropped in one map would be a norm of rounding errors
    y, grads = run(cpu, 0.5, 0.8, False, causal, p, seed)
    check(cpu, False, y, grads, causal=causal, keep1=m1, keep2=m2, dropout_p=p)
