"""The rules that choose between the 64-row and the 128-row forward and between one grid and two launches of a backward
(csrc/dispatch.hpp) against measured times, on the CPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-diff-attn_amd", "csrc")

# (D, causal, N, blocks): us of a launch in 64-row and in 128-row workgroups, fp16, MI355X
FORWARD = {
    (32, True, 128, 256): (7.6, 7.4), (32, True, 256, 192): (8.2, 9.1), (32, True, 512, 256): (10.4, 12.0),
    (32, True, 1024, 240): (15.6, 18.0), (32, True, 2048, 256): (25.3, 29.7),
    (64, True, 128, 128): (8.6, 9.3), (64, True, 128, 136): (15.0, 9.4), (64, True, 128, 192): (15.2, 9.7),
    (64, True, 256, 128): (10.7, 12.0), (64, True, 256, 144): (15.2, 12.1), (64, True, 256, 192): (17.3, 12.5),
    (64, True, 384, 159): (19.6, 14.4), (64, True, 512, 128): (13.6, 16.0), (64, True, 512, 152): (18.3, 16.3),
    (64, True, 512, 192): (19.6, 16.4), (64, True, 640, 135): (17.1, 18.2), (64, True, 640, 175): (21.5, 19.0),
    (64, True, 768, 144): (17.5, 19.9), (64, True, 768, 174): (22.5, 20.7), (64, True, 1024, 160): (21.9, 24.0),
    (64, True, 1024, 208): (26.1, 24.6), (64, True, 1536, 192): (27.7, 31.8), (64, True, 2048, 208): (36.8, 40.4),
    (64, True, 2048, 256): (40.1, 42.5),
    (128, True, 128, 128): (13.1, 15.4), (128, True, 128, 136): (19.7, 15.6), (128, True, 128, 240): (24.3, 18.5),
    (128, True, 256, 192): (23.9, 19.7), (128, True, 384, 159): (26.1, 23.3), (128, True, 512, 144): (22.5, 26.1),
    (128, True, 512, 192): (28.7, 26.8), (128, True, 640, 160): (25.6, 29.6), (128, True, 640, 205): (35.7, 31.7),
    (128, True, 768, 174): (33.2, 33.9), (128, True, 768, 222): (40.6, 36.2), (128, True, 1024, 192): (37.9, 40.5),
    (128, True, 1536, 192): (46.8, 55.0), (128, True, 2048, 240): (70.8, 74.0),
    (32, False, 128, 128): (5.2, 6.1), (32, False, 512, 128): (8.7, 10.7), (32, False, 2048, 144): (30.3, 28.4),
    (32, False, 2048, 192): (31.2, 28.6), (128, False, 128, 128): (11.5, 14.2), (128, False, 512, 144): (37.8, 25.2),
    (128, False, 2048, 128): (58.5, 67.4), (128, False, 2048, 256): (114.3, 94.2),
    # bf16
    (64, False, 2048, 128): (33.8, 39.6), (64, False, 2048, 144): (56.8, 38.3), (64, False, 2048, 192): (56.9, 41.4),
    (64, True, 8192, 256): (116, 139), (64, True, 2048, 384): (61, 46), (128, True, 3072, 768): (328, 230),
}


# (D, causal, N, blocks): time of the whole backward in two launches over that in one grid, fp16, N a multiple of 256 or D = 32
BACKWARD = {
    (32, False, 256, 288): 1.17, (32, False, 512, 512): 0.96, (32, False, 1024, 448): 0.93, (32, False, 1024, 576): 1.20,
    (32, False, 2048, 640): 1.14, (32, False, 2048, 1024): 0.96, (32, False, 4096, 1088): 1.11,
    (64, False, 256, 192): 1.13, (64, False, 256, 512): 0.94, (64, False, 512, 544): 1.14, (64, False, 1024, 448): 0.94,
    (64, False, 2048, 256): 1.12, (64, False, 2048, 576): 1.18, (64, False, 2048, 1024): 0.94, (64, False, 4096, 640): 1.11,
    (32, True, 128, 288): 1.10, (32, True, 128, 448): 0.91, (32, True, 128, 480): 0.94, (32, True, 128, 672): 0.92,
    (32, True, 256, 288): 1.11, (32, True, 256, 544): 1.16, (32, True, 256, 640): 1.12, (32, True, 256, 704): 1.07,
    (64, True, 256, 384): 1.13, (64, True, 256, 512): 0.96, (64, True, 256, 576): 1.14, (64, True, 256, 640): 1.11,
    (64, True, 256, 704): 1.07, (64, True, 256, 1088): 1.10,
    (64, True, 512, 192): 1.48, (64, True, 512, 528): 1.07, (64, True, 1024, 288): 1.31, (32, True, 1024, 1024): 0.90,
    (64, True, 2048, 512): 1.10, (64, True, 2048, 576): 1.06, (64, True, 2048, 1280): 0.95, (64, True, 4096, 480): 1.12,
}

# (E, tokens): us of the layer's input projections as one product with packed weights and as three, and of their input
# gradient, fp16.  (The library has kernels that fall out of their row by up to half, on either side: at 128 and 256 tokens
# of E 2304 to 4608 and at 256 and 512 of E 5120.  A rule on sizes cannot follow those, and they are not listed.  Nor are few
# tokens of E 4096 to 4608, where the host time of three products decides, as for the gradient at E 5120.)
PACKED = {
    (512, 77): (10.6, 17.7, 11.3, 19.1), (512, 8192): (32.7, 36.1, 25.6, 50.0), (1024, 32): (14.2, 18.4, 17.6, 25.6),
    (1024, 1024): (22.4, 30.0, 25.6, 33.6), (1024, 8192): (65.6, 70.4, 58.3, 94.1), (1536, 256): (26.1, 26.7, 31.1, 32.7),
    (1536, 4096): (78.4, 75.4, 75.6, 96.2), (2048, 77): (24.0, 28.5, 32.2, 33.6), (2048, 1024): (39.7, 50.5, 55.8, 63.0),
    (2048, 8192): (164.2, 162.3, 173.7, 233.2), (2304, 77): (25.9, 30.4, 35.4, 37.0), (2560, 1024): (51.6, 65.4, 98.1, 101.5),
    (2560, 4096): (131.2, 158.4, 165.9, 203.4), (3072, 1024): (76.1, 84.9, 122.5, 123.8),
    (3072, 4096): (215.9, 206.3, 218.8, 249.2), (3072, 8192): (466.4, 406.3, 419.1, 493.0),
    (3584, 77): (44.7, 58.3, 69.4, 66.1), (3584, 800): (80.7, 95.5, 111.1, 118.3), (3584, 4096): (254.0, 243.7, 270.7, 308.1),
    (4096, 512): (83.1, 90.6, 119.8, 113.3), (4096, 1024): (117.0, 129.0, 147.1, 149.3),
    (4096, 4096): (321.6, 299.4, 352.6, 399.5), (4608, 1024): (138.1, 157.8, 185.1, 183.1),
    (5120, 32): (81.7, 56.8, 0, 0), (5120, 77): (89.1, 65.4, 0, 0), (5120, 1024): (189.2, 196.7, 253.1, 242.2),
    (5120, 4096): (527.5, 575.9, 674.6, 731.3),
    (5632, 32): (115.2, 60.7, 147.5, 106.1), (5632, 1024): (242.9, 217.5, 326.1, 259.3),
    (5632, 4096): (711.6, 660.6, 1006.3, 747.5), (6144, 77): (146.1, 97.9, 247.7, 140.1),
    (6144, 4096): (889.0, 748.8, 867.5, 882.6), (8192, 77): (238.3, 124.8, 319.9, 175.4),
    (8192, 512): (299.4, 249.0, 442.0, 285.8), (8192, 4096): (1237.9, 1130.2, 1382.3, 1395.5),
    (12288, 200): (563.7, 335.1, 692.0, 543.6), (12288, 2048): (1919.3, 1465.6, 1865.3, 1666.9),
}


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    tmp = tmp_path_factory.mktemp("rules")
    (tmp / "rules.cpp").write_text('#include "dispatch.hpp"\nextern "C" {\n'
                                   "int fwd(int d, int causal, int n, long long blocks) { return da_abi::fwd_64_rows(d, causal, n, blocks); }\n"
                                   "int bwd(int d, int causal, int n, long long blocks) { return da_abi::bwd_one_grid(d, false, causal, n, blocks, 15u); }\n"
                                   "int packed(int backward, long long E, long long tokens) { return da_abi::layer_packed(backward, E, tokens); }\n}\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(tmp / "rules.cpp"), "-o", str(tmp / "rules.so")], check=True)
    lib = ctypes.CDLL(str(tmp / "rules.so"))
    for f in (lib.fwd, lib.bwd):
        f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_longlong]
    lib.packed.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong]
    return lib


def test_the_projections_take_the_faster_products(rules):
    """Of every measured pair the rule takes the faster one, or one within 6 % of it."""
    for backward in (0, 1):
        pairs = {k: t[2 * backward:2 * backward + 2] for k, t in PACKED.items()}
        assert not {k: (backward, one, three) for k, (one, three) in pairs.items()
                    if (one if rules.packed(backward, *k) else three) > 1.06 * min(one, three)}


def test_the_forward_takes_the_faster_workgroups(rules):
    """Of every measured pair the rule takes the faster one, or one that is within the 5 % that such a pair moves by."""
    assert not {k: (t64, t128) for k, (t64, t128) in FORWARD.items() if (t64 if rules.fwd(*k) else t128) > 1.05 * min(t64, t128)}


def test_the_backward_takes_the_faster_grid(rules):
    assert not {k: gain for k, gain in BACKWARD.items() if (1 / gain if rules.bwd(*k) else gain) > 1.04}
