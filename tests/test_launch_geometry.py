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

# (weights, E, tokens): us of a layer's weight gradients by wgrad_kernel and as library products, fp16
WGRAD = {
    (1, 256, 77): (8.3, 13.9), (1, 256, 16384): (25.5, 91.8), (1, 384, 77): (8.4, 6.6), (1, 384, 1000): (12.3, 14.0),
    (1, 512, 256): (8.9, 7.1), (1, 512, 1000): (12.7, 14.0), (1, 512, 2048): (15.6, 17.1), (1, 512, 16384): (22.9, 98.5),
    (1, 640, 256): (8.9, 7.2), (1, 640, 8192): (27.1, 49.7), (1, 768, 1000): (15.4, 14.1), (1, 768, 2048): (18.3, 17.2),
    (1, 768, 4096): (21.8, 28.5), (1, 1024, 77): (8.6, 6.8), (1, 1024, 1000): (20.6, 14.3), (1, 1024, 2048): (22.2, 18.1),
    (1, 1024, 4096): (23.7, 30.8), (1, 1152, 1000): (18.7, 17.7), (1, 1152, 2048): (23.5, 21.7), (1, 1152, 4096): (33.0, 34.2),
    (1, 1280, 1000): (20.3, 17.5), (1, 1280, 8192): (41.4, 65.3), (1, 1536, 77): (9.0, 9.6), (1, 1536, 1000): (15.4, 21.0),
    (1, 2048, 256): (10.2, 10.7), (1, 2048, 16384): (146.4, 164.3), (1, 2560, 256): (16.5, 14.1),
    (1, 3072, 8192): (202.7, 158.2), (1, 4096, 1000): (66.9, 43.2), (2, 512, 77): (8.6, 11.9), (2, 1024, 1000): (23.1, 27.2),
    (2, 1152, 2048): (22.8, 42.0), (2, 2048, 77): (16.7, 18.8), (3, 384, 77): (8.5, 16.9), (3, 1280, 256): (16.8, 22.5),
    (3, 1792, 8192): (204.8, 235.0), (3, 3072, 2048): (162.0, 143.8), (4, 256, 1000): (12.9, 139.9),
    (4, 768, 8192): (60.8, 198.2), (4, 1024, 77): (9.7, 23.4), (4, 1024, 8192): (72.6, 211.9), (4, 1152, 77): (15.9, 27.7),
    (4, 1152, 8192): (147.2, 242.9), (4, 1536, 2048): (64.1, 100.3), (4, 2048, 77): (29.6, 36.0),
    (4, 2048, 16384): (637.0, 686.0), (4, 2560, 2048): (156.1, 143.4), (4, 2560, 8192): (516.2, 479.6),
    (4, 3072, 8192): (722.0, 637.6), (4, 4096, 16384): (2576.7, 1875.5),
}


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    tmp = tmp_path_factory.mktemp("rules")
    (tmp / "rules.cpp").write_text('#include "dispatch.hpp"\nextern "C" {\n'
                                   "int fwd(int d, int causal, int n, long long blocks) { return da_abi::fwd_64_rows(d, causal, n, blocks); }\n"
                                   "int bwd(int d, int causal, int n, long long blocks) { return da_abi::bwd_one_grid(d, false, causal, n, blocks, 15u); }\n"
                                   "int packed(int backward, long long E, long long tokens) { return da_abi::layer_packed(backward, E, tokens); }\n"
                                   "int wgrad(int weights, long long E, long long tokens) { return da_abi::wgrad_own(weights, E, tokens); }\n"
                                   "void split(long long tiles, int tokens, int* out) { auto s = da_abi::wgrad_split(tiles, tokens); out[0] = s.splits; out[1] = s.slabs; }\n"
                                   "}\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(tmp / "rules.cpp"), "-o", str(tmp / "rules.so")], check=True)
    lib = ctypes.CDLL(str(tmp / "rules.so"))
    for f in (lib.fwd, lib.bwd):
        f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_longlong]
    lib.packed.argtypes = lib.wgrad.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong]
    lib.split.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    return lib


def test_the_projections_take_the_faster_products(rules):
    """Of every measured pair the rule takes the faster one, or one within 6 % of it."""
    for backward in (0, 1):
        pairs = {k: t[2 * backward:2 * backward + 2] for k, t in PACKED.items()}
        assert not {k: (backward, one, three) for k, (one, three) in pairs.items()
                    if (one if rules.packed(backward, *k) else three) > 1.06 * min(one, three)}


def test_the_weight_gradients_take_the_faster_way(rules):
    """Within 11 %: that of a single weight at 1000 tokens of E 512, on the near side of a line that fits E 1024."""
    assert not {k: (own, lib) for k, (own, lib) in WGRAD.items() if (own if rules.wgrad(*k) else lib) > 1.11 * min(own, lib)}
    assert not rules.wgrad(4, 64, 1000) and not rules.wgrad(4, 1088, 1000)      # the kernel's tiles are 128 wide


def test_the_split_of_a_weight_gradient(rules):
    """Every slab of 64 tokens in exactly one split, none without slabs, no split of fewer than four slabs (but for the last,
    which takes what is left), and no more workgroups than CUs where there is anything to split."""
    out = (ctypes.c_int * 2)()
    for tiles in (1, 2, 4, 9, 36, 64, 100, 127, 128, 129, 144, 255, 256, 257, 1024, 4 * 128 * 128):
        for tokens in (1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1000, 4095, 4096, 4129, 16384, 100001, 2 ** 31 - 64):
            rules.split(tiles, tokens, out)
            splits, slabs = out
            whole = -(-tokens // 64)
            assert splits >= 1 and slabs >= 1 and (splits - 1) * slabs < whole <= splits * slabs, (tiles, tokens)
            assert splits == 1 or (slabs >= 4 and splits * tiles <= 256), (tiles, tokens)


def test_the_forward_takes_the_faster_workgroups(rules):
    """Of every measured pair the rule takes the faster one, or one that is within the 5 % that such a pair moves by."""
    assert not {k: (t64, t128) for k, (t64, t128) in FORWARD.items() if (t64 if rules.fwd(*k) else t128) > 1.05 * min(t64, t128)}


def test_the_backward_takes_the_faster_grid(rules):
    assert not {k: gain for k, gain in BACKWARD.items() if (1 / gain if rules.bwd(*k) else gain) > 1.04}
