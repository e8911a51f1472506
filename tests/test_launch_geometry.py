"""The rule that chooses between the 64-row and the 128-row forward (csrc/dispatch.hpp) against measured times, on the CPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-diff-attn_amd", "csrc")

# (D, causal, N, blocks): us of a launch in 64-row and in 128-row workgroups, fp16, MI355X
MEASURED = {
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
    # bf16
    (64, False, 2048, 128): (33.8, 39.6), (64, False, 2048, 144): (56.8, 38.3), (64, False, 2048, 192): (56.9, 41.4),
    (64, True, 8192, 256): (116, 139), (64, True, 2048, 384): (61, 46), (128, True, 3072, 768): (328, 230),
}


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_the_forward_takes_the_faster_workgroups(tmp_path):
    """Of every measured pair the rule takes the faster one, or one that is within the 5 % that such a pair moves by."""
    (tmp_path / "rule.cpp").write_text('#include "dispatch.hpp"\nextern "C" int rule(int d, int causal, int n, long long blocks)'
                                       " { return da_abi::fwd_64_rows(d, causal, n, blocks); }\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(tmp_path / "rule.cpp"), "-o", str(tmp_path / "rule.so")], check=True)
    rule = ctypes.CDLL(str(tmp_path / "rule.so")).rule
    rule.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_longlong]
    slower = {k: (t64, t128) for k, (t64, t128) in MEASURED.items() if (t64 if rule(*k) else t128) > 1.05 * min(t64, t128)}
    assert not slower
