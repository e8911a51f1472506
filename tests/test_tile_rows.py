"""The clamped rows of a tile copy (csrc/tile_rows.hpp) against their definition, on the CPU: every piece of a tile in front of, across
and behind the end of its tensor, as the copies that are always clamped meet them."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-diff-attn_amd", "csrc")


@pytest.fixture(scope="module")
def clamp_piece(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("tile_rows")
    src, out = d / "t.cpp", d / "t.so"
    src.write_text('#include "tile_rows.hpp"\n'
                   'extern "C" int piece_base(int f, int l, int n) { return da_abi::clamp_piece(f, l, n).base; }\n'
                   'extern "C" int piece_most(int f, int l, int n) { return da_abi::clamp_piece(f, l, n).most; }\n')
    subprocess.run([cxx, "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(src), "-o", str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    return lambda *a: (lib.piece_base(*a), lib.piece_most(*a))


@pytest.mark.parametrize("rows", [2, 4, 8, 16])      # of a piece of 256, 128, 64 and 32 columns
def test_every_row_is_the_tensors_or_its_last(clamp_piece, rows):
    for first in range(0, 64, rows):
        for last_row in list(range(-200, 72)) + [1 << 20]:
            base, most = clamp_piece(first, last_row, rows)
            assert 0 <= most < rows                  # a lane's way down stays inside the piece
            for r in range(rows):
                assert base + min(r, most) == min(first + r, last_row), (first, last_row, r)
