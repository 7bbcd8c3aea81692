"""Index and address arithmetic that kernels share with the host
(csrc/index_math.hpp), compiled for the CPU: the addresses that the kernels
form stay within their operands, also at sizes no test can hold in memory."""

import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "index_math.hpp"
using namespace clspmv::launch;
extern "C" {
unsigned piece_offset(unsigned piece, unsigned kc) { return spmm_piece_offset(piece, kc); }
int piece_end(unsigned piece, unsigned kc) { return spmm_piece_end(piece, kc); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("index_math")
    src, so = d / "index_math.cpp", d / "index_math.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "clspmv_mic_amd", "csrc"), str(src), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


@pytest.mark.parametrize("k", range(5, 70))
def test_spmm_pieces_stay_in_their_tile(lib, k):
    """Every 16-byte piece that the block SpMM stages from X in 4-row tiles of
    k right-hand sides, 8 bytes each, lies in its tile (so the last tile's lies
    in X), and those that are multiplied hold their right-hand sides."""
    chunk = 8 if k <= 8 else 16
    for first in range(0, k, chunk):
        kc = min(chunk, k - first)
        for piece in range(chunk // 2):
            at = first * 8 - 8 + lib.piece_offset(piece, kc)
            assert 0 <= at and at + 16 <= 8 * k, f"chunk {first}, piece {piece}: bytes {at}..{at + 16} of {8 * k}"
            if 2 * piece + 1 < kc:
                assert at == (first + 2 * piece) * 8 and not lib.piece_end(piece, kc)
            elif 2 * piece < kc:  # the piece's second half is the right-hand side
                assert at + 8 == (first + 2 * piece) * 8 and lib.piece_end(piece, kc)
