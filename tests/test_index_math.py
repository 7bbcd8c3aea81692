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
int shadow(unsigned row, int rows) { return shadow_row(row, rows); }
int writes_y(int known, int device_memory, int at, int server) {
    return kernel_writes_y(known, device_memory, at, server);
}
long long plane(int aligned) { return block_plane(aligned); }
// Visits of strided(); -1: one of them outside [0, n).
long long visits(long long first, long long step, long long n) {
    long long count = 0;
    try {
        strided(first, step, n, [&](long long i) {
            if (i < 0 || i >= n) throw 0;
            ++count;
        });
    } catch (int) {
        return -1;
    }
    return count;
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("index_math")
    src, so = d / "index_math.cpp", d / "index_math.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "clspmv_mic_amd", "csrc"), str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.plane.restype = lib.visits.restype = ctypes.c_longlong
    lib.visits.argtypes = [ctypes.c_longlong] * 3
    return lib


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


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 513, 2**31 - 513, 2**31 - 512, 2**31 - 257, 2**31 - 64, 2**31 - 1])
@pytest.mark.parametrize("group", [64, 256, 512, 1024])
def test_rows_past_the_end_shadow_the_last(lib, rows, group):
    """The rows of a grid's last work-group, also where they pass 2^31."""
    first = (rows - 1) // group * group
    for t in range(group):
        row = first + t
        assert lib.shadow(ctypes.c_uint(row), rows) == min(row, rows - 1)


@pytest.mark.parametrize("aligned", [64, 2**29 - 64, 2**29, 2**31 - 64])
def test_block_plane(lib, aligned):
    assert lib.plane(aligned) == 4 * aligned


@pytest.mark.parametrize("n", [0, 1, 300, 524_288, 524_289, 2**31 - 524_289, 2**31 - 524_288, 2**31 - 1])
def test_strided_ends_at_n(lib, n):
    """The copy of y columns: a grid of up to 2,048 x 256 threads."""
    step = min((n + 255) // 256, 2048) * 256
    for first in (0, 1, step - 1):
        if first >= 0 and step:
            assert lib.visits(first, step, n) == max(0, (n - first + step - 1) // step)


@pytest.mark.parametrize("known, device_memory, at, server, kernel", [
    (1, 1, 0, 0, 1), (1, 1, 3, 3, 1),  # the server's GPU
    (1, 1, 1, 0, 0), (1, 1, 0, 1, 0),  # another device: there may be no peer access
    (1, 0, 0, 0, 0),                   # host memory
    (0, 0, 0, 0, 0), (0, 1, 0, 0, 0),  # a pointer that the runtime does not know
])
def test_who_writes_device_y(lib, known, device_memory, at, server, kernel):
    assert lib.writes_y(known, device_memory, at, server) == kernel
