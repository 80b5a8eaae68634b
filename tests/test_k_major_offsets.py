"""The byte arithmetic of the K-major loads (csrc/k_major.h), compiled for the CPU, at the bounds of what the library
sends to it: every load lands on the row and column that it stands for, and nothing past the matrix is readable."""
import ctypes
import os
import subprocess

import pytest

from conftest import PKG_ROOT

CSRC = os.path.join(PKG_ROOT, "csrc")
SOURCE = r"""
#define __host__
#define __device__
#include "k_major.h"
extern "C" int fits(int64_t k, int64_t cols) { return wx::k_major_fits(k, cols); }
extern "C" uint32_t offset(int lane, int wave, int i, int tile_cols, uint32_t row_bytes) {
  return wx::k_major_offset(lane, wave, i, tile_cols, row_bytes);
}
extern "C" uint32_t left(uint32_t bytes, uint32_t step) { return wx::k_major_left(bytes, step); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("k_major")
    (d / "k.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "k.cpp"), "-o", str(d / "k.so")], check=True)
    lib = ctypes.CDLL(str(d / "k.so"))
    lib.fits.argtypes = [ctypes.c_int64, ctypes.c_int64]
    lib.offset.argtypes = [ctypes.c_int] * 4 + [ctypes.c_uint32]
    lib.offset.restype = lib.left.restype = ctypes.c_uint32
    lib.left.argtypes = [ctypes.c_uint32, ctypes.c_uint32]
    return lib


# 2^22 - 8: the longest row that B may have; 2^23: where a 24-bit product of a pitch in bytes begins to be wrong; 2^26 - 8:
# the longest row that A may have
COLS = [8, 264, 2 ** 22 - 8, 2 ** 23 - 8, 2 ** 23, 2 ** 23 + 8, 2 ** 24 + 8, 2 ** 26 - 8]


@pytest.mark.parametrize("tile_cols", [128, 256])
@pytest.mark.parametrize("cols", COLS)
def test_offsets_are_those_of_the_matrix(lib, tile_cols, cols):
    chunks, rows = tile_cols // 8, 1024 // (2 * tile_cols)
    seen = set()
    for wave in range(4):
        for i in range(8 // rows):
            for lane in range(64):
                row = 8 * wave + rows * i + lane // chunks
                at = lib.offset(lane, wave, i, tile_cols, 2 * cols)
                # the chunk's place inside the tile's row: its 32-byte unit u of row r lies at u ^ 2 (r & 3) ^ ((r >> 3) & 1)
                unit = (lane % chunks >> 1) ^ (2 * (row & 3)) ^ ((row >> 3) & 1)
                want = row * 2 * cols + (2 * unit + (lane & 1)) * 16
                assert at == want < 2 ** 32, (wave, i, lane)
                seen.add((row, at - row * 2 * cols))
    assert seen == {(r, 16 * c) for r in range(32) for c in range(chunks)}


@pytest.mark.parametrize("cols", COLS)
def test_nothing_past_the_matrix_is_readable(lib, cols):
    top = min((2 ** 32 - 1) // (2 * cols), 100)
    for k in sorted({1, 5, min(31, top), min(32, top), min(33, top), top}):
        assert lib.fits(k, cols)
        for col0 in (0, (cols - 1) // 256 * 256):
            left = (k * cols - col0) * 2
            for step in range((k + 31) // 32 + 8):  # the ring's padding steps among them
                exact = (k * cols - col0) * 2 - step * 64 * cols
                assert left == max(exact, 0)
                for row in range(32):  # the first byte of a row past K is never inside what is left
                    if 32 * step + row >= k:
                        assert row * 2 * cols >= left
                left = lib.left(left, 64 * cols)


def test_what_does_not_fit_is_refused(lib):
    assert lib.fits(1, 2 ** 26 - 8) and not lib.fits(1, 2 ** 26) and not lib.fits(1, 2 ** 27 + 8)
    assert lib.fits(2 ** 20 - 1, 2 ** 11) and not lib.fits(2 ** 20, 2 ** 11)
