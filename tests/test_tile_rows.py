"""The compress kernel's unconditional loads stay inside the matrix: the row a
lane reads (row_step of csrc/tile_rows.h plus the lane's own clamped part),
for every number of rows a last tile row can hold."""
import ctypes
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "tile_rows.h"
// largest row (from the tile's first) read by any lane of any round, the
// lane's part clamped as the kernel clamps it
extern "C" long long largest_row(long long rows_in_tile)
{
    long long most = -1;
    for (int k = 0; k < 8; k++)
        for (int lane = 0; lane < 64; lane++) {
            const long long row = 8 * k + lane / 8;
            const long long r = bs::row_step(k, rows_in_tile) + (row < rows_in_tile ? lane / 8 : 0);
            if (row < rows_in_tile && r != row) return 1 << 20;     // a row inside is read itself
            if (r > most) most = r;
        }
    return most;
}
"""


def test_rows_past_the_matrix_are_not_read(tmp_path):
    src, so = tmp_path / "rows.cpp", tmp_path / "rows.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "bitsparse_amd", "csrc"),
                    str(src), "-o", str(so)], check=True)
    f = ctypes.CDLL(str(so)).largest_row
    f.argtypes, f.restype = [ctypes.c_longlong], ctypes.c_longlong
    for rows in list(range(1, 65)) + [65, 128, 4096]:
        assert f(rows) == min(rows, 64) - 1, rows
