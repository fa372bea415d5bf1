"""k_gemm_f32's loads stay inside the rows they are given: f32_tile.h, compiled
for the CPU, over every lane and load of both tile sizes, for full tiles and
tiles that end anywhere inside."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include <cstdio>
#include <initializer_list>
#include "f32_tile.h"
int main() {
    for (int tile : {16, 32, 64})                 // rows a buffer is read for
        for (int K : {32, 96, 800, 2080, 8192})
            for (int rows = 1; rows <= tile; rows++) {
                unsigned seen[64] = {};           // pieces of each row that some lane reads
                for (int i = 0; i < tile / 8; i++)
                    for (int lane = 0; lane < 64; lane++) {
                        const int off = ehip::f32_load_offset(lane, i, K, rows), row = 8 * i + lane / 8;
                        // with the last block's scalar offset
                        if (off < 0 || off + (K / 32 - 1) * 128 + 16 > rows * K * 4) {
                            printf("tile %d K %d rows %d lane %d load %d: offset %d\n", tile, K, rows, lane, i, off);
                            return 1;
                        }
                        if (row < rows) {
                            const int piece = off - row * K * 4;
                            if (piece < 0 || piece >= 128 || piece % 16) { printf("row %d: piece at %d\n", row, piece); return 1; }
                            // the place in LDS (16 bytes a lane) that the fragment reads look for it
                            if (((piece / 16) ^ ((row >> 1) & 7)) != (lane & 7)) { printf("row %d lane %d: swizzle\n", row, lane); return 1; }
                            seen[row] |= 1u << piece / 16;
                        }
                    }
                for (int r = 0; r < rows; r++)
                    if (seen[r] != 0xff) { printf("row %d: pieces %x\n", r, seen[r]); return 1; }
            }
    puts("ok");
}
"""


def test_loads_stay_inside_their_rows(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no C++ compiler")
    (tmp_path / "b.cc").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-I", os.path.join(ROOT, "emberllm_amd", "csrc", "hip"), "-o", str(tmp_path / "b"),
                    str(tmp_path / "b.cc")], check=True)
    r = subprocess.run([str(tmp_path / "b")], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
