"""The key ranges of a prefill chunk cover what its tiles walk: the planner's host arithmetic, compiled here and run over shapes."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinytitan_amd", "csrc")

# For every row the blocks of the keys it sees, row by row; a tile's are those from its first row's to its last row's.
PROGRAM = r'''
#include <cstdio>
#include <cstdlib>
#include "chunk_plan.h"

static int check(int n_cus, int D, int H, int KH, int start, int rows, int valid, int window) {
    const tt::KeyRanges r = window > 0 ? tt::plan_window_ranges(n_cus, D, H, KH, start, rows, valid, window)
                                       : tt::plan_key_ranges(n_cus, D, H, KH, rows, (valid + 31) / 32);
    if (r.n_splits < 2) return 0;
    for (int t = 0; 32 * t < rows; ++t) {
        long long first = 1LL << 40, last = -1;
        for (int row = 32 * t; row < 32 * t + 32 && row < rows; ++row) {
            const long long end = start + row + 1 < valid ? start + row + 1 : valid;
            const long long lo = window > 0 && start + row + 1 > window ? start + row + 1 - window : 0;
            if (lo / 32 < first) first = lo / 32;
            if ((end - 1) / 32 > last) last = (end - 1) / 32;
        }
        if (tt::chunk_tile_blocks(start, rows, valid, window, t) != last - first + 1 || last - first + 1 > (long long)r.n_splits * r.split_blocks) {
            std::printf("%d/%d heads of %d, %d rows behind %d keys, window %d: tile %d walks %lld blocks, %d ranges of %d\n", H, KH, D, rows,
                        start, window, t, last - first + 1, r.n_splits, r.split_blocks);
            return 1;
        }
    }
    return 0;
}

int main() {
    int bad = 0;
    // a window that begins to clip inside the chunk, and a ragged last tile: tiles in the middle walk the most
    bad += check(256, 256, 16, 2, 3980, 650, 4630, 4096) + check(256, 256, 16, 2, 3617, 513, 4130, 4096);
    bad += check(256, 128, 32, 8, 3873, 257, 4130, 4096) + check(256, 256, 24, 2, 8159, 577, 8736, 8192);
    const int heads[][3] = {{256, 16, 2}, {256, 8, 2}, {256, 24, 2}, {128, 32, 8}, {64, 16, 4}, {64, 12, 1}, {128, 12, 3}};
    for (const auto &h : heads)
        for (int window : {0, 96, 500, 1024, 3000, 4096, 8192})
            for (int rows = 256; rows < 1500; rows += 1 + (rows * 7) % 31)
                for (int at = -3; at <= 3; ++at)
                    for (int odd : {0, 1, 17, 31}) {
                        const int start = (window > 0 ? window : 6000) - rows / 2 + at * rows / 4 + odd;
                        if (start >= 0) bad += check(256, h[0], h[1], h[2], start, rows, start + rows + (odd == 17 ? 40 : 0), window);
                    }
    std::printf("%d\n", bad);
    return bad != 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_ranges_cover_every_tile(tmp_path):
    source, program = tmp_path / "plan.cpp", tmp_path / "plan"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-I", CSRC, str(source), "-o", str(program)], check=True)
    ran = subprocess.run([str(program)], capture_output=True, text=True)
    assert ran.returncode == 0, ran.stdout[-4000:]
