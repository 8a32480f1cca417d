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

# The chunk kernel's copies into its rings, in the order one wavefront issues them.  A copy in flight lands at any time up to the wait
# that covers it, in any order, so until then its place may hold either block: no other copy may be on its way there unless it
# brings the same block, and what a step reads has landed and is not being overwritten.
COPIES = r'''
#include <algorithm>
#include <cstdio>
#include <map>
#include <vector>
#include "chunk_plan.h"

struct Ring {
    int ahead;
    std::map<int, int> landed;                 // slot -> block
    std::vector<std::vector<std::pair<int, int>>> flying;  // by turn: (slot, block)
    int slot_off = 0, bad = 0;
    void copy(int i, int first, int nb, int carry) {
        const int j = i + ahead, slot = tt::in_ring(j + slot_off), block = tt::copied_block(j, first, nb, carry);
        for (const auto &turn : flying)
            for (const auto &c : turn) bad += c.first == slot && c.second != block;
        flying.push_back({{slot, block}});
    }
    void wait(size_t turns) {
        for (; flying.size() > turns; flying.erase(flying.begin()))
            for (const auto &c : flying.front()) landed[c.first] = c.second;
    }
    void read(int j, int first, int nb) {  // step j's block, while this step's copies fly
        const int slot = tt::in_ring(j + slot_off), want = first + std::min(j, nb - 1);
        bad += landed.count(slot) == 0 || landed[slot] != want;
        for (const auto &turn : flying)
            for (const auto &c : turn) bad += c.first == slot && c.second != want;
    }
};

static int run(bool of_v, int first, int nb, int carry) {
    Ring r{tt::copies_ahead(of_v), {}, {}};
    for (int tile = 0; tile < (carry > 0 ? 2 : 1); ++tile) {
        const int jb = tile ? 0 : first, steps = tile ? carry : nb, next = tile ? 0 : carry;
        if (tile == 0)
            for (int i = -r.ahead; i < 0; ++i) r.copy(i, jb, steps, next);
        r.wait(0);
        if (!of_v) r.read(0, jb, steps);
        for (int i = 0; i <= steps + 1; ++i) {
            r.copy(i, jb, steps, next);
            if (!of_v && i + 1 < steps) r.read(i + 1, jb, steps);
            if (of_v && i >= 1 && i - 1 < steps) r.read(i - 1, jb, steps);
            r.wait(tt::kChunkRing - 2);
        }
        r.wait(0);
        r.slot_off = tt::in_ring(r.slot_off + steps);
    }
    if (r.bad) std::printf("%s, %d blocks, then %d: %d\n", of_v ? "V" : "K", nb, carry, r.bad);
    return r.bad != 0;
}

int main() {
    int bad = 0;
    for (int of_v = 0; of_v < 2; ++of_v)
        for (int nb = 1; nb < 24; ++nb) {
            for (int carry = 0; carry < 24; ++carry) bad += run(of_v != 0, 0, nb, carry);
            bad += run(of_v != 0, 5, nb, 0);
        }
    return bad != 0;
}
'''

# The same of the kernel over halves of the keys: in step i its wavefronts read step i (K and V) and step i + 1 (K), then hand their results over in the
# place that the copies of the step behind a tile's last three would have taken.
HALVES = r'''
#include <algorithm>
#include <cstdio>
#include <map>
#include <vector>
#include "chunk_plan.h"

struct Half {
    int half = 0, off = 0, bad = 0;
    std::map<int, int> landed;
    std::vector<std::vector<std::pair<int, int>>> flying;
    int slot(int step) const { return (step + off) % tt::kHalvesRing; }
    void copy(int step, int first, int nb, int next_first, int next_nb) {
        const int block = tt::halves_block(step, half, first, nb, next_first, next_nb);
        for (const auto &turn : flying)
            for (const auto &c : turn) bad += c.first == slot(step) && c.second != block;
        flying.push_back({{slot(step), block}});
    }
    void wait(size_t turns) {
        for (; flying.size() > turns; flying.erase(flying.begin()))
            for (const auto &c : flying.front()) landed[c.first] = c.second;
    }
    void read(int step, int first, int nb) {
        if (2 * step + half >= nb) return;  // (past the half's last block: whatever is there, it is not used)
        bad += landed.count(slot(step)) == 0 || landed[slot(step)] != first + 2 * step + half;
        for (const auto &turn : flying)
            for (const auto &c : turn) bad += c.first == slot(step);
    }
};

static int run(int half, int first, int nb, int next_first, int next_nb) {
    Half h;
    h.half = half;
    for (int tile = 0; tile < (next_nb > 0 ? 2 : 1); ++tile) {
        const int jb = tile ? next_first : first, n = tile ? next_nb : nb, steps = (n + 1) / 2, nf = tile ? 0 : next_first, nn = tile ? 0 : next_nb;
        if (tile == 0) {
            for (int i = 0; i + 1 < tt::kHalvesAhead; ++i) h.copy(i, jb, n, nf, nn);
            h.wait(0);
            h.copy(tt::kHalvesAhead - 1, jb, n, nf, nn);
        }
        h.read(0, jb, n);
        for (int i = 0; i < steps; ++i) {
            h.read(i, jb, n);
            h.read(i + 1, jb, n);
            h.copy(i + tt::kHalvesAhead, jb, n, nf, nn);
            h.read(i, jb, n);
            h.read(i + 1, jb, n);
            h.wait(1);
        }
        h.wait(0);
        // where the results meet no later step's block lies
        const int meet = h.slot(steps + tt::kHalvesRing - 1);
        for (int i = 0; i < tt::kHalvesAhead; ++i) h.bad += h.slot(steps + i) == meet;
        h.landed.erase(meet);
        h.off = (h.off + steps) % tt::kHalvesRing;
    }
    if (h.bad) std::printf("half %d, %d blocks, then %d: %d\n", half, nb, next_nb, h.bad);
    return h.bad != 0;
}

int main() {
    int bad = 0;
    for (int half : {0, 1})
        for (int nb = 1; nb < 24; ++nb)
            for (int next = 0; next < 24; ++next)
                for (int next_first : {0, 3}) bad += run(half, next ? 0 : 5, nb, next_first, next);
    return bad != 0;
}
'''


def _runs(tmp_path, text):
    source, program = tmp_path / "plan.cpp", tmp_path / "plan"
    source.write_text(text)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-I", CSRC, str(source), "-o", str(program)], check=True)
    ran = subprocess.run([str(program)], capture_output=True, text=True)
    assert ran.returncode == 0, ran.stdout[-4000:]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_ranges_cover_every_tile(tmp_path):
    _runs(tmp_path, PROGRAM)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_copies_into_the_rings_meet_nowhere(tmp_path):
    _runs(tmp_path, COPIES)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_copies_of_the_halves_meet_nowhere(tmp_path):
    _runs(tmp_path, HALVES)
