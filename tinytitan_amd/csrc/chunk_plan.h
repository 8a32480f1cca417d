// The routes of a prefill chunk: what its tiles walk, what the routes cost and how keys are cut into ranges.  Host arithmetic
// without a device, so that it can be run over any shape anywhere.
#pragma once

#include <algorithm>

namespace tt {

// Query heads that the split-K kernel packs into a tile of at most 32 rows: the largest divisor of a KV head's group.
inline int packed_heads(int group) {
    int gh = group;
    while (gh > 32 || group % gh != 0) --gh;
    return gh;
}

// Key blocks of 32 that the chunk's tile of rows [32 t, 32 t + 32) walks: from the block of the first key its first row sees (a
// window: the last `window` keys up to the row's own) to the block of its last row's own key.
inline int chunk_tile_blocks(int start, int q_len, int kv_valid, int window, int t) {
    const long long end = std::min<long long>(kv_valid, (long long)start + std::min<long long>(q_len, 32LL * t + 32));
    const long long first = window > 0 && start + 32LL * t + 1 > window ? start + 32LL * t + 1 - window : 0;
    return (int)((end + 31) / 32 - first / 32);
}
// The longest of them.  With a window it need be neither the first tile, whose window may still reach over key 0, nor the
// last, which may end early.
inline int longest_tile_blocks(int start, int q_len, int kv_valid, int window) {
    if (window <= 0) return chunk_tile_blocks(start, q_len, kv_valid, window, (q_len + 31) / 32 - 1);
    int longest = 0;
    for (int t = 0; t < (q_len + 31) / 32; ++t) longest = std::max(longest, chunk_tile_blocks(start, q_len, kv_valid, window, t));
    return longest;
}

// ---- The rings in LDS that the chunk kernels' copies fill (attn_prefill.hip): how many steps, a key block each, of K and of V they hold.
constexpr int kChunkRing = 4;
constexpr int in_ring(int j) { return (int)((unsigned)j % (unsigned)kChunkRing); }  // j >= 0
// Step i, and in front of step 0 a turn for each i below it down to -copies_ahead, issues the copies of step i + copies_ahead.
constexpr int copies_ahead(bool of_v) { return of_v ? kChunkRing - 2 : kChunkRing; }
// The block copied for step j of a range of `nb` blocks from block `first` on.  Past the range's last the last again, or, when a second
// tile follows (of `carry` blocks, from block 0), that tile's first, a ring of them; then a slot's blocks again: the same bytes.
constexpr int copied_block(int j, int first, int nb, int carry) {
    if (j < nb || carry == 0) return first + (j < nb ? j : nb - 1);
    const int at = in_ring(j - nb);
    return at < carry ? at : carry - 1;
}

// The kernel over halves of the keys takes two blocks a step, one for either half, and copies K and V `kHalvesAhead` steps ahead.  The last
// step's copies are left out (where they would go the halves meet), so a tile leaves kHalvesAhead steps behind its own.
constexpr int kHalvesRing = 4, kHalvesAhead = 3;
// The block that step `step` of a range of `nb` blocks from `first` on holds for `half`.  Past the range's last the last again, or, when a second
// tile follows, that tile's first ones.
constexpr int halves_block(int step, int half, int first, int nb, int next_first, int next_nb) {
    const int steps = (nb + 1) / 2, at = 2 * step + half, next = at - 2 * steps;
    return step < steps || next_nb <= 0 ? first + (at < nb ? at : nb - 1) : next_first + (next < next_nb ? next : next_nb - 1);
}
// Whether a launch over heads of 128 goes by halves of the keys: not where a tile walks so few blocks (`walk`) that what the halves hand each
// other outweighs them, which is sooner so in a launch of one round.  By halves / by roles, us: 64/8 heads, 2,048 rows behind windows of 33,
// 64, 128 and 320 keys (3, 4, 6 and 12 blocks; four rounds) 44.5 / 43.8, 44.9 / 45.2, 47.5 / 50.0, 59.0 / 63.4; 8/2 heads, 4,096 rows (one
// round) behind 128, 256 and 320 16.0 / 15.7, 17.7 / 17.7, 18.7 / 18.9.
inline bool halves_of_keys(int walk, long long workgroups, int n_cus) { return walk >= (workgroups > n_cus ? 4 : 11); }

// At most this many blocks a tile walks: of all keys up to its last row's, those that the windows of 32 rows can touch.
inline int most_tile_blocks(int start, int q_len, int kv_valid, int window) {
    const int all = (int)((std::min<long long>(kv_valid, (long long)start + q_len) + 31) / 32);
    return window > 0 ? (int)std::min<long long>(all, ((long long)window + 61) / 32 + 1) : all;
}

// What a chunk costs by the routes that serve it, in us, from timings at 16 q heads / 2 KV heads of 256, 8 / 2 of 256, 32 / 8 of
// 128 and 16 / 4 of 64, 512 to 4096 rows behind 0 to 9000 keys, whole and through windows of 1024 and 4096 keys.  `first_blocks`
// and `last_blocks`: the key blocks its first and its last tile of 32 rows walk.

// One key block of the chunk kernel's step, by how much of the chip takes part (at D = 256 the card's clock follows it; at 128 the kernel
// over halves of the keys is 10 % below, but the estimates of the other routes belong to this figure: with its own, 717 rows of 16/4 heads behind a
// window of 4,096 keys went whole, 56 us, and not in ranges, 49).
inline double chunk_step_us(int D, double fill) { return D == 256 ? 0.47 + 0.50 * fill : D == 128 ? 0.38 + 0.20 * fill : 0.45 + 0.05 * fill; }

struct ChunkEstimate {
    double us;
    bool single_tiles;  // a workgroup per tile of 32 rows instead of one per pair of them
};
// The chunk kernel over all of a tile's keys.  Tiles in pairs (long with short) make workgroups of one length whatever the
// triangle; a workgroup per tile, the longest first, uses twice the CUs where pairs leave some idle (1024 rows at position
// 0 39.4 -> 33.5 us, behind 2000 keys 124 -> 77, 2048 rows behind 8000 keys 404 -> 298, 1024 rows of 32 / 8 heads of 128 behind
// a window of 4096 keys 150 -> 80) and splits the rounds of several finer (2500 rows of 32 / 8 of 128 at position 0
// 107 -> 80).  Where both need the same rounds pairs are ahead -- the second tile's first blocks ride in behind the first's
// last: 4096 rows at position 0 138 against 148 us, 2500 rows behind 8000 keys 424 against 464 -- so single tiles have to
// promise an eighth less.
inline ChunkEstimate estimate_chunk(int n_cus, int D, int n_q_heads, int n_kv_heads, int q_len, int first_blocks, int last_blocks) {
    // a kv head's workgroups run on its own XCDs where it has whole ones
    const int xs = (n_kv_heads <= 8 && 8 % n_kv_heads == 0) ? 8 / n_kv_heads : 0;
    const int cus = xs > 0 ? xs * (n_cus / 8 > 0 ? n_cus / 8 : 1) : n_cus;
    const int n_tiles = (q_len + 31) / 32, sets = (xs > 0 ? n_q_heads / n_kv_heads : n_q_heads) / 4;
    const int singles = sets * n_tiles, pairs = sets * ((n_tiles + 1) / 2);
    const double hi = first_blocks > last_blocks ? first_blocks : last_blocks, lo = first_blocks + last_blocks - hi;
    // the longest first: no CU is done before its longest tile, before its share of all of them, or, with k rounds begun,
    // before k + 1 tiles of the length the last of those rounds begins with
    double by_tile = hi, share = singles * (hi + lo) / 2.0 / cus;
    if (share > by_tile) by_tile = share;
    for (int k = 1; k * cus < singles; ++k) {
        const double round = (k + 1) * (hi - (hi - lo) * (double)(k * cus) / (singles - 1));
        if (round > by_tile) by_tile = round;
    }
    const double by_pair = (double)((pairs + cus - 1) / cus) * (hi + lo);
    ChunkEstimate e;
    e.single_tiles = singles <= cus || by_tile < 0.88 * by_pair;
    const int workgroups = e.single_tiles ? singles : pairs;
    const double fill = workgroups < cus ? (double)workgroups / cus : 1.0;
    e.us = (D == 256 ? 11.0 : D == 128 ? 7.0 : 5.0) + (e.single_tiles ? by_tile : by_pair) * chunk_step_us(D, fill);
    return e;
}

// The chunk kernel over ranges of the key blocks that a tile walks, at most `nb_total` of them.
struct KeyRanges {
    int n_splits = 1, split_blocks = 0;
    double us = 0.0;
};
inline KeyRanges plan_key_ranges(int n_cus, int D, int n_q_heads, int n_kv_heads, int q_len, int nb_total) {
    // With ranges a workgroup takes one 32-row tile of 4 heads (not a pair of tiles) over one range of key
    // blocks.  The number of ranges by a small model of the two costs: rounds of workgroups on the chip x the
    // blocks of a range (0.8 us a block at D = 256), and the partial results -- rows x heads x D floats per range,
    // written by the kernel and read by the combine pass (~3 TB/s for the pair).  At least 8 blocks a range.
    KeyRanges r;
    const long long range_wgs = (long long)((q_len + 31) / 32) * (n_q_heads / 4);
    const double partial_us = (double)q_len * n_q_heads * D * 4.0 * 2.0 / 3.0e6;
    double best_us = 0.0;
    // (1, 2, 4 or 8 kv heads: a kv head's workgroups run on its 8 / n XCDs, an equal share each)
    const int xs = (n_kv_heads <= 8 && 8 % n_kv_heads == 0) ? 8 / n_kv_heads : 0;
    const long long xcd_cus = n_cus / 8 > 0 ? n_cus / 8 : 1;
    for (int s = 2; s <= 32 && nb_total / s >= 8; ++s) {
        const int blocks = (nb_total + s - 1) / s;
        long long rounds = (range_wgs * s + n_cus - 1) / n_cus;
        if (xs > 0) rounds = ((range_wgs / n_kv_heads * s + xs - 1) / xs + xcd_cus - 1) / xcd_cus;
        const double us = (double)rounds * blocks * 0.8 * D / 256.0 + s * partial_us;
        if (r.n_splits < 2 || us < best_us) {
            best_us = us;
            r.split_blocks = blocks;
            r.n_splits = (nb_total + blocks - 1) / blocks;
            r.us = (double)rounds * blocks * chunk_step_us(D, 1.0) + s * partial_us;
        }
    }
    return r;
}
// ... of the keys that a window leaves each tile.
inline KeyRanges plan_window_ranges(int n_cus, int D, int n_q_heads, int n_kv_heads, int start, int q_len, int kv_valid, int window) {
    return plan_key_ranges(n_cus, D, n_q_heads, n_kv_heads, q_len, longest_tile_blocks(start, q_len, kv_valid, window));
}

// Tiles of 32 packed rows that the split-K kernel makes of a chunk, and how many of them run at once.
inline long long splitk_tiles(int n_q_heads, int n_kv_heads, int q_len) {
    const int group = n_q_heads / n_kv_heads, gh = packed_heads(group), tt = 32 / gh;
    return (long long)((q_len + tt - 1) / tt) * n_kv_heads * (group / gh);
}
inline long long splitk_tiles_at_once(int n_cus, int D) { return (long long)n_cus * (D == 256 ? 1 : D == 128 ? 2 : 3); }

// The split-K kernel's tiles of 32 packed rows: key blocks per wavefront, dearer while a tile walks few of them.
inline double estimate_splitk_chunk_us(int n_cus, int D, int n_q_heads, int n_kv_heads, int q_len, int first_blocks, int last_blocks) {
    const double tiles = (double)splitk_tiles(n_q_heads, n_kv_heads, q_len), blocks = (first_blocks + last_blocks) / 2.0;
    const double block_us = D == 256 ? 1.6 * (1.0 + 18.0 / blocks) : D == 128 ? 0.87 * (1.0 + 11.0 / blocks) : 0.46 * (1.0 + 8.0 / blocks);
    return 5.0 + tiles * blocks / (4.0 * n_cus) * block_us;
}
// Tiles of one length, as a window makes them, in the whole rounds that the planner's splits leave (from 64 blocks a tile
// on; shorter walks start apart and even out).
inline double splitk_rounds_us(int n_cus, int n_q_heads, int n_kv_heads, int q_len, int blocks, double even_us) {
    const long long tiles = splitk_tiles(n_q_heads, n_kv_heads, q_len);
    if (blocks < 64 || tiles <= 0) return even_us;
    const long long splits = std::max<long long>(n_cus / tiles, 1), rounds = (tiles * splits + n_cus - 1) / n_cus;
    return 5.0 + (even_us - 5.0) * ((double)rounds * n_cus / ((double)tiles * splits));
}

}  // namespace tt
