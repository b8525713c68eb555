// hq_prefill_place.h - which queries, heads and chunks the blocks and waves of
// the prompt attention (hq_prefill_attn.hip) take, and which of them write an
// output.  Plain constexpr C++, the same code for the kernels, their launches
// and a host compiler (tests/test_prefill_place.py counts the writers of every
// output and partial).
#pragma once

namespace hq {

constexpr int kPaTile = 16;      // queries per wave
constexpr int kPaWaves = 4;      // waves (query tile, head) per block, one kv head
constexpr int kPaChunk = 64;     // positions per chunk
constexpr int kPaCUs = 256;      // (for the order of the blocks and the number of splits)

constexpr int pa_min(int a, int b) { return a < b ? a : b; }

// Queries p0 .. p0 + rows - 1; query p attends positions 0 .. p.
struct PaBatch {
    int p0, rows, kv_heads, groups;
};

constexpr int pa_chunks(int tile) { return tile * kPaTile / kPaChunk + 1; }
constexpr int pa_tiles(const PaBatch& b) { return (b.p0 + b.rows - 1) / kPaTile - b.p0 / kPaTile + 1; }
constexpr int pa_blocks_per_kv(const PaBatch& b) { return (pa_tiles(b) * b.groups + kPaWaves - 1) / kPaWaves; }

// A wave's place in the launch: block b serves kv head b % kv_heads and four
// (query tile, head) slots of it, the blocks with the longest contexts
// first -- but the second block of each CU in the opposite order, so that the
// blocks a CU starts with sum to about the same work (2000 tokens: 72 to 48
// chunks per wave slot otherwise, 64 to 56 so).  Four layers of 32 / 8 heads:
// 1024 tokens 1142 us against 1202, 1500 1713 against 1787, 2000 after 500
// 3165 against 3329; 2000 from position 0 are even, 1700 after 2000 4443
// against 4364.
struct PaSlot {
    int kvh, h, tile, nc, nc_block;   // tile: 16 positions from 16 * tile; nc: its chunks; the block's most
    bool live;                        // (false: the block's last slots repeat another wave's)
};
constexpr PaSlot pa_slot(const PaBatch& b, int block, int wave)
{
    const int tile0 = b.p0 / kPaTile;
    const int slots = pa_tiles(b) * b.groups;
    const int blocks = pa_blocks_per_kv(b);
    const int round = kPaCUs / b.kv_heads;
    int rank = block / b.kv_heads;
    if (rank >= round && rank < 2 * round && 2 * round <= blocks) rank = 3 * round - 1 - rank;
    const int slot0 = (blocks - 1 - rank) * kPaWaves;
    const int slot = pa_min(slot0 + wave, slots - 1);
    const int kvh = block % b.kv_heads;
    const int tile = tile0 + slot / b.groups;
    const int last = tile0 + pa_min(slot0 + kPaWaves - 1, slots - 1) / b.groups;
    return PaSlot{kvh, kvh * b.groups + slot % b.groups, tile, pa_chunks(tile), pa_chunks(last), slot0 + wave < slots};
}

// Launches that write chunk partials: block (x, y) takes chunks y * cpb ..
// y * cpb + cpb - 1 of its slots, with as many y as fill two blocks per CU.
struct PaPartGrid {
    int blocks, splits, cpb;
};
constexpr PaPartGrid pa_part_grid(const PaBatch& b)
{
    const int blocks = pa_blocks_per_kv(b) * b.kv_heads;
    const int nc = (b.p0 + b.rows - 1) / kPaChunk + 1;
    const int fill = 2 * kPaCUs / blocks;
    const int splits = pa_min(nc, fill > 1 ? fill : 1);
    const int cpb = (nc + splits - 1) / splits;
    return PaPartGrid{blocks, (nc + cpb - 1) / cpb, cpb};
}

// Chunks of the tiles before `tile` (tile i has i / 4 + 1).
constexpr long long pa_chunks_before(int tile)
{
    const long long a = tile / 4, b = tile % 4;
    return 2 * a * (a + 1) + b * (a + 1);
}

// What a batch's launch keeps in the workspace, per head: chunk partials (of
// every query and chunk) below kPaCUs blocks, else scores (of every tile and
// chunk).
constexpr bool pa_takes_partials(const PaBatch& b) { return pa_blocks_per_kv(b) * b.kv_heads < kPaCUs; }
constexpr long long pa_partials(const PaBatch& b) { return (long long)b.rows * ((b.p0 + b.rows - 1) / kPaChunk + 1); }
constexpr long long pa_tile_chunks(const PaBatch& b)
{
    return pa_chunks_before(b.p0 / kPaTile + pa_tiles(b)) - pa_chunks_before(b.p0 / kPaTile);
}

// The most of either over all batches of up to `rows` queries in a cache of
// `capacity` positions; neither falls as the capacity grows.  Partials: a
// launch below kPaCUs blocks has fewer than kPaCUs * kPaWaves (tile, head)
// slots.  Scores: the cache's last tiles (a batch may begin inside one).
constexpr long long pa_max_partials(int rows, int heads, int capacity)
{
    const int chunks = (capacity + kPaChunk - 1) / kPaChunk;
    return (long long)pa_min(rows, (kPaCUs * kPaWaves / heads + 1) * kPaTile) * chunks;
}
constexpr long long pa_max_tile_chunks(int rows, int capacity)
{
    const int end = (capacity + kPaTile - 1) / kPaTile;
    return pa_chunks_before(end) - pa_chunks_before(end - pa_min(end, (rows + kPaTile - 1) / kPaTile + 1));
}

// Whether a wave stores its queries' outputs at the end of its chunks, which
// begin at c_begin.  Beside partials (part) only one-chunk tiles have outputs
// to store, in the block that took their chunk: a block's slots may mix tiles
// of one and of two chunks, so such a wave can also be in a block of later
// chunks, where it has computed nothing.
constexpr bool pa_stores_output(bool part, int nc, int c_begin) { return !part || (nc == 1 && c_begin == 0); }

}  // namespace hq
