// Limits of the screened scans (kern_screen.h), as host code reads them too. Plain C++.
#pragma once

#include <cstddef>
#include <cstdint>

namespace epi {

constexpr int SCR_A = 16;  // a-SNPs of a wave

// Blocks of a tile that the exact tiles redo: 32 x 64 pairs (FAST) or 32 x 32 (tiles with missing calls), the pairs of
// two waves, each of which marks its half. They are numbered tile * blocks + k over a list of one kind, in 32 bits.
constexpr int scr_blocks(int TA, int TB, bool gen) { return TA / 32 * (gen ? TB / 32 : 1); }

// Tiles of a list whose blocks can be numbered, whatever the kind.
constexpr size_t SCR_TILES = (1ull << 32) / scr_blocks(64, 64, true);

// Tiles of a screened piece of a scan under the caller's bound: half of it, since the blocks to redo take the room of as
// many tiles again, and half of what can be numbered, since a piece ends with a whole row of super-tiles.
constexpr size_t scr_piece(size_t max_tiles)
{
    const size_t n = max_tiles / 2;
    return n < 1 ? 1 : n < SCR_TILES / 2 ? n : SCR_TILES / 2;
}

// Candidates that the list holds (16 MiB). A wave whose candidates find no room hands its pairs to the exact tiles.
constexpr uint32_t CAND_CAP = 1u << 20;

// Most tiles of TA x TB that one launch of the bound takes before the list is resolved and emptied, with `rate`
// candidates predicted per pair and `threads` threads per tile: half a list of them, within the 2^31 work-items that
// the runtime counts in a launch and so few pairs that the list's 32-bit counter cannot wrap even if a wave
// appended all of its own. A multiple of 256 (xcd_tile). A list for the whole scan, whatever its pairs, filled up early at
// a high rate, and the pairs around all later candidates went to the exact tiles: N = 8000, M = 50000, test f at p < 1e-3
// took 110 ms (exact tiles alone 96 ms), now 43.
constexpr int scr_chunk(double rate, int TA, int TB, int threads)
{
    const double pairs = (double)TA * TB;
    double n = 2147483648.0 / threads;
    if (n * pairs > 2147483648.0) n = 2147483648.0 / pairs;
    if (n * pairs * rate > 0.5 * CAND_CAP) n = 0.5 * CAND_CAP / (pairs * rate);
    return n < 512.0 ? 256 : (int)n / 256 * 256;
}

}  // namespace epi
