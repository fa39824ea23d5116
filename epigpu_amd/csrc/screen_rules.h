// Limits of the screened scans (kern_screen.h), as host code reads them too. Plain C++.
#pragma once

#include <cstddef>
#include <cstdint>

namespace epi {

constexpr int SCR_A = 16;  // a-SNPs of a wave

// Regions that a tile can hand to the exact tiles: one of SCR_A x 64 pairs per wave (FAST), or of SCR_A x 32
// (tiles with missing calls; those of 64 b-SNPs run as two halves). They are numbered tile * regions + k over
// a launch's list of one kind, in 31 bits: the highest marks a whole tile.
constexpr int scr_regions(int TA, int TB, bool gen) { return TA / SCR_A * (gen ? TB / 32 : 1); }
constexpr uint32_t SCR_WHOLE = 1u << 31;

// Tiles of a list whose regions can be numbered, whatever the kind.
constexpr size_t SCR_TILES = SCR_WHOLE / scr_regions(64, 64, true);

// Tiles of a screened piece of a scan under the caller's bound: half of it, since the regions take the room of as
// many tiles again, and half of what can be numbered, since a piece ends with a whole row of super-tiles.
constexpr size_t scr_piece(size_t max_tiles)
{
    const size_t n = max_tiles / 2;
    return n < 1 ? 1 : n < SCR_TILES / 2 ? n : SCR_TILES / 2;
}

// Candidates that the list holds (16 MiB). A region whose candidates find no room is redone by exact tiles.
constexpr uint32_t CAND_CAP = 1u << 20;

// Most tiles of TA x TB that one launch of the bound takes before the list is resolved and emptied, with `rate`
// candidates predicted per pair and `threads` threads per tile: half a list of them, within the 2^31 work-items that
// the runtime counts in a launch and so few pairs that the list's 32-bit counter cannot wrap even if a wave
// appended all of its own. A multiple of 256 (xcd_tile). A list for the whole scan, whatever its pairs, filled up early at
// a high rate, and the regions of all later candidates went to the exact tiles: N = 8000, M = 50000, test f at p < 1e-3
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
