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

}  // namespace epi
