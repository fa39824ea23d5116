"""Limits of the screened scans, on the CPU: a C++ program that includes epigpu_amd/csrc/screen_rules.h (no HIP)
checks them at the ends of their ranges. No GPU is used."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include "screen_rules.h"
#include <cstdio>
#include <initializer_list>
using namespace epi;
static int bad = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); bad = 1; } } while (0)

int main()
{
    // a block's number leads back to its tile, up to the longest list
    for (int TA : {32, 64})
        for (int kind = 0; kind < 3; kind++) {
            const uint64_t n = scr_blocks(TA, kind == 1 ? 32 : 64, kind != 0);
            CHECK(n >= 1 && n <= 4);
            for (uint64_t tile : {(uint64_t)0, (uint64_t)SCR_TILES / 2, (uint64_t)SCR_TILES - 1})
                for (uint64_t k = 0; k < n; k++) {
                    const uint64_t r = tile * n + k;
                    CHECK(r < (uint64_t)1 << 32);
                    CHECK((uint32_t)r / n == tile && (uint32_t)r % n == k);
                }
        }
    // every bound that epi_set_max_tiles takes: a piece stays below the longest list with as much room to spare
    for (uint64_t m : {(uint64_t)1, (uint64_t)2, (uint64_t)3, (uint64_t)1 << 25, (uint64_t)1 << 28, ((uint64_t)1 << 30) - 1}) {
        CHECK(scr_piece(m) >= 1 && (scr_piece(m) <= m / 2 || m < 2));
        CHECK(2 * (uint64_t)scr_piece(m) <= SCR_TILES);
    }
    CHECK(scr_piece((uint64_t)1 << 25) == (uint64_t)1 << 24);
    // launches of the bound: whole XCD groups, half a list of predicted candidates, within the runtime's work-items, and
    // no more pairs than the 32-bit counter counts
    for (int TA : {32, 64})
        for (int TB : {32, 64})
            for (double rate : {0.0, 1e-12, 1e-7, 2.5e-4, 2e-3}) {
                const int threads = 64 * TA / SCR_A * (TB / 32);
                const uint64_t n = scr_chunk(rate, TA, TB, threads), pairs = n * TA * TB;
                CHECK(n >= 256 && n % 256 == 0);
                CHECK(n * threads <= (uint64_t)1 << 31);
                CHECK(pairs < (uint64_t)1 << 32);
                CHECK(pairs * rate <= 0.5 * CAND_CAP);
                // not needlessly short: one more group would pass one of the bounds
                const uint64_t m = n + 256;
                CHECK(m * threads > (uint64_t)1 << 31 || m * TA * TB > (uint64_t)1 << 31 || m * TA * TB * rate > 0.5 * CAND_CAP);
            }
    return bad;
}
"""


def test_limits(tmp_path):
    src = tmp_path / "rules.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "rules"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "epigpu_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
