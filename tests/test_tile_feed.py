"""The hand-out of an image's tiles (csrc/tile_feed.h), compiled for the CPU: every tile belongs to one entry of one
group, and the blocks' first tiles are entries of their groups."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "tile_feed.h"
using namespace noor;
int main() {
    const uint32_t waves[] = {4096, 2048, 100, 37, 8, 3};
    for (uint32_t w : waves)
        for (uint32_t k = 0; k < 400; ++k) {
            // around multiples of the groups and of the waves
            const uint32_t tiles = k < 200 ? k + 1 : (k - 200) * (k - 200) * 7 + w - 3 + k % 7;
            const uint32_t blocks = tile_blocks(tiles, w);
            std::vector<uint32_t> seen(tiles, 0);
            uint32_t total = 0;
            for (uint32_t g = 0; g < kTileGroups; ++g)
                for (uint32_t i = 0; i < group_size(g, tiles); ++i, ++total) {
                    const uint32_t t = group_tile(g, i);
                    if (t >= tiles || seen[t]++) return printf("tile %u of %u\n", t, tiles), 1;
                }
            if (total != tiles) return printf("%u of %u tiles\n", total, tiles), 1;
            if (blocks >= tiles) continue;  // one block per tile
            if (blocks % kTileGroups || (blocks > w && blocks != kTileGroups)) return printf("%u blocks\n", blocks), 1;
            for (uint32_t g = 0; g < kTileGroups; ++g)
                if (group_size(g, tiles) < blocks / kTileGroups) return printf("short group of %u\n", tiles), 1;
        }
    return 0;
}
"""


def test_groups_cover_the_tiles(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "noor_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
