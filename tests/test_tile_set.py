"""The work list of the pair tiles (host code of libssu.so, called from a small program
built here): every tile once, parts whole and in slots of their own, the workspace
within its bound, selections cut as the whole."""
import os
import subprocess

import pytest

from conftest import PKG, ROOT

PROGRAM = r"""
#include "ssu_tiles.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>
using namespace ssu;
static bool whole(const TileSet& t, size_t tiles) {   // every tile once, in parts with consecutive slots of their own
    std::map<uint32_t, std::vector<uint32_t>> seen;
    std::vector<char> used(t.slots, 0);
    for (const TileUnit& u : t.units)
        if (u.bij != TILE_NONE) seen[u.bij].push_back(u.part);
    size_t cut = 0;
    for (auto& [bij, parts] : seen) {
        const uint32_t np = (parts[0] & 63) + 1;
        if (parts.size() != np) return false;
        cut += np > 1;
        for (uint32_t p = 0; p < np; ++p) {
            if (((parts[p] >> 6) & 63) != p || (parts[p] & 63) + 1 != np) return false;
            if (np == 1) continue;
            const uint32_t slot = parts[p] >> 12;
            if (slot != (parts[0] >> 12) + p || slot >= t.slots || used[slot]++) return false;
        }
    }
    return seen.size() == tiles && t.tiles == tiles && t.split.size() == cut;
}
int main(int, char** v) {
    const uint32_t n = atoi(v[1]), rows = atoi(v[2]), nodes = atoi(v[3]);
    const TileSet t = tile_set(n, rows, nodes);
    const size_t nb = (n + rows - 1) / rows;
    const auto keep = [](uint32_t bi, uint32_t bj) { return (bi + bj) % 3 == 0; };
    const TileSet s = tile_subset(t, keep);
    size_t kept = 0;
    for (uint32_t i = 0; i < nb; ++i)
        for (uint32_t j = i; j < nb; ++j) kept += keep(i, j);
    printf("%d %d %zu %zu\n", whole(t, nb * (nb + 1) / 2), whole(s, kept), t.slots * tile_slot_bytes(rows),
           t.units.size() == 8 * (size_t)t.per_xcd ? (size_t)1 : 0);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_set")
    src, exe = str(d / "t.cpp"), str(d / "t")
    with open(src, "w") as fh:
        fh.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "unifrac-binaries_amd", "csrc"), "-o", exe, src, "-L" + PKG, "-lssu",
                    "-Wl,-rpath," + PKG], check=True)
    return exe


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("n,nodes", [(1, 0), (2, 5), (127, 63), (128, 64), (129, 2000), (1000, 3000), (2939, 15609),
                                     (3001, 3700), (3217, 44626), (3600, 43545), (8056, 30000), (15160, 30000),
                                     (16384, 9790)])
def test_tile_set(program, rows, n, nodes):
    all_ok, some_ok, ws, padded = map(int, subprocess.run([program, str(n), str(rows), str(nodes)], check=True,
                                                           capture_output=True, text=True).stdout.split())
    assert all_ok and some_ok and padded
    assert ws <= 256 << 20
