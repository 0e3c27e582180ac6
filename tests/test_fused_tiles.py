"""What the one-launch networks (csrc/dense_fused.hip) ask for ahead of need, checked on the host: the kernel's own functions
for its tiles and its packed weights, compiled for the CPU and walked for every workgroup of a launch."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "khan_amd", "csrc")
PROGRAM = r"""
#include "dense_fused_tiles.h"
#include <cstdio>
#include <cstdlib>
using namespace khan;
static void require(bool ok, const char* what) { if (!ok) { std::puts(what); std::exit(1); } }

// The last byte that a workgroup's lanes load of chunk c (each column's two halves of 16 bytes) lies in the packed weights.
static void inside(int type, int matrix, int cols, int K, int column_tile, int c)
{
    const int from = packed_chunk_at(type, matrix, cols, K, column_tile, c);
    require(from >= 0 && from + kFusedParts * cols * kFusedKC * 2 <= kPackBytes, "a chunk past the end of the packed weights");
}

int main(int argc, char** argv)
{
    int n[4], tile_end[4], tiles = 0;
    for (int t = 0; t < 4; ++t) { n[t] = std::atoi(argv[1 + t]); tile_end[t] = tiles += (n[t] + kFusedRows - 1) / kFusedRows; }
    const int grid = tiles < 512 ? tiles : 512;
    int* taken = static_cast<int*>(std::calloc(tiles, sizeof(int)));
    for (int b = 0; b < grid; ++b) {
        for (FusedTile at = fused_tile(tile_end, b);;) {
            require(at.type >= 0 && at.type < 4 && at.row0 >= 0 && at.row0 < n[at.type], "a tile outside its type's rows");
            require(at.row0 % kFusedRows == 0 && ++taken[at.tile] == 1, "a tile taken twice");
            const FusedTile next = fused_next(tile_end, at, grid);
            // the next tile's first weights are asked for whether there is one or not
            require(next.type >= 0 && next.type < 4 && next.row0 >= 0 && next.row0 < n[next.type], "a next tile outside its type's rows");
            for (int c = 0; c < kFusedK1 / kFusedKC; ++c) inside(next.type, kPackF1, kFusedN1, kFusedK1, 0, c);
            if (next.tile == at.tile) { require(at.tile + grid >= tiles, "a workgroup that ends too early"); break; }
            at = next;
        }
    }
    for (int i = 0; i < tiles; ++i) require(taken[i] == 1, "a tile that no workgroup takes");
    for (int t = 0; t < 4; ++t) {
        for (int c = 0; c < kFusedN1 / kFusedKC; ++c) inside(t, kPackF2, kFusedN2, kFusedN1, 0, c);
        for (int c = 0; c < kFusedN2 / kFusedKC; ++c) inside(t, kPackF3, kFusedN3, kFusedN2, 0, c);
        for (int ct = 0; ct < 3; ++ct)
            for (int c = 0; c < kFusedN1 / kFusedKC; ++c) inside(t, kPackB1, 128, kFusedN1, ct, c);
        for (int c = 0; c < kFusedN2 / kFusedKC; ++c) inside(t, kPackB2, kFusedN1, kFusedN2, 0, c);
        for (int c = 0; c < kFusedN3 / kFusedKC; ++c) inside(t, kPackB3, kFusedN2, kFusedN3, 0, c);
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host compiler")
    at = tmp_path_factory.mktemp("fused_tiles")
    (at / "tiles.cpp").write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", str(at / "tiles"), str(at / "tiles.cpp")], check=True)
    return str(at / "tiles")


@pytest.mark.parametrize("rows", [(1, 0, 0, 0), (0, 0, 0, 1), (0, 5, 0, 64), (65, 64, 63, 1), (64 * 512, 0, 1, 0), (0, 64 * 511, 0, 65),
                                  (64 * 700 + 5, 1, 0, 64 * 400 + 33), (400000, 260000, 60000, 47292)])
def test_what_is_asked_for_ahead_lies_in_the_buffers(program, rows):
    got = subprocess.run([program, *map(str, rows)], stdout=subprocess.PIPE, text=True)
    assert got.returncode == 0, got.stdout
