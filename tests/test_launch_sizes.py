"""The pieces of a one-dimensional launch (csrc/vx_launch.hpp), compiled for the
host: every launch holds fewer than 2^32 threads and the pieces cover all blocks
once, up to the largest volume that vx_volume_create takes (4096 x 4096 x 2040
texels)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "voxelengine_amd", "csrc")

SRC = r'''
#include <cstdio>
#include <cstdlib>
#include "vx_launch.hpp"
int main(int, char** a) {
    const long long sx = atoll(a[1]), sy = atoll(a[2]), sz = atoll(a[3]);
    const size_t bricks = (size_t)(sx / 4 + 1) * (sy / 4 + 1) * (sz / 4 + 1);
    const size_t grid = (size_t)(((2 * sx + 2) >> 2) + 2) * (((2 * sy + 2) >> 2) + 2) * (((2 * sz + 2) >> 2) + 2);
    const uint64_t blocks = vx::clear_blocks(8 * bricks) + vx::clear_blocks(bricks) + vx::clear_grid_blocks(grid);
    std::printf("%llu\n", (unsigned long long)blocks);
    vx::launch_pieces(blocks, [](uint32_t first, uint32_t count) { std::printf("%u %u\n", first, count); return true; });
    unsigned calls = 0;
    const bool all = vx::launch_pieces(3 * vx::kMaxBlocks256, [&](uint32_t, uint32_t) { return ++calls < 2; });
    std::printf("%u %d\n", calls, (int)all);
}
'''


@pytest.fixture(scope="module")
def pieces(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("launch")
    (d / "p.cpp").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "p.cpp"), "-o", str(d / "p")], check=True)

    def run(dims):
        lines = subprocess.run([str(d / "p"), *map(str, dims)], check=True, capture_output=True, text=True).stdout.split("\n")
        rows = [tuple(map(int, l.split())) for l in lines if l]
        return rows[0][0], rows[1:-1], rows[-1]
    return run


@pytest.mark.parametrize("dims,launches", [((1, 1, 1), 1), ((256, 256, 256), 1), ((1024, 1024, 1024), 1),
                                           ((4096, 4096, 1250), 1), ((4096, 4096, 1400), 2), ((4096, 4096, 2040), 2)])
def test_clear_launches_hold_fewer_than_2_to_32_threads(pieces, dims, launches):
    blocks, got, stopped = pieces(dims)
    assert len(got) == launches
    at = 0
    for first, count in got:
        assert first == at and count > 0 and count * 256 < 2 ** 32
        at += count
    assert at == blocks
    # and a launch that fails ends the sequence
    assert stopped == (2, 0)
