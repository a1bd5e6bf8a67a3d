"""The order in which quantizers with a transposed copy deal their tiles out to the XCDs, compiled for the host: every tile once, and up to 1280 tiles,
where patches gather nothing and cost the block-scaled copies up to 4 %, each workgroup its own."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mdy_triton_amd", "csrc")
PROGRAM = r"""
#include "common.h"
#include <cstdio>
#include <cstdlib>
#include <vector>

int main(int argc, char** argv) {
    for (int a = 1; a + 1 < argc; a += 2) {
        const int cols = std::atoi(argv[a]), rows = std::atoi(argv[a + 1]);
        std::vector<int> seen((size_t)cols * rows);
        bool plain = true, once = true;
        for (int r = 0; r < rows; ++r)
            for (int c = 0; c < cols; ++c) {
                int row = r, col = c;
                mdy::xcd_patch(row, col, cols, rows);
                plain = plain && row == r && col == c;
                once = once && row >= 0 && row < rows && col >= 0 && col < cols && ++seen[(size_t)row * cols + col] == 1;
            }
        std::printf("%d %d\n", plain, once);
    }
}
"""
# columns x rows of tiles and whether their order changes (an eighth of 8 columns is one: plain order)
CASES = [((1, 1), False), ((32, 32), False), ((32, 40), False), ((40, 32), False), ((16, 80), False), ((160, 8), False), ((8, 160), False), ((1280, 1), False),
         ((183, 7), False), ((1300, 1), False), ((1, 2000), False), ((161, 8), True), ((8, 161), False), ((9, 161), True), ((143, 9), True), ((59, 22), True), ((427, 3), False),
         ((61, 21), True), ((32, 42), True), ((56, 64), True), ((7, 1001), True)]


def test_every_tile_once_and_in_patches_beyond_1280_tiles(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "order.hip", tmp_path / "order"
    src.write_text(PROGRAM)
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", CSRC, "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe), *[str(v) for size, _ in CASES for v in size]], check=True, capture_output=True, text=True).stdout.split("\n")
    for (size, patches), line in zip(CASES, out):
        assert line == "%d 1" % (not patches), (size, line)
