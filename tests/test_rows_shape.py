"""The host-only rules of the multi-row dispatch on 256 CUs: the block shapes of the row-tiled GEMM's GPU cases are
the ones the launcher picks, with all shapes among them, and linears and norms go to the kernel or block that
measured faster. rows_shape.h is compiled here as it stands."""

import os
import shutil
import subprocess

import pytest

from test_rows_gemm import SHAPES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "haskell-infer-demo_amd", "csrc")

MAIN = """
#include <cstdio>
#include <cstdlib>
#include "rows_shape.h"
int main(int argc, char **argv) {
    for (int i = 1; i + 2 < argc; i += 3) {
        const auto &s = w4a16::kRowsShapes[w4a16::rows_shape(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), 256)];
        std::printf("%d %d %d %d %d %d\\n", s.rows, s.tile_pairs, s.groups,
                    (int)w4a16::rows_streams(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), 256),
                    w4a16::rows_slices(atoi(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), 256),
                    w4a16::rmsnorm_chunks(atoi(argv[i + 1]), atoi(argv[i]), 256));
    }
    std::printf("%d\\n", (int)(sizeof(w4a16::kRowsShapes) / sizeof(w4a16::kRowsShapes[0])));
}
"""

# row tiles x tile pairs x groups a step of each of SHAPES, or the tile pairs of its slices of 16 rows
PICKED = [1, (1, 1, 16), (1, 1, 16), 1, (1, 2, 8), 2, (1, 3, 8), (1, 4, 4), 4, (1, 6, 4), (1, 8, 4),
          4, (1, 10, 2), (2, 4, 4), (2, 6, 4), (2, 9, 4), (2, 10, 2), (2, 6, 2), (4, 10, 2), 1, 1, 2, 4, 4]


@pytest.fixture(scope="module")
def picked(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("shape")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", "-o", str(d / "shape"), str(d / "main.cpp")], check=True)

    def ask(sizes):
        argv = [str(v) for size in sizes for v in size]
        lines = subprocess.run([str(d / "shape"), *argv], check=True, capture_output=True, text=True).stdout.split("\n")
        return [tuple(map(int, line.split())) for line in lines[:len(sizes)]], int(lines[len(sizes)])

    return ask


def test_shapes_of_the_gpu_cases(picked):
    shapes, count = picked(SHAPES)
    assert [m > 16 and s[4] or s[:3] for (m, _, _), s in zip(SHAPES, shapes)] == PICKED
    assert len({p for p in PICKED if not isinstance(p, int)}) == count


def test_few_rows_and_more_share_their_groups_a_step(picked):
    shapes, _ = picked([(16, 28672, 8192), (17, 28672, 8192), (11, 14344, 8192), (24, 14344, 8192)])
    assert [s[2] for s in shapes] == [4, 4, 4, 4]


@pytest.mark.parametrize("m,n,k,streams", [
    (2, 5120, 12288, False), (2, 5120, 17408, True), (3, 5120, 10752, True), (3, 5120, 9728, False),
    (4, 5120, 8704, False), (4, 5120, 9728, True), (4, 9728, 8704, True),
    (5, 4224, 5248, False), (5, 8192, 6144, False), (5, 9728, 5248, True), (5, 4224, 8192, True),
    (6, 5120, 5248, False), (6, 5120, 6144, True), (7, 4224, 5248, True), (8, 4104, 5248, True),
    (5, 4104, 7168, False), (4, 4104, 8704, False), (5, 4104, 8192, True), (7, 4104, 5248, False),
    (8, 4096, 17408, False), (8, 5120, 5120, False),
])
def test_few_rows_route(picked, m, n, k, streams):
    assert picked([(m, n, k)])[0][0][3] == streams


@pytest.mark.parametrize("m,n,k,tile_pairs", [
    (24, 1024, 1024, 1), (24, 1024, 1536, 1), (24, 1024, 1664, 0), (24, 1024, 2048, 0), (24, 1024, 2560, 1),
    (24, 1024, 3840, 1), (24, 1024, 3968, 0), (64, 1024, 2560, 1), (65, 1024, 2560, 2), (128, 1024, 2560, 2),
    (128, 1024, 1024, 0), (128, 1024, 640, 2), (24, 2560, 3712, 0), (128, 2048, 3200, 4), (80, 2048, 3200, 0),
    (128, 4096, 2560, 0), (128, 128, 128, 1), (100000, 128, 128, 0),
])
def test_slices_route(picked, m, n, k, tile_pairs):
    assert picked([(m, n, k)])[0][0][4] == tile_pairs


@pytest.mark.parametrize("rows,cols,chunks", [
    (1, 5120, 1), (384, 5120, 1), (385, 5120, 2), (16384, 4096, 1), (16384, 4104, 2), (385, 8192, 2), (1, 8200, 2),
])
def test_rmsnorm_block(picked, rows, cols, chunks):
    assert picked([(rows, cols, 128)])[0][0][5] == chunks
