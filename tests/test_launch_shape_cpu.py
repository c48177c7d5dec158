"""The batched launches' shapes (csrc/pgrav_grid.h, compiled for the host): a persistent grid
counts workgroups as asked for, covers every XCD, and no launch exceeds 2^32 - 1 lanes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <initializer_list>
#include "pgrav_grid.h"
using namespace pgrav;
int main() {
    for (int groups : {1, 7, 8, 9, 4095, 4096, 6143, 6144, 10239, 10240, 32767, 32768, 1 << 20, (1 << 24) - 8, (1 << 24) - 7,
                       1 << 24, (1 << 25) - 8, (1 << 25) - 7, 1 << 25, (1 << 26) - 8})
        for (int blocks : {-8192, 1, 8, 9, 256, 2048, 2147483647}) {
            const int waves = 1 << split_log2(groups, 8192);
            printf("%d %d %d %d\\n", groups, blocks, waves, persistent_grid(blocks, groups, waves));
            for (bool fp64 : {false, true}) {
                const int w = 1 << split_log2_ewald(groups, 8192, fp64);
                printf("%d %d %d %d\\n", groups, blocks, w, persistent_grid(blocks, groups, w));
            }
        }
}
"""


def test_launch_shapes(tmp_path):
    (tmp_path / "shape.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "shape")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "ahotsph-2hot-apps_amd", "csrc"), str(tmp_path / "shape.cpp"), "-o", exe],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    rows = [[int(x) for x in line.split()] for line in out.splitlines()]
    assert len(rows) == 20 * 7 * 3
    for i, (groups, blocks, waves, grid) in enumerate(rows):
        asked = 8192 // waves if blocks < 0 else min(blocks, groups)
        assert grid == -(-asked // 8) * 8, (groups, blocks, waves, grid)
        assert max(groups, grid) * 64 * waves < 2 ** 32, (groups, blocks, waves, grid)
        assert waves == [
            16 if groups < 4096 else 8 if groups < 32768 else 4 if groups < 2 ** 24 - 7 else
            2 if groups < 2 ** 25 - 7 else 1,
            8 if groups < 6144 else 4 if groups < 10240 else 2 if groups < 2 ** 25 - 7 else 1,
            8 if groups < 6144 else 1][i % 3]
