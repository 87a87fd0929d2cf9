"""The rule by which a wave of the four-wave product counts its output stores, against the lanes themselves: a store that
is counted but has no lane to store makes the kernel read a stage before its last copy has landed."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "transformers-qwen3-moe-fused_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "store_lanes.h"
int main() {
    int wrong = 0;
    const int widths[] = {8, 12};  // pieces of a row of 64 and of 96 columns
    for (int cpr : widths)
        for (int rows = -40; rows <= 330; ++rows)
            for (int cols = -192; cols <= 192; cols += 8)
                for (int u = 0; u < 32 * cpr / 64; ++u) {
                    bool any = false;
                    for (int q = 64 * u; q < 64 * u + 64; ++q) any |= q / cpr < rows && q % cpr * 8 < cols;
                    if (any != mfl::store_has_lane(u, cpr, rows, cols)) {
                        if (wrong++ < 5) std::printf("store %d of rows of %d pieces, %d rows, %d columns\n", u, cpr, rows, cols);
                    }
                }
    return wrong ? 1 : 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_a_store_is_counted_where_a_lane_stores(tmp_path):
    src, exe = tmp_path / "store_lanes.cpp", tmp_path / "store_lanes"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
