"""Which elements of the reduction the lanes of the packed matrix-vector kernel take, and under how many scales they lie, for
every size and block size that it is given."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "transformers-qwen3-moe-fused_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "gemv_layout.h"
int main() {
    int wrong = 0;
    for (int K = 320; K <= 2048; K += 64)
        for (int at = 0; at < 4 * 6; ++at) {
            const int N = 32 << at % 4, bs_shift = 3 + at / 4;
            const mfl::GemvLayout l = mfl::gemv_layout(K, N, bs_shift);
            std::vector<int> taken(K);
            bool whole = true;  // a lane's dwords are inside the row together or not at all where they lie side by side
            for (int lane = 0; lane < l.lanes; ++lane)
                for (int i = 0; i < l.dwords; ++i) {
                    const int k = l.side_by_side ? (lane * l.dwords + i) * 8 : (i * l.lanes + lane) * 8;
                    if (l.side_by_side && (lane * l.dwords * 8 < K) != (k < K)) whole = false;
                    for (int u = 0; u < 8 && k < K; ++u) ++taken[k + u];
                }
            // side by side, the kernel loads one scale for a lane's four dwords and two for six, of which the second is that of
            // the dwords past a multiple of 64
            if (l.side_by_side)
                for (int lane = 0; lane < l.lanes; ++lane)
                    for (int k = lane * l.dwords * 8, first = k; k < first + l.dwords * 8; ++k) {
                        const int loaded = l.dwords == 6 && (k ^ first) >> 6 != 0 ? first + 40 : first;
                        if (k < K && k >> bs_shift != loaded >> bs_shift) whole = false;
                    }
            bool ok = whole && l.reach() >= K;
            for (int t : taken) ok = ok && t == 1;
            // with the dwords of a short reduction apart, past a row per expert the streaming kernel takes what it can, and the
            // register-decoding one the shortest
            const int half_rows = mfl::gemv_half_rows(K, l, bs_shift);
            const bool left = K <= 1024 && ((K % 128 == 0 && bs_shift >= 6 && (K == 384 || !l.side_by_side)) ||
                                            (K < 512 && bs_shift >= 5 && !l.side_by_side));
            ok = ok && half_rows == (K > 1024 ? 4 : left ? 2 : 3);
            if (!ok && wrong++ < 8) std::printf("K = %d, N = %d, blocks of %d: %d lanes of %d dwords\n", K, N, 1 << bs_shift, l.lanes, l.dwords);
        }
    return wrong ? 1 : 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_every_element_of_a_reduction_is_taken_once_and_under_its_scale(tmp_path):
    src, exe = tmp_path / "gemv_layout.cpp", tmp_path / "gemv_layout"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
