"""The index arithmetic of csrc/tile_index.hpp, compiled for the CPU: which
bytes the kernels touch, swept over sizes at the edges."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vibeblade_amd", "csrc")

ROWS = r"""
#include <cstdio>
#include <initializer_list>
#include "tile_index.hpp"
// 16-byte loads of every slot of every group, and of two groups past the last
// (the prefetch): a load whose lane offset is at or past the tensor's end
// reads nothing, every other one starts inside it at its own row's bytes
int main() {
    for (uint32_t block : {176u, 210u, 272u})
        for (int nsb = 1; nsb <= 16; nsb++)
            for (int n : {1, 2, 15, 16, 17, 31, 33, 300, 4099}) {
                const uint32_t rb = block * nsb;
                const uint64_t bytes = uint64_t(n) * rb;
                const int groups = (n + 15) / 16;
                uint64_t seen = 0;
                for (int g = 0; g < groups + 2; g++)
                    for (uint32_t slot = 0; slot < 9 * 512; slot++) {
                        const uint32_t at = vb::rows_fetch_at(g, groups, slot, rb);
                        if (at >= bytes) continue;
                        if (g >= groups || slot >= rb || at != (uint64_t(g) * rb + slot) * 16) {
                            std::printf("block %u nsb %d n %d group %d slot %u: offset %u\n", block, nsb, n, g, slot, at);
                            return 1;
                        }
                        seen++;
                    }
                if (seen != (bytes + 15) / 16) {
                    std::printf("block %u nsb %d n %d: %llu slots\n", block, nsb, n, (unsigned long long)seen);
                    return 1;
                }
            }
    return 0;
}
"""


def _run(tmp_path, code):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(code)
    subprocess.run([cxx, "-std=c++17", "-O2", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_rows_fetch_stays_inside(tmp_path):
    """Row groups of gemm_rows.hip: no load behind a ragged last group."""
    _run(tmp_path, ROWS)
