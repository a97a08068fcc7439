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

PITCH = r"""
#include <cstdio>
#include <initializer_list>
#include "tile_index.hpp"
// Q5_K and Q8_0 rows of up to 16 super-blocks: the same offset of 16 rows in
// 16 different slots of a bank round, and the image in its 16 rows + 32 slots
int main() {
    for (uint32_t block : {176u, 272u})
        for (uint32_t nsb = 1; nsb <= 16; nsb++) {
            const uint32_t rb = block * nsb, pitch = vb::rows_pitch(rb);
            uint32_t banks = 0;
            for (uint32_t j = 0; j < 16; j++) banks |= 1u << (j * pitch / 16 % 16);
            if (pitch % 16 != 0 || pitch < rb || banks != 0xFFFFu || 16 * pitch > 16 * (16 * block + 32) - 16) {
                std::printf("rows of %u bytes: pitch %u\n", rb, pitch);
                return 1;
            }
        }
    return 0;
}
"""

RULE = r"""
#include <cstdio>
#include <initializer_list>
#include "tile_index.hpp"
// calls that ran slower on the row-streaming kernel stay off it, calls that
// gained stay on it
struct Call { bool q5k, q8; int64_t n, k; bool on; };
int main() {
    for (Call c : {Call{true, false, 8192, 2560, false}, Call{true, false, 4096, 3584, false},
                   Call{true, false, 2048, 3072, false}, Call{true, false, 8192, 3072, false},
                   Call{false, true, 14336, 1536, false}, Call{false, true, 12606, 1792, false},
                   Call{false, false, 128256, 4096, true}, Call{false, true, 14336, 4096, true},
                   Call{true, false, 2048, 4096, true}, Call{true, false, 14336, 3072, true},
                   Call{false, false, 10240, 2048, true}, Call{false, true, 24576, 1536, true}})
        if (vb::rows_lead(c.q5k, c.q8, c.n, c.k) != c.on) {
            std::printf("%lld x %lld\n", (long long)c.n, (long long)c.k);
            return 1;
        }
    return 0;
}
"""

MOE = r"""
#include <cstdio>
#include <initializer_list>
#include "tile_index.hpp"
static uint32_t rnd = 1;
static int next(int n) { rnd = rnd * 1664525u + 1013904223u; return int((rnd >> 8) % uint32_t(n)); }
// Slot counts of a routing (sum <= nslots): every tile is accepted, the tiles
// cover the experts' blocks once and number at most moe_wreg_tiles.  Counts
// each within [0, nslots] but of any sum, as overwritten lists can hold:
// every accepted tile stays below moe_wreg_blocks.
int main() {
    // the rows fit from 16 slots per expert (where moe_wreg_leads begins), not
    // from 14 (15 n_exp rows of padding)
    for (int e = 1; e <= 64; e++)
        for (int n = 1; n <= 1024; n++) {
            const bool fits = vb::moe_wreg_fits(n, e);
            if ((n >= 16 * e && !fits) || (n % 16 == 0 && n <= 14 * e && fits)) return 5;
            if (fits && 16 * vb::moe_wreg_blocks(n, e) > 2 * n) return 6;
        }
    for (int rep = 0; rep < 20000; rep++) {
        const int n_exp = 1 + next(64), nslots = 1 + next(1024), cap = vb::moe_wreg_blocks(nslots, n_exp);
        const bool wild = rep & 1;
        int count[64], left = nslots, first = 0, tiles = 0;
        for (int e = 0; e < n_exp; e++) {
            count[e] = wild ? next(nslots + 1) : (e + 1 < n_exp ? next(left + 1) >> next(4) : left);
            if (!wild) left -= count[e];
        }
        for (int mb : {1, 10, 16}) {
            first = tiles = 0;
            for (int e = 0; e < n_exp; e++) {
                const int nb = (count[e] + 15) / 16, nt = (nb + mb - 1) / mb;
                int blocks = 0, slots = 0;
                for (int ti = 0; ti < nt; ti++) {
                    vb::MoeTile t{};
                    const bool ok = vb::moe_wreg_tile(e, ti, count[e], first, mb, cap, t);
                    if (ok && (t.blk0 < 0 || t.nblk < 1 || t.nblk > mb || t.blk0 + t.nblk > cap)) {
                        std::printf("experts %d slots %d: tile at %d + %d of %d\n", n_exp, nslots, t.blk0, t.nblk, cap);
                        return 1;
                    }
                    if (!wild && (!ok || t.blk0 != first + blocks || t.m0 != 16 * blocks)) return 2;
                    blocks += t.nblk;
                    slots += t.cnt;
                }
                if (!wild && (blocks != nb || slots != count[e])) return 3;
                first += nb;
                tiles += nt;
            }
            if (!wild && tiles > (mb == 1 ? cap : vb::moe_wreg_tiles(nslots, n_exp, mb))) return 4;
        }
    }
    return 0;
}
"""

MOE_RULE = r"""
#include <cstdio>
#include <initializer_list>
#include "tile_index.hpp"
// MoE calls that ran slower on the prefill kernels stay off them
struct Call { bool gu, dn; int64_t t, topk, e, h; bool on; };
int main() {
    for (Call c : {Call{true, true, 16, 8, 8, 4096, false}, Call{true, false, 16, 8, 8, 2048, false},
                   Call{true, true, 32, 4, 8, 4096, false}, Call{true, true, 34, 4, 8, 4096, false},
                   Call{true, true, 36, 4, 8, 4096, true}, Call{true, false, 64, 2, 8, 4096, true},
                   Call{false, false, 16, 8, 8, 4096, true}, Call{true, false, 500, 2, 8, 4096, true},
                   Call{false, true, 15, 8, 8, 4096, false}, Call{true, false, 64, 1, 4, 2048, false},
                   Call{true, false, 128, 1, 4, 2048, true}, Call{true, true, 16, 2, 8, 4096, false}})
        if (vb::moe_wreg_leads(c.gu, c.dn, c.t, c.topk, c.e, c.h) != c.on) {
            std::printf("%lld tokens, top-%lld of %lld\n", (long long)c.t, (long long)c.topk, (long long)c.e);
            return 1;
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


def test_rows_image_spreads_over_banks(tmp_path):
    """Row images of gemm_rows.hip: no two rows of a read on the same banks."""
    _run(tmp_path, PITCH)


def test_rows_rule(tmp_path):
    """Which calls gemm_rows.hip takes: none of those that lost time on it."""
    _run(tmp_path, RULE)


def test_moe_tiles_stay_inside(tmp_path):
    """Expert tiles of moe_wreg.hip: any routing's tiles are all there, and
    none of overwritten lists lies past the packed blocks."""
    _run(tmp_path, MOE)


def test_moe_rule(tmp_path):
    """Which calls moe_wreg.hip takes: none of those that lost time on it."""
    _run(tmp_path, MOE_RULE)
