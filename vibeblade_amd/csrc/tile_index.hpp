// Index arithmetic that decides which addresses a kernel touches, in plain
// C++ (constexpr: host and device): tests/test_tile_index.py compiles this
// header alone for the CPU and sweeps it.
#pragma once

#include <cstdint>

namespace vb {

// ---- weight rows in groups of 16 (gemm_rows.hip) ---------------------------------

constexpr uint32_t ROWS_NONE = 0x80000000u;  // lane offset past every tensor (below 2 GiB): reads zeros, no traffic

// Byte offset of 16-byte slot `slot` of the rows 16 grp .. + 15 (rb bytes
// each).  The whole offset is the lane's: a buffer load compares its lane
// offset with the tensor's size and is documented to leave the uniform offset
// out of that, so with the group's start there the rows past N of a ragged
// last group were fetched from behind the tensor.
constexpr uint32_t rows_fetch_at(int grp, int ngroups, uint32_t slot, uint32_t rb) {
    return grp < ngroups && slot < rb ? (static_cast<uint32_t>(grp) * rb + slot) * 16u : ROWS_NONE;
}

// Bytes from one row to the next in the LDS image, for rows of whole 16-byte
// slots.  The 16 rows that a read touches at the same offset fall on distinct
// banks when a row is an odd number of slots (64 banks of 4 bytes: 16 slots a
// round); a row of an even number gets one more.
constexpr uint32_t rows_pitch(uint32_t rb) { return rb | 16u; }

// ---- expert tiles (moe_wreg.hip) -------------------------------------------------

// Most 16-row blocks, and most tiles of up to `mb_max` blocks, that any
// routing of `nslots` slots over `n_exp` experts makes: every expert with
// slots may leave one partly filled.
constexpr int moe_wreg_blocks(int nslots, int n_exp) { return nslots / 16 + (n_exp < nslots ? n_exp : nslots); }
constexpr int moe_wreg_tiles(int nslots, int n_exp, int mb_max) {
    return nslots / (16 * mb_max) + (n_exp < nslots ? n_exp : nslots);
}

// Whether the blocks' fp16 rows fit where moe_ws (moe.hip) lays fp32 rows of
// the slots: packed activations in obuf, hidden rows in hbuf.
constexpr bool moe_wreg_fits(int nslots, int n_exp) {
    return 16 * moe_wreg_blocks(nslots, n_exp) * 2 <= nslots * 4;
}

struct MoeTile {
    int e;        // expert
    int blk0;     // first packed block (of all experts' blocks)
    int nblk;     // blocks, 1 .. mb_max
    int m0, cnt;  // first of the expert's slots, slots in the tile
};

// Tile `ti` of expert e with `slots` slots, whose blocks start at `first` of
// all experts' and fill tiles of up to mb_max blocks (equal sizes).  False if
// the tile's blocks do not all lie below `cap`: never so for lists the
// routing wrote, but lists that another stream overwrote can claim more slots
// than there are, and the packed and hidden rows hold `cap` blocks.
constexpr bool moe_wreg_tile(int e, int ti, int slots, int first, int mb_max, int cap, MoeTile& t) {
    const int nb = (slots + 15) / 16, nt = (nb + mb_max - 1) / mb_max, bpt = (nb + nt - 1) / nt, bb = ti * bpt;
    t.e = e;
    t.blk0 = first + bb;
    t.nblk = nb - bb < bpt ? nb - bb : bpt;
    t.m0 = 16 * bb;
    t.cnt = slots - t.m0 < 16 * t.nblk ? slots - t.m0 : 16 * t.nblk;
    return t.nblk > 0 && t.blk0 + t.nblk <= cap;
}

}  // namespace vb
