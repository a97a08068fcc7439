// Index arithmetic that decides which addresses a kernel touches, and rules of
// dispatch on sizes alone, in plain C++ (constexpr: host and device): tests/test_tile_index.py compiles this
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

// Where that kernel leads the K-split kernel, at every number of rows from 2 to
// 16 and for both types of X.  MI355X, K-split over row-streaming time, the
// least over those rows at the shapes measured:
//   Q5_K      K = 2048, 4096   other K >= 2048      1024 <= K < 2048
//     N <=  4096     1.15 - 1.18      0.87 - 0.94           -
//     N <=  8192     1.21 - 1.61      0.86 - 1.15           -
//     N <= 16384     1.60 - 1.88      1.00 - 1.30           -
//     above          1.91 - 2.46      1.41 - 1.94      1.20 - 1.64
//   K >= 2048, N 10240 .. 16384 and above: Q6_K 1.09 - 1.59, 1.48 - 2.07; Q8_0
//     1.03 - 1.70, 1.48 - 2.19
//   1536 <= K < 2048: Q6_K 0.98 - 1.19, 1.29 - 1.56; Q8_0 0.92 - 1.12, 1.33 - 1.60
//   1024 <= K < 1536, N >= 24576: Q6_K 1.18 - 1.57, Q8_0 1.08 - 1.33
// (a wave owns an eighth of K in steps of 128, so only multiples of 1024 give
// the waves equal work, and up to N = 8192 a workgroup has two groups at most
// to make up for its first loads)
constexpr bool rows_lead(bool q5k, bool q8, int64_t N, int64_t K) {
    if (K < 1024) return false;
    if (q5k) return K >= 2048 ? N > 8192 || (N >= 2048 && K % 2048 == 0) : N >= 16384;
    return K >= 2048 ? N >= 10240 : (K >= 1536 ? N >= (q8 ? 16385 : 10240) : N >= 24576);
}

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

// Where those kernels lead the 16-slot ones of moe.hip and gemm_kq.hip: they
// decode each weight once per up to 160 slots but cannot fill the chip with a
// small down product (its workgroups take 128 of the h columns of one expert).
// MI355X, Q4_K gate/up and Q6_K down, us there / on the 16-slot kernels, mean
// slots per expert in brackets, top-1 to top-8 and even to skewed routings: 8 experts of 4096 x
// 14336 304 / 307 at [12], 297 - 402 / 367 - 454 [16], 302 - 444 / 452 - 515
// [20], 361 - 385 / 1156 - 1177 [64]; 32 of 2048 x 4096, top-4, 190 / 201 [8],
// 194 / 318 [16], 212 / 510 [31]; 4 of 2048 x 8192 (64 down workgroups) 107 / 76
// [16], 98 - 154 / 111 - 214 [32].  The skinny tiles of Q4_K gate/up decode each
// weight once as well where no expert can have more than 16 slots (top-8 of 8 at
// [16]: 4096 x 14336, Q4_K down, 241 / 203; 2048 x 1536, Q6_K down, 52 / 48),
// and with Q4_K down they lead up to [17] on some routings (252 / 229 at [16],
// 267 / 258 at [17], 255 - 305 / 291 - 342 at [18]).
constexpr bool moe_wreg_leads(bool q4k_gate_up, bool q4k_down, int64_t n_tokens, int64_t topk, int64_t n_exp, int64_t h) {
    const int64_t wgs = n_exp * (h / 128);
    int64_t per = wgs >= 128 ? 16 : (wgs >= 64 ? 32 : 64);
    if (q4k_gate_up && n_tokens <= 16) return false;
    if (q4k_gate_up && q4k_down && per < 18) per = 18;
    return n_tokens * topk >= per * n_exp;
}

}  // namespace vb
