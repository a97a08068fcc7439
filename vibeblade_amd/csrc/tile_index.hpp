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

}  // namespace vb
