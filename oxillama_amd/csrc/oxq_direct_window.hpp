// Where the direct kernel's weight requests may reach (oxq_gemm_direct.hpp): the descriptor of one row tile's bytes.
// (No HIP header here: a host test walks the requests.)
#pragma once
#include <cstddef>
#include <cstdint>

#include "oxq_tile_order.hpp"

namespace oxq {

struct DirectWindow {
    uint32_t row0;     // the descriptor's first row
    uint32_t records;  // its bytes, to the end of the dword of the matrix's last byte
};
// Row tile `set` * RG + rg of an n-row matrix.  Sets past the last, and a tile past n in the last one: the matrix's last row or two, so
// that what is requested ahead of the end costs little.  Their first row is an even one: rows of 210-byte blocks start off a
// dword in turn, and from such a base the rounding up to a dword would go past the matrix's end.  No branch: behind one the
// compiler moves the fmas of a super-block that was begun before it, and spills the matrix core's results.
OXQ_HOST_DEVICE DirectWindow direct_window(uint32_t set, uint32_t sets, uint32_t rg, uint32_t RG, uint32_t n, uint32_t row_bytes) {
    const uint32_t past = (uint32_t)((int32_t)(sets - 1 - set) >> 31) & 0x7FFFFFFu;
    const uint32_t first = 16 * (set * RG + rg) + past, last = (n - 1) & ~1u, row0 = first < last ? first : last;
    const size_t left = ((size_t)(n - row0) * row_bytes + 3) & ~(size_t)3;
    return DirectWindow{row0, left < 0x7FFFFFFF ? (uint32_t)left : 0x7FFFFFFFu};
}
// Super-block `at` of a row of nb; for a part of k (or the end of one) past the last, whose values are not used, the last one: the offset
// in a row goes to the request's scalar offset, and what the range check makes of one beyond the descriptor's size is
// nowhere written down.
OXQ_HOST_DEVICE uint32_t direct_super_block(uint32_t at, uint32_t nb) { return at < nb ? at : nb - 1; }

}  // namespace oxq
