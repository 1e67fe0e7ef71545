// The lines between the tile kernel's tiles of more than 64 token rows, for launch_tiles, which launches by them (the
// measurements stand there), and for the rules that weigh another kernel against the tile that a call would get.
// groups: expert groups, 1 for a plain matmul.
#pragma once
#include <cstddef>
#include <cstdint>
#include "../../include/oxq.h"

namespace oxq {

inline size_t tile_count(uint32_t rows, uint32_t n, uint32_t tile_tokens, uint32_t tile_rows) {
    return (size_t)((rows + tile_tokens - 1) / tile_tokens) * ((n + tile_rows - 1) / tile_rows);
}
// the f16 scales of a work group's tokens for the whole k in LDS
inline bool tile_scales_fit(uint32_t k, uint32_t tile_tokens) { return (size_t)((k + 255) / 256 * 8) * tile_tokens * 2 <= 128 * 1024; }
// a matrix so narrow that even 128 x 64 tiles leave compute units without one
inline bool tile_narrow(uint32_t rows, uint32_t n, uint32_t k, size_t groups, size_t cus) {
    return rows > 384 && tile_scales_fit(k, 128) && tile_count(rows, n, 128, 64) * groups < cus;
}
// 128-token tiles
inline bool tile_big(uint32_t rows, uint32_t n, uint32_t k, size_t groups, size_t cus) {
    return rows > 384 && tile_scales_fit(k, 128) && !tile_narrow(rows, n, k, groups, cus);
}
// ... of 128 weight rows, for `tiles` of them, not 64
inline bool tile_square(uint32_t type, size_t tiles, uint32_t k, size_t cus) {
    return 2 * tiles >= 3 * cus || (2 * tiles > cus && tiles <= cus && (type != OXQ_TYPE_Q4_K || k >= 8192));
}
// 64 x 128 tiles, of which there are tiles_32nds / 32, and not 64 x 32 ones with k split: the line in 32nds per compute unit
constexpr uint32_t TILE_MID_WIDE_LINE = 56;
inline bool tile_mid_wide(size_t tiles_32nds, size_t cus, uint32_t line = TILE_MID_WIDE_LINE) { return tiles_32nds >= line * cus; }

}  // namespace oxq
