// Which tile of m_tiles x n_tiles a work group takes, by its number: ids are dealt round-robin to the 8 XCDs, and the
// token tiles of one set of weight rows sit next to each other on one XCD, so that their weight reads meet in its L2.  Sets of
// weight rows go to the XCDs in turn while there are eight left; the tiles of the last few sets are dealt out in eighths.
// No XCD has more than an eighth of all tiles, rounded up: a grid of as many tiles as there are compute units is one round
// of the chip whatever its sides (whole sets to the end instead, 36 sets of 7 token tiles gave four XCDs 35 work groups for
// 32 compute units: 448 x 4608 x 4096, Q4_K, 74 us against 40; 1480 x 4608 x 4608 218 against 130 on the prefill kernel, 1073 x
// 3328 x 8192, IQ4_XS, 192 against 137 on the tile kernel).
// (No HIP header here: a host test walks the grids.)
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define OXQ_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define OXQ_HOST_DEVICE inline
#endif

namespace oxq {

OXQ_HOST_DEVICE uint32_t tile_order_grid(uint32_t m_tiles, uint32_t n_tiles) { return (m_tiles * n_tiles + 7) / 8 * 8; }

// false: no tile left for this work group
OXQ_HOST_DEVICE bool tile_order_at(uint32_t block, uint32_t grid, uint32_t m_tiles, uint32_t n_tiles, uint32_t &m_tile, uint32_t &n_tile) {
    const uint32_t xcd = block & 7, at = block >> 3, set = at / m_tiles, sets = n_tiles / 8;
    if (set < sets) {
        n_tile = set * 8 + xcd;
        m_tile = at - set * m_tiles;
        return true;
    }
    const uint32_t t = xcd * ((grid >> 3) - sets * m_tiles) + (at - sets * m_tiles);
    n_tile = t / m_tiles;
    m_tile = t - n_tile * m_tiles;
    n_tile += sets * 8;
    return n_tile < n_tiles;
}

// The f16 kernel's order on the same grid: runs of an eighth of the tiles to each XCD, the token tiles of one set of weight rows next
// to each other.  One division, where the order above takes two and a branch, which its small shape shows (114 matmuls with 130 to
// 2048 rows, in the mean: Q5_K 1.6 % over the runs, Q4_K and Q6_K 0.5 %, the large shape 0.2 %; Q5_K 2048 x 8960 x 1536 177.6 us
// against 170.8).
OXQ_HOST_DEVICE bool tile_run_at(uint32_t block, uint32_t grid, uint32_t m_tiles, uint32_t n_tiles, uint32_t &m_tile, uint32_t &n_tile) {
    const uint32_t t = (block & 7) * (grid >> 3) + (block >> 3);
    n_tile = t / m_tiles;
    m_tile = t - n_tile * m_tiles;
    return n_tile < n_tiles;
}

// The same order as the first for a grid of (8 x m_tiles, sets of eight n_tiles and the tail, more of them) work groups, whose coordinates
// spare the kernel the division: for short work groups.
struct TileGrid {
    uint32_t x, y, z;
};
OXQ_HOST_DEVICE TileGrid tile_order_grid3(uint32_t m_tiles, uint32_t n_tiles) {
    const uint32_t sets = (n_tiles + 7) / 8, y = sets < 32768 ? sets : 32768;
    return TileGrid{8 * m_tiles, y, (sets + y - 1) / y};
}
OXQ_HOST_DEVICE bool tile_order_at3(uint32_t x, uint32_t set, uint32_t m_tiles, uint32_t n_tiles, uint32_t &m_tile, uint32_t &n_tile) {
    m_tile = x >> 3;
    n_tile = set * 8 + (x & 7);
    const uint32_t left = n_tiles - set * 8;  // sets of weight rows from here on
    if (set * 8 < n_tiles && left < 8) {
        const uint32_t per = (left * m_tiles + 7) / 8, t = (x & 7) * per + m_tile;
        if (m_tile >= per) return false;
        m_tile = t % m_tiles;
        n_tile = set * 8 + t / m_tiles;
    }
    return n_tile < n_tiles;
}

// The same with the tiles of the last, shorter token tile behind all others (of several token tiles): a grid of more work groups
// than the chip holds at a time ends on the shorter ones.  Its width tells it from the other grid.
OXQ_HOST_DEVICE TileGrid tile_order_grid3_short_last(uint32_t m_tiles, uint32_t n_tiles) {
    const uint32_t full = m_tiles - 1, sets = (n_tiles + 7) / 8, all = sets + (sets + full - 1) / full;
    const uint32_t y = all < 32768 ? all : 32768;
    return TileGrid{8 * full, y, (all + y - 1) / y};
}
OXQ_HOST_DEVICE bool tile_order_at3_short_last(uint32_t x, uint32_t set, uint32_t m_tiles, uint32_t n_tiles, uint32_t &m_tile, uint32_t &n_tile) {
    const uint32_t full = m_tiles - 1, sets = (n_tiles + 7) / 8;
    if (set < sets) return tile_order_at3(x, set, full, n_tiles, m_tile, n_tile);
    m_tile = full;
    n_tile = ((set - sets) * full + (x >> 3)) * 8 + 7 - (x & 7);  // (from the XCDs to which the last full ones go least)
    return n_tile < n_tiles;
}

// An even deal of units (a unit: one super-block of one tile, the tiles one after another) over as many work groups as there
// are compute units: a work group takes a run of units, so that at most two of the tiles it meets are not all its own, the
// first and the last of its run, and their sums go to its two slots.  Neighbouring runs sit on one XCD.
struct DealRange {
    uint32_t begin, end;
};
OXQ_HOST_DEVICE uint32_t deal_rank(uint32_t block, uint32_t groups) { return (block & 7) * (groups >> 3) + (block >> 3); }
OXQ_HOST_DEVICE DealRange deal_range(uint32_t rank, uint32_t groups, uint32_t units) {
    return DealRange{(uint32_t)((uint64_t)rank * units / groups), (uint32_t)((uint64_t)(rank + 1) * units / groups)};
}
// whose run holds this unit
OXQ_HOST_DEVICE uint32_t deal_owner(uint32_t unit, uint32_t groups, uint32_t units) {
    return (uint32_t)((((uint64_t)unit + 1) * groups - 1) / units);
}
// where work group `rank` leaves its sums of the tile whose first unit is tile_begin
OXQ_HOST_DEVICE uint32_t deal_slot(uint32_t rank, uint32_t tile_begin, uint32_t groups, uint32_t units) {
    return 2 * rank + (deal_range(rank, groups, units).begin < tile_begin ? 1 : 0);
}

}  // namespace oxq
