// The order in which work groups take the tiles of a matmul: every tile once, and no XCD with more than an eighth of them
// rounded up (ids are dealt round-robin to the 8 XCDs).  The even deal of (tile, part of k) units: every unit in one run, runs
// that differ by one unit, and the sums of a shared tile where the kernel that adds them looks.
#include <cstdio>
#include <vector>

#include "../../oxillama_amd/csrc/oxq_tile_order.hpp"

int main() {
    int failed = 0, grids = 0;
    for (uint32_t m = 1; m <= 40; m++)
        for (uint32_t n = 1; n <= 260; n += n < 40 ? 1 : 7) {
            const uint32_t grid = oxq::tile_order_grid(m, n), most = (m * n + 7) / 8;
            std::vector<int> taken(m * n, 0), in_run(m * n, 0);
            uint32_t on_xcd[8] = {0};
            bool ok = grid == 8 * most;
            for (uint32_t b = 0; b < grid; b++) {
                uint32_t mt, nt;
                if (oxq::tile_run_at(b, grid, m, n, mt, nt)) {  // (an XCD's work groups: `most` at most)
                    ok = ok && mt < m && nt < n;
                    if (!ok) break;
                    in_run[nt * m + mt]++;
                }
                if (!oxq::tile_order_at(b, grid, m, n, mt, nt)) continue;
                ok = ok && mt < m && nt < n;
                if (!ok) break;
                taken[nt * m + mt]++;
                on_xcd[b & 7]++;
            }
            for (int t : taken) ok = ok && t == 1;
            for (int t : in_run) ok = ok && t == 1;
            for (uint32_t x : on_xcd) ok = ok && x <= most;
            const oxq::TileGrid g = oxq::tile_order_grid3(m, n);  // (x fastest, a multiple of 8: the XCD is x % 8)
            uint32_t on3[8] = {0};
            ok = ok && g.x == 8 * m;
            for (uint32_t s = 0; ok && s < g.y * g.z; s++)
                for (uint32_t x = 0; x < g.x; x++) {
                    uint32_t mt, nt;
                    if (!oxq::tile_order_at3(x, s, m, n, mt, nt)) continue;
                    ok = ok && mt < m && nt < n;
                    if (!ok) break;
                    taken[nt * m + mt]++;
                    on3[x & 7]++;
                }
            for (int t : taken) ok = ok && t == 2;
            for (uint32_t x : on3) ok = ok && x <= most;
            if (m > 1) {  // the last token tile's behind all others; an XCD at most one of them above its share
                const oxq::TileGrid l = oxq::tile_order_grid3_short_last(m, n);
                uint32_t on_last[8] = {0};
                bool last = false;
                ok = ok && l.x == 8 * (m - 1);
                for (uint32_t s = 0; ok && s < l.y * l.z; s++)
                    for (uint32_t x = 0; x < l.x; x++) {
                        uint32_t mt, nt;
                        if (!oxq::tile_order_at3_short_last(x, s, m, n, mt, nt)) continue;
                        last = last || mt == m - 1;
                        ok = ok && mt < m && nt < n && (mt == m - 1) == last;
                        if (!ok) break;
                        taken[nt * m + mt]++;
                        on_last[x & 7]++;
                    }
                for (int t : taken) ok = ok && t == 3;
                for (uint32_t x : on_last) ok = ok && x <= most + 1;
            }
            grids++;
            if (!ok) {
                std::printf("%u x %u tiles\n", m, n);
                failed++;
            }
        }
    int deals = 0;
    for (uint32_t groups : {8u, 240u, 256u})
        for (uint32_t per_tile : {1u, 3u, 16u, 43u, 56u})
            for (uint32_t tiles = 1; tiles <= 700; tiles += tiles < 20 ? 1 : 13) {
                const uint32_t units = tiles * per_tile;
                std::vector<uint32_t> rank_of(units, ~0u), slot_of(units, ~0u);  // slot: 2 * groups for a tile of one's own
                std::vector<int> ranks(groups, 0);
                bool ok = true;
                for (uint32_t b = 0; b < groups; b++) {  // as the kernel walks them
                    const uint32_t rank = oxq::deal_rank(b, groups);
                    ok = ok && rank < groups && ranks[rank]++ == 0;
                    const oxq::DealRange r = oxq::deal_range(rank, groups, units);
                    ok = ok && r.end <= units && r.end - r.begin <= (units + groups - 1) / groups;
                    uint32_t slot = 2 * rank;
                    for (uint32_t u = r.begin; ok && u < r.end;) {
                        const uint32_t lo = u % per_tile, left = r.end - u, hi = lo + left < per_tile ? lo + left : per_tile;
                        for (uint32_t i = 0; i < hi - lo; i++) {
                            ok = ok && rank_of[u + i] == ~0u;
                            rank_of[u + i] = rank;
                            slot_of[u + i] = hi - lo == per_tile ? 2 * groups : slot;
                        }
                        if (hi - lo != per_tile)  // no slot twice
                            ok = ok && (slot == 2 * rank || u != r.begin) && (u == r.begin || u + (hi - lo) == r.end);
                        slot |= 1;
                        u += hi - lo;
                    }
                }
                for (uint32_t u = 0; ok && u < units; u++) {
                    const uint32_t begin = u / per_tile * per_tile, owner = oxq::deal_owner(u, groups, units);
                    const bool shared = oxq::deal_owner(begin, groups, units) != oxq::deal_owner(begin + per_tile - 1, groups, units);
                    ok = owner == rank_of[u] && slot_of[u] == (shared ? oxq::deal_slot(owner, begin, groups, units) : 2 * groups);
                }
                // whole rounds of tiles before the runs: every tile once, as a work group's own or by units of its runs
                const uint32_t own = tiles / groups, tile0 = own * groups, rest = (tiles - tile0) * per_tile;
                std::vector<uint32_t> had(tiles, 0);
                for (uint32_t b = 0; ok && b < groups; b++) {
                    const uint32_t rank = oxq::deal_rank(b, groups);
                    const oxq::DealRange r = oxq::deal_range(rank, groups, rest);
                    for (uint32_t i = 0; i < own; i++) had[rank * own + i] += per_tile;
                    for (uint32_t u = r.begin; u < r.end; u++) had[tile0 + u / per_tile]++;
                }
                for (uint32_t h : had) ok = ok && h == per_tile;
                deals++;
                if (!ok) {
                    std::printf("%u tiles of %u units to %u work groups\n", tiles, per_tile, groups);
                    failed++;
                }
            }
    std::printf("%d grids, %d deals, %d failed\n", grids, deals, failed);
    return failed != 0;
}
