// The order in which work groups take the tiles of a matmul: every tile once, and no XCD with more than an eighth of them
// rounded up (ids are dealt round-robin to the 8 XCDs).
#include <cstdio>
#include <vector>

#include "../../oxillama_amd/csrc/oxq_tile_order.hpp"

int main() {
    int failed = 0, grids = 0;
    for (uint32_t m = 1; m <= 40; m++)
        for (uint32_t n = 1; n <= 260; n += n < 40 ? 1 : 7) {
            const uint32_t grid = oxq::tile_order_grid(m, n), most = (m * n + 7) / 8;
            std::vector<int> taken(m * n, 0);
            uint32_t on_xcd[8] = {0};
            bool ok = grid == 8 * most;
            for (uint32_t b = 0; b < grid; b++) {
                uint32_t mt, nt;
                if (!oxq::tile_order_at(b, grid, m, n, mt, nt)) continue;
                ok = ok && mt < m && nt < n;
                if (!ok) break;
                taken[nt * m + mt]++;
                on_xcd[b & 7]++;
            }
            for (int t : taken) ok = ok && t == 1;
            for (uint32_t x : on_xcd) ok = ok && x <= most;
            grids++;
            if (!ok) {
                std::printf("%u x %u tiles\n", m, n);
                failed++;
            }
        }
    std::printf("%d grids, %d failed\n", grids, failed);
    return failed != 0;
}
