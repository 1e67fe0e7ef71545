// The descriptors of the direct kernel's weight requests, those past the last row tile among them: on a dword, with the tile's rows in
// them, and not a byte behind the dword in which the matrix ends; every scalar offset, also of parts of k past the last super-block, in them.
#include <cstdio>
#include <initializer_list>

#include "../../oxillama_amd/csrc/oxq_direct_window.hpp"

int main() {
    int failed = 0, windows = 0;
    for (uint32_t block : {136u, 144u, 176u, 210u, 272u})
        for (uint32_t nb = 2; nb <= 18; nb++)
            for (uint32_t n = 1; n <= 130; n++)
                for (uint32_t RG : {1u, 2u})
                    for (uint32_t step : {1u, 3u}) {
                        const uint32_t row_bytes = nb * block, sets = ((n + 15) / 16 + RG - 1) / RG;
                        const size_t end = (size_t)n * row_bytes, last_dword = (end + 3) & ~(size_t)3;
                        for (uint32_t set = 0; set < sets + 2 * step; set++)  // two row tiles of weights are in flight
                            for (uint32_t rg = 0; rg < RG; rg++) {
                                const oxq::DirectWindow w = oxq::direct_window(set, sets, rg, RG, n, row_bytes);
                                const size_t base = (size_t)w.row0 * row_bytes;
                                const uint32_t row = 16 * (set * RG + rg);
                                bool ok = base % 4 == 0 && base + w.records <= last_dword && w.records >= row_bytes;
                                if (set < sets && row < n) {
                                    const size_t tile_end = (size_t)(row + 16 < n ? row + 16 : n) * row_bytes;
                                    ok = ok && w.row0 == row && base + w.records >= tile_end;
                                }
                                for (uint32_t parts : {4u, 8u, 16u})  // of one super-block, eight also of two
                                    for (uint32_t at = 0; at < (parts == 8 ? 16 : parts); at++)
                                        ok = ok && (oxq::direct_super_block(at, nb) + 1) * block <= w.records &&
                                             (at >= nb || oxq::direct_super_block(at, nb) == at);
                                windows++;
                                if (!ok && failed++ < 10)
                                    std::printf("block %u x %u, n %u, set %u of %u, tile %u of %u: row %u, %u bytes\n", block, nb, n, set,
                                                sets, rg, RG, w.row0, w.records);
                            }
                    }
    std::printf("%d windows, %d failed\n", windows, failed);
    return failed != 0;
}
