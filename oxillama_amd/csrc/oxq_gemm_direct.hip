// The few-token kernel that keeps its tokens in registers (oxq_gemm_direct.hpp), instantiated for its formats.
#include "oxq_gemm_direct_launch.hpp"

namespace oxq {

// Token tiles a work group takes: as many as registers hold, fewer where the matrix has so few row tiles that work groups for more
// runs of tokens still find a compute unit each (256 x 1536 of Q4_K, 77 rows: five runs of one tile, 3.5 us).
static uint32_t direct_token_tiles(uint32_t m, uint32_t n, uint32_t k) {
    const uint32_t tiles = (m + 15) / 16, most = k > 2048 && k <= 4096 ? 2 : 4, rows = (n + 15) / 16;
    const uint32_t fewest = (tiles + most - 1) / most, fill = device_cus() / rows;
    const uint32_t chunks = fill > tiles ? tiles : fill > fewest ? fill : fewest;
    return (tiles + chunks - 1) / chunks;
}
// Row tiles that a work group walks.
static uint32_t direct_walk(uint32_t m, uint32_t n, uint32_t k, uint32_t tt) {
    const uint32_t chunks = (m + 16 * tt - 1) / (16 * tt), room = device_cus() > chunks ? device_cus() / chunks : 1;
    const uint32_t rows = (n + 15) / 16, sets = k <= 1024 ? (rows + 1) / 2 : rows;
    return (sets + room - 1) / room;
}

static bool direct_format(uint32_t type) {
    return type == OXQ_TYPE_Q4_K || type == OXQ_TYPE_Q5_K || type == OXQ_TYPE_Q6_K || type == OXQ_TYPE_IQ4_XS || type == OXQ_TYPE_Q4_0 ||
           type == OXQ_TYPE_Q8_0;
}
// Where it is the better kernel, us, against what such calls took before (the few-token kernel with k split over work groups or the
// whole k in LDS, the tile kernel, GEMV launches), 1036 calls of 3 to 32 rows on 25 matrices, weights from HBM, 0.73 of the time
// in the mean.  Sixteen rows: Q4_K 4096 x 4096 8.0 to 5.9, 1024 x 4096 6.8 / 5.2, 14336 x 4096 17 / 12.6, 8960 x 1536 7.6 / 5.5,
// 128256 x 4096 116 / 68; Q6_K 4096 x 4096 10.4 / 7.2, 14336 x 4096 24 / 19.7; Q8_0 9.9 / 8.8, 25 / 22.9; 32 rows of Q4_K
// 4096 x 4096 12.5 / 8.7, 14336 x 4096 22 / 16.8.
//  * Longer rows (streamed: a wave's tokens pass through its registers once per row tile): while no work group walks a second row
//    tile.  16 rows of 4096 x 14336: Q4_K 19.3 / 16.4, Q6_K 25.3 / 20.8, IQ4_XS 20 / 15.2, Q8_0 26.7 / 25.6; 28672 x 8192 of Q4_K
//    39 / 61.  Q8_0 of 1024 x 8192 13.5 / 14.3, 1536 x 8960 16.6 / 12.3.  Beyond 32768 columns: not measured.
//  * Q8_0 vocabularies, where the bytes are the time: 128256 x 4096 119 / 136.
// More than 32 rows, up to 512 (3000 calls of Q4_K, IQ4_XS, Q6_K, Q8_0 against the tile kernel and its token re-layout launch): the tile
// kernel is a serial chain of k / 4 where the work groups here meet k / 8 or k / 16, and gains on this one only by weights unpacked
// for more tokens.  So the line is drawn at the tiles of 16 x 16 a work group goes through (`work`):
//  * up to 2048 columns 28 (0.63 of the time in the mean, the worst 1.04: Q6_K 333 rows of 4096 x 1536 26.6 / 27.7; from 32 on 0.81 to
//    1.14), Q8_0 56.  77 rows of Q4_0: 1536 x 1536 12.2 / 6.3, 256 x 1536 12.1 / 3.7, 8960 x 1536 22.4 / 13.3;
//  * up to 4096 columns, two token tiles at most and two super-blocks a wave, a part of which is idle in shorter rows (hence the
//    square): Q4_K 28 (64 rows of 4096 x 4096 13.7 / 11, 1024 x 4096 12.2 / 5.4, 128 of 14336 x 4096 44 / 35.5), IQ4_XS 14, Q6_K
//    8 (64 rows of 4096 x 4096 18.9 / 15.2; 112 of 14336 x 4096, 16, 1.13 of the f16 kernel's), Q8_0 4 (16.1 / 7.9; 80 rows of 4096 x 4096, 8, 20.7 / 23.1);
//  * longer rows (streamed): one row tile a work group, as with 16 rows.  64 rows of 2048 x 8192 Q4_K 0.66 of the time, 4096 x
//    14336 Q6_K 48.9 / 39; two row tiles 0.9 to 1.3.  Four token tiles where they fill the chip: not for the light formats
//    (Q4_K 64 rows of 4096 x 14336 31.3 / 32.3), nor against the f16 kernel (Q4_K 128 rows of 2048 x 14336 1.06).  17 to 32
//    rows beyond 20480 columns: a tie in the light ones.
// Q4_0 and Q5_K at Q4_K's lines: 320 calls of 21 matrices 0.68 of the tile kernel's time in the mean, none above 1.04.
// Where the f16 kernels would serve the call they are faster or level (Q6_K 112 rows of 14336 x 1536 1.17; longer rows up to three token tiles 0.86).
bool gemm_direct_pays(uint32_t type, uint32_t m, uint32_t n, uint32_t k) {
    if (!direct_format(type) || m == 0 || m > DIRECT_MAX_ROWS || k % 256 != 0 || k < 512 || k > 32768) return false;
    const bool heavy = type == OXQ_TYPE_Q6_K || type == OXQ_TYPE_Q8_0;
    if (m <= 16 && k > 4096) return n <= 16 * device_cus() && (type != OXQ_TYPE_Q8_0 || n >= 1536);
    if (m <= 32 && k <= 4096) return type != OXQ_TYPE_Q8_0 || n < 256 * device_cus();
    const uint32_t tt = direct_token_tiles(m, n, k), walk = direct_walk(m, n, k, tt), nb = k / 256;
    const bool f16 = gemm_f16_shape(type, m, n, k) != 0 || gemm_f16_deal_pays(type, m, n, k) ||
                     (gemm_prefill_supported(type, m, n, k) && gemm_prefill_pays(m, n));
    if (k > 4096) return walk == 1 && (m > 32 || heavy || k <= 20480) && (tt <= 3 || (!f16 && (heavy || m > 64)));
    if (f16) return false;
    const uint64_t work = (uint64_t)walk * tt;
    if (k <= 2048) return work <= (type == OXQ_TYPE_Q8_0 ? 56u : 28u);
    return work * 256 <= (uint64_t)nb * nb * (type == OXQ_TYPE_Q8_0 ? 4u : type == OXQ_TYPE_Q6_K ? 8u : type == OXQ_TYPE_IQ4_XS ? 14u : 28u);
}

hipError_t launch_gemm_direct(uint32_t type, const GemmArgs &a, hipStream_t stream) {
    if (a.offsets || a.m == 0 || a.m > DIRECT_MAX_ROWS || a.k % 256 != 0 || a.k < 512 ||
        (size_t)a.m * (a.k / 32) * Q8_BLOCK_BYTES > 0x7FFFFFFF || (reinterpret_cast<uintptr_t>(a.W) & 3) ||
        (reinterpret_cast<uintptr_t>(a.A) & 15))  // (what loads straight to LDS and the dword-wise loads were built for)
        return hipErrorNotSupported;
    uint32_t tt = direct_token_tiles(a.m, a.n, a.k);
    if (a.sums && tt > 2) tt = 2;  // (the dump: the same parts of k, so the same bits)
    return tt > 2 ? launch_direct_wide(type, tt, a, stream) : launch_direct_of<1, 2>(type, tt, a, stream);
}

}  // namespace oxq
