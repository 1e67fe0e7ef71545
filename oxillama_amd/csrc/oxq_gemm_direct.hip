// The few-token kernel that keeps its tokens in registers (oxq_gemm_direct.hpp), instantiated for its formats.
#include "oxq_gemm_direct_launch.hpp"

namespace oxq {

// Token tiles a work group takes: as many as registers hold, fewer where the matrix has so few row tiles that work groups for more
// runs of tokens still find a compute unit each (256 x 1536 of Q4_K, 77 rows: five runs of one tile, 3.6 us).
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
// Up to 32 rows of more than 4096 columns, of which a wave goes through nb / 8 super-blocks, against the few-token kernel's split of k: a
// chain of `per` of them in every work group and a reduction launch, which this kernel does not have.  So the line is what its
// chain may be longer by, in super-blocks of the matrix (8 a wave), fitted to 2400 calls of 3 to 16 rows: Q5_K, Q6_K 20,
// Q4_K 24, IQ4_XS 28, and 8 more up to eight rows (Q4_K 16 rows of 2048 x 13312, 20 above: 0.85 of the split's time, x 16384, 32: 0.95 to 1.03,
// x 20480, 32: 1.14); the light Q4_0 8 and 16, Q8_0, whose split reads as fast as memory gives, -4 and 4 (2048 x 7680, -18, 0.80; 2048 x 14336, 24, 1.24).
// Where the split makes more work groups than there are compute units, two of them share some: 48 (Q5_K 40, Q4_0 32, Q8_0 28; 4096 x
// 14336, 16 rows, Q4_K 0.83, Q6_K 0.83, Q8_0 0.98).  17 to 32 rows are split from 2^25 weights on, and take two passes
// in Q6_K and Q8_0.
static bool direct_chain_pays(uint32_t type, uint32_t m, uint32_t n, uint32_t k, uint32_t tt) {
    const uint32_t per = skinny_sb_per_split(n, k), cus = device_cus();
    if (per == 0 || (m > 16 && (uint64_t)n * k < (1ull << 25))) return true;  // (no split)
    const int above = (int)(k / 256) - (int)(8 * per);
    const bool shared = (n + 127) / 128 * skinny_splits(n, k) > cus;
    if (m <= 16) {
        const int most = type == OXQ_TYPE_Q8_0   ? (shared ? 28 : -4)
                         : type == OXQ_TYPE_Q4_0 ? (shared ? 32 : 8)
                         : shared                ? (type == OXQ_TYPE_Q5_K ? 40 : 48)
                                                 : (type == OXQ_TYPE_IQ4_XS ? 28 : type == OXQ_TYPE_Q4_K ? 24 : 20);
        return above <= most + (m <= 8 ? 8 : 0);
    }
    if (type == OXQ_TYPE_Q8_0 || type == OXQ_TYPE_Q6_K) {
        if (n >= 14 * cus) return true;  // (3584 x 28672, 17 to 32 rows: Q6_K 0.78, Q8_0 0.92)
        if (type == OXQ_TYPE_Q6_K || n >= 12 * cus) return k <= 28672;  // (2048 x 28672 / 32768 Q6_K 0.94 / 1.06; 3072: Q8_0 1.04 / 1.16)
        return above <= (shared ? 28 : tt == 1 ? 24 : 16);
    }
    return tt == 1 || shared || above <= 16;  // (two token tiles; Q4_K 2560 x 16384 0.89, x 17408, 20 above, 1.02)
}
// Where it is the better kernel, us, against what such calls took before (the few-token kernel with k split over work groups or the
// whole k in LDS, the tile kernel, GEMV launches).  Up to 32 rows of up to 4096 columns: 672 calls of six formats on 18
// matrices, weights from HBM, 0.66 of the time in the mean, the worst 1.02.  Sixteen rows: Q4_K 4096 x 4096 7.9 to 5.9, 1024 x 4096 6.7 / 5.2,
// 14336 x 4096 16.5 / 12.5, 8960 x 1536 7.9 / 5.9, 128256 x 4096 71 / 67; Q6_K 4096 x 4096 10.3 / 7.2, 14336 x 4096 23.1 / 19.7; Q8_0 10.1 / 8.7,
// 24.2 / 22.8; 32 rows of Q4_K 4096 x 4096 13.3 / 8.7, 14336 x 4096 21.5 / 16.4.
//  * Longer rows (streamed: a wave's tokens pass through its registers once per row tile): while no work group walks a second row
//    tile, and by direct_chain_pays (887 calls of up to 32 rows on 29 matrices, 0.70 of the time in the mean, the worst 1.07).  16 rows of 4096 x 14336: Q4_K 19.3 / 15.8, Q6_K 25.4 / 21.2, IQ4_XS 19.9 / 15.2, Q8_0 26.5 / 26;
//    28672 x 8192 of Q4_K 42 / 63.  Beyond 32768 columns: not measured.  Q8_0 of 1024 x 8192 14.3 / 15.9.
//  * Q8_0 vocabularies, where the bytes are the time: 128256 x 4096, 16 rows, 117 / 134.
// More than 32 rows, up to 512, against the tile kernel and its token re-layout launch: 2480 calls of six formats on 57
// matrices, 0.61 of the time in the mean.  The tile kernel is a serial chain
// of k / 4 where the work groups here meet k / 8 or k / 16, and gains on this one only by weights unpacked
// for more tokens.  So the line is drawn at the tiles of 16 x 16 a work group goes through (`work`):
//  * up to 2048 columns 28, Q6_K beyond 1024 24 (1116 calls, 0.64 of the time in the mean, the worst 1.05; beyond 0.81 to 1.14, Q6_K 333 rows of 4096 x
//    1536, 28, 27.8 / 29.3), Q8_0 56.  77 rows of Q4_0: 1536 x 1536 12.2 / 5.6, 256 x 1536 11.6 / 3.6, 8960 x 1536 22.3 / 12.2;
//  * up to 4096 columns, two token tiles at most and two super-blocks a wave, a part of which is idle in shorter rows (hence the
//    square): Q4_K 28 (64 rows of 4096 x 4096 13.5 / 11.1, 1024 x 4096 12.2 / 5.4, 128 of 14336 x 4096 42.8 / 36.9), IQ4_XS 14, Q6_K
//    8 (64 rows of 4096 x 4096 18.8 / 15.2; 112 of 14336 x 4096, 16, 1.12 of the f16 kernel's), Q8_0 4 (64 rows of 4096 x 4096 19.4 / 14.9; 80, 8, 21.2 / 21.9);
//  * longer rows (streamed): one row tile a work group, as with 16 rows.  64 rows of 2048 x 8192 Q4_K 20 / 13, 4096 x
//    14336 Q6_K 48.6 / 38.5; two row tiles 0.9 to 1.3.  Four token tiles where they fill the chip: not for the light formats
//    (Q4_K 64 rows of 4096 x 14336 32.3 / 33.9), nor against the f16 kernel (Q4_K 128 rows of 2048 x 14336 1.02).  17 to 32
//    rows beyond 20480 columns: a tie in the light ones.
// Where the f16 kernels would serve the call they are faster or level (Q6_K 112 rows of 14336 x 1536 1.13; longer rows up to three token tiles
// 0.66 to 1.05 up to 28672 columns, on three up to 20480: Q4_K 96 rows of 2048 x 24576 36 / 38.1, x 32768 43.3 / 50.7).
bool gemm_direct_pays(uint32_t type, uint32_t m, uint32_t n, uint32_t k) {
    if (!direct_format(type) || m == 0 || m > DIRECT_MAX_ROWS || k % 256 != 0 || k < 512 || k > 32768) return false;
    const bool heavy = type == OXQ_TYPE_Q6_K || type == OXQ_TYPE_Q8_0;
    if (m <= 16 && k > 4096)
        return n <= 16 * device_cus() && (type != OXQ_TYPE_Q8_0 || n >= 1536) && direct_chain_pays(type, m, n, k, 1);
    if (m <= 32 && k <= 4096) return type != OXQ_TYPE_Q8_0 || n < 256 * device_cus();
    const uint32_t tt = direct_token_tiles(m, n, k), walk = direct_walk(m, n, k, tt), nb = k / 256;
    const bool f16 = gemm_f16_shape(type, m, n, k) != 0 || gemm_f16_deal_pays(type, m, n, k) ||
                     (gemm_prefill_supported(type, m, n, k) && gemm_prefill_pays(m, n));
    if (k > 4096) {
        if (walk != 1) return false;
        if (m <= 32) return (heavy || k <= 20480) && direct_chain_pays(type, m, n, k, tt);
        return tt <= 3 ? !f16 || k <= (tt == 3 ? 20480u : 28672u) : !f16 && (heavy || m > 64);
    }
    if (f16) return false;
    const uint64_t work = (uint64_t)walk * tt;
    if (k <= 2048) return work <= (type == OXQ_TYPE_Q8_0 ? 56u : type == OXQ_TYPE_Q6_K && k > 1024 ? 24u : 28u);
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
