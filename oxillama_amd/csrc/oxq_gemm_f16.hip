// Matmul on the f16 matrix cores straight from the caller's Q8_0 rows, for Q4_K, Q5_K and Q6_K weights:
//   out[m x n] (+)= A_q8[m rows of Q8_0 blocks] x W[n x k]^T
// i.e. m fused matvecs over the same weight blocks (the reference's gemm is that loop,
// crates/oxillama-quant/src/reference/q4_k.rs:186-201).
//
// The arithmetic is the prefill kernel's (oxq_gemm_prefill.hip): the integer scale of a sub-block rides inside the f16
// weight operand, the matrix core's fp32 result T[token][row][sub-block] = scale * (integer group sum) is exact, one fma
// per result applies the token's block scale, d (and dmin) are applied once per 256-weight super-block.
//   Q4_K  sc * q <= 63 * 15, Q5_K sc * q <= 63 * 31 = 1953: eleven bits, one f16 operand.
//   Q6_K  sc * (q - 32), up to 128 * 32 in size, has thirteen bits.  With sc = s + p, p = sc & 1, the parts s * (q - 32)
//         (even, so at most eleven bits after the factor 2) and p * (q - 32) are both exact in f16: two operands, the
//         matrix core adds them up.  The scale changes every 16 weights, and a lane's 16 bytes are one such half.
//
// What differs: no preparation launch and no workspace.  A stage (64 columns of the work group's tokens) is read as raw
// Q8_0 blocks by the work group's threads, widened to f16 (a byte becomes the low mantissa bits of 1024.0 by one
// v_perm per pair, one packed add takes 1152 off again) and written to LDS in operand order, two stages before it is
// read; the block sums P of the zero-point term are formed on the way.  That is about 3.5 vector instructions per step of
// 27 (the prefill kernel's preparation launch is 6 us at 512 x 4096 and reads and writes the tokens once more).
//
// The even deal (DEAL; the large shape): whole tiles cost a round of the chip what the fullest compute unit has, and most
// prompts' grids lie between rounds (333 rows on 11008 weight rows: 129 tiles for 256 compute units).  Here a work group per
// compute unit takes the same number of whole tiles and then a run of (tile, super-block) units of the rest; a tile that
// several have runs of is added up by a second launch, in the order of k.  What it costs: a ramp of the pipeline per run and 128 KB
// of sums, 32 to 64 MB written together at the end and read by the second launch (9 to 14 us: 10 of 96 tiles of 333 x 4096 x
// 11008, 14 of 129 of 333 x 11008 x 4096): 128 x 4096 x 14336, Q4_K, runs of four super-blocks, 36 us + 8, where whole tiles take 5.8
// per super-block.  And registers: what a work group keeps from run to run takes Q5_K and Q6_K over the 256 there are (ten and
// eighteen spilled, 44 and 76 bytes of scratch a lane; without the deal one and none), part of why a super-block of a run is
// 7.4 / 9.5 us where it is 6.2 / 7.6 of a whole tile.  Storing the sums past the caches: no gain (333 x 11008 x 4096 77 us
// against 75).
//
// Shapes: MT token tiles of 32 against RW waves of 32 rows, KS parts of k; eight waves, one work group per compute unit.
//   (4, 8, 1)  128 tokens x 256 rows: the least unpacking and staging per result
//   (2, 4, 2)  64 tokens x 128 rows, each half of k by four waves (their sums meet in LDS): four times the work groups,
//              for matrices and prompts that do not fill the chip with the large tile
// What bounds it: the issue of a SIMD's instructions.  Matrix and vector instructions of its two waves take turns (measured
// with mixes of both: 64 cycles for two MFMAs, and 2.2 a v_fmac, 3 to 4.4 an integer or packed instruction on top of
// them).  By rocprofv3's counters a step of the large shape takes 254 to 266 cycles
// for Q6_K: 128 of matrix work, 37 other vector instructions, 67 cycles of both at once.  The small shape, which unpacks
// and stages twice as much per result, takes 415 (Q6_K, 56 vector instructions; k = 14336), 432 (Q4_K, 46) and 468 (Q5_K, 57;
// k = 4096, the launch's ramp and the exchange of the halves included).
// Measured, us, this kernel against the tile kernel: Q6_K 2048 x 8192 x 28672 1893 against 2946 (508 TOPS), 2048 x 8192 x
// 8192 542 / 656, 512 x 14336 x 4096 130 / 166, 512 x 4096 x 14336 175 / 207; Q4_K 512 x 4096 x 4096 42 / 48.5, 2048 x 1024 x 4096
// 42 / 51; Q5_K 2048 x 4096 x 14336 388 / 454, 512 x 4096 x 4096 48 / 54.
#include "oxq_gemm_f16_util.hpp"
#include "oxq_tile_order.hpp"
#include "oxq_tile_rule.hpp"

namespace oxq {
namespace {

// Per format:
//   Raw, fetch_ql / fetch_qh   the lane's bytes of group g (64 weights) of a super-block, requested two groups (qh: up to a super-block) ahead
//   sub_block(g, e)            which sub-block of the super-block the e-th of group g is; e-th minus first: E_STEP
//   Hdr, load_hdr, decode      the scales of the lane's row: the tables of one super-block of the wave's rows in LDS
//   Const, load_const, unpack  the operands of one sub-block from the lane's 16 raw bytes: wf[piece][kk]
// Constants of the unpacking in registers, hidden from constant folding: an instruction takes no second literal, and
// (w & mask) | x is one v_and_or_b32 only with the mask in a scalar register.
struct Masks {
    uint32_t magic;    // f16 1024.0 twice (vector register)
    uint32_t q[2];     // the low nibble's bits of both 16-bit halves; the high one's
    uint32_t high[2];  // the bits above them: of 5- and 6-bit weights
};

struct F16Q4K {
    static constexpr uint32_t TYPE = OXQ_TYPE_Q4_K, BLOCK = 144, E_STEP = 1;
    static constexpr bool HAS_MIN = true;
    static constexpr int PIECES = 1, NQH = 0;
    static constexpr uint32_t HIGH[2] = {0, 0};
    // sck [group][row][c1 lo, c2 lo, c1 hi, c2 hi] f16 pairs; mnb [row][8 bf16]; d, -dmin [row] fp32
    static constexpr uint32_t T_MNB = 2048, T_D = 2560, T_NDM = 2688, T_BYTES = 2816;
    struct Hdr {
        u32x4 w;
    };
    typedef u32x2 Const;
    static __device__ __forceinline__ constexpr uint32_t sub_block(uint32_t g) { return 2 * g; }
    static __device__ __forceinline__ u32x4 fetch_ql(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t blk, uint32_t g) {
        return buf16(rs, off, blk * BLOCK + 16 + 32 * g);
    }
    static __device__ __forceinline__ u32x4 fetch_qh(__amdgpu_buffer_rsrc_t, uint32_t, uint32_t, uint32_t) { return u32x4{0, 0, 0, 0}; }
    static __device__ __forceinline__ Hdr load_hdr(__amdgpu_buffer_rsrc_t rs, uint32_t row_off, uint32_t blk) {
        return Hdr{buf16(rs, row_off, blk * BLOCK)};
    }
    // lane (row c, half h) decodes sub-blocks 4h .. 4h + 3 (decode_scales_mins, reference/q4_k.rs:27-49)
    static __device__ __forceinline__ void decode(const Hdr &hdr, uint8_t *tab, uint32_t c, uint32_t h) {
        const u32x4 hd = hdr.w;
        const float d = h2f(hd[0] & 0xFFFF), dmin = h2f(hd[0] >> 16);
        uint32_t mnq[2] = {0, 0};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t s = 4 * h + i, sh = 8 * i;
            const uint32_t sc_lo = (hd[1] >> sh) & 63, mn_lo = (hd[2] >> sh) & 63;
            const uint32_t sc_hi = ((hd[3] >> sh) & 15) | (((hd[1] >> (sh + 6)) & 3) << 4);
            const uint32_t mn_hi = ((hd[3] >> (sh + 4)) & 15) | (((hd[2] >> (sh + 6)) & 3) << 4);
            const uint32_t sc = h ? sc_hi : sc_lo, mn = h ? mn_hi : mn_lo;
            const float fs = (float)sc;
            // low nibbles enter as 1024 + q, high ones in place as 1024 + 16 q
            const uint32_t g = s >> 1, e = s & 1;
            u32x2 ck;
            ck[0] = f16x2_of(e ? fs * 0.0625f : fs);
            ck[1] = f16x2_of(e ? -64.0f * fs : -1024.0f * fs);
            *reinterpret_cast<lds_u32x2 *>(tab + (g * 32 + c) * 16 + e * 8) = ck;
            const uint32_t mb = __builtin_bit_cast(uint32_t, (float)mn) >> 16;  // bf16 of an integer <= 63: exact
            if (i & 1) mnq[i >> 1] |= mb << 16; else mnq[i >> 1] = mb;
        }
        *reinterpret_cast<lds_u32x2 *>(tab + T_MNB + c * 16 + h * 8) = u32x2{mnq[0], mnq[1]};
        *reinterpret_cast<lds_f32 *>(tab + T_D + c * 4) = d;  // (both halves: the same value)
        *reinterpret_cast<lds_f32 *>(tab + T_NDM + c * 4) = -dmin;
    }
    static __device__ __forceinline__ Const load_const(const uint8_t *tab, uint32_t g, uint32_t e, uint32_t c, uint32_t) {
        return *reinterpret_cast<const lds_u32x2 *>(tab + (g * 32 + c) * 16 + e * 8);
    }
    template <int G, int E>
    static __device__ __forceinline__ void unpack(const u32x4 ql, const u32x4, const Const ck, const Masks &mk, h8 (&wf)[PIECES][2]) {
        const h2v c1 = __builtin_bit_cast(h2v, ck[0] + 0u), c2 = __builtin_bit_cast(h2v, ck[1] + 0u);
        const uint32_t mask = mk.q[E];
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            uint32_t o[4];
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const uint32_t w = ql[2 * kk + d];
                const h2v t0 = __builtin_bit_cast(h2v, (w & mask) | mk.magic);         // bytes 0 and 2
                const h2v t1 = __builtin_bit_cast(h2v, ((w >> 8) & mask) | mk.magic);  // bytes 1 and 3
                o[2 * d] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t0, c1, c2));
                o[2 * d + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t1, c1, c2));
            }
            wf[0][kk] = __builtin_bit_cast(h8, u32x4{o[0], o[1], o[2], o[3]});
        }
    }
};

// Q5_K: the same header; the fifth bits of weight l of sub-blocks 2g and 2g + 1 are bits g and g + 4 of qh[l].
struct F16Q5K : F16Q4K {
    static constexpr uint32_t TYPE = OXQ_TYPE_Q5_K, BLOCK = 176;
    static constexpr int NQH = 1;
    static constexpr uint32_t HIGH[2] = {0x00100010u, 0x01000100u};
    static __device__ __forceinline__ u32x4 fetch_ql(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t blk, uint32_t g) {
        return buf16(rs, off, blk * BLOCK + 48 + 32 * g);
    }
    static __device__ __forceinline__ u32x4 fetch_qh(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t blk, uint32_t) {
        return buf16(rs, off, blk * BLOCK + 16);
    }
    static __device__ __forceinline__ Hdr load_hdr(__amdgpu_buffer_rsrc_t rs, uint32_t row_off, uint32_t blk) {
        return Hdr{buf16(rs, row_off, blk * BLOCK)};
    }
    template <int G, int E>
    static __device__ __forceinline__ void unpack(const u32x4 ql, const u32x4 qh, const Const ck, const Masks &mk, h8 (&wf)[PIECES][2]) {
        const h2v c1 = __builtin_bit_cast(h2v, ck[0] + 0u), c2 = __builtin_bit_cast(h2v, ck[1] + 0u);
        const uint32_t mask = mk.q[E], bit = mk.high[E];
        // bit G + 4E of a byte goes to bit 4 (E = 0) or 8 (E = 1) of its 16-bit half: up by 4 - G either way, and down
        // by 4 + G from the odd bytes
        constexpr int up = 4 - G, down = 4 + G;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            uint32_t o[4];
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const uint32_t w = ql[2 * kk + d], b = qh[2 * kk + d];
                const h2v t0 = __builtin_bit_cast(h2v, ((b << up) & bit) | ((w & mask) | mk.magic));
                const h2v t1 = __builtin_bit_cast(h2v, ((b >> down) & bit) | (((w >> 8) & mask) | mk.magic));
                o[2 * d] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t0, c1, c2));
                o[2 * d + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t1, c1, c2));
            }
            wf[0][kk] = __builtin_bit_cast(h8, u32x4{o[0], o[1], o[2], o[3]});
        }
    }
};

// Q6_K (reference/q6_k.rs:25-75): ql[128], qh[64], 16 int8 scales, d.  Group g = (half g / 2, pair g % 2): ql[64 (g/2) +
// 32 (g%2) + l] holds the low bits of weight l of sub-blocks 4 (g/2) + g%2 (low nibble) and of that + 2 (high nibble), bits
// 2 (g%2) and + 4 of qh[32 (g/2) + l] their upper two.
struct F16Q6K {
    static constexpr uint32_t TYPE = OXQ_TYPE_Q6_K, BLOCK = 210, E_STEP = 2;
    static constexpr bool HAS_MIN = false;
    static constexpr int PIECES = 2, NQH = 2;
    static constexpr uint32_t HIGH[2] = {0x00300030u, 0x03000300u};
    // sc [group][row][half][e]: f16 s and p of the scale (both over 16 for e = 1, whose weights enter as 16 q); d [row] fp32
    static constexpr uint32_t T_D = 2048, T_BYTES = 2176;
    struct Hdr {
        u32x4 sc;
        uint32_t d;
    };
    typedef uint32_t Const;
    static __device__ __forceinline__ constexpr uint32_t sub_block(uint32_t g) { return 4 * (g >> 1) + (g & 1); }
    static __device__ __forceinline__ u32x4 fetch_ql(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t blk, uint32_t g) {
        return buf16(rs, off, blk * BLOCK + 32 * g);
    }
    static __device__ __forceinline__ u32x4 fetch_qh(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t blk, uint32_t hh) {
        return buf16(rs, off, blk * BLOCK + 128 + 32 * hh);
    }
    static __device__ __forceinline__ Hdr load_hdr(__amdgpu_buffer_rsrc_t rs, uint32_t row_off, uint32_t blk) {
        Hdr hd;
        hd.sc = buf16(rs, row_off, blk * BLOCK + 192);
        hd.d = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, row_off, blk * BLOCK + 208, 0);
        return hd;
    }
    // lane (row c, half h) decodes the scales of half h of all eight sub-blocks: scales[2 s + h]
    static __device__ __forceinline__ void decode(const Hdr &hd, uint8_t *tab, uint32_t c, uint32_t h) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            u32x2 k;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const uint32_t s = sub_block(g) + 2 * e;  // its pair of scales: bytes 2 (s % 2) and + 1 of dword s / 2
                const int sc = (int)(int8_t)((hd.sc[s >> 1] >> (16 * (s & 1) + 8 * h)) & 0xFF);
                const float f = e ? 0.0625f : 1.0f;
                k[e] = f2h((float)(sc & ~1) * f) | (f2h((float)(sc & 1) * f) << 16);
            }
            *reinterpret_cast<lds_u32x2 *>(tab + (g * 32 + c) * 16 + h * 8) = k;
        }
        *reinterpret_cast<lds_f32 *>(tab + T_D + c * 4) = h2f(hd.d);
    }
    static __device__ __forceinline__ Const load_const(const uint8_t *tab, uint32_t g, uint32_t e, uint32_t c, uint32_t h) {
        return *reinterpret_cast<const lds_u32 *>(tab + (g * 32 + c) * 16 + h * 8 + e * 4);
    }
    template <int G, int E>
    static __device__ __forceinline__ void unpack(const u32x4 ql, const u32x4 qh, const Const ck, const Masks &mk, h8 (&wf)[PIECES][2]) {
        const h2v k = __builtin_bit_cast(h2v, ck);
        const h2v s = {k[0], k[0]}, p = {k[1], k[1]};
        // 1024 + q - 1056, or 1024 + 16 q - 1536: q - 32 and 16 (q - 32), exact
        const h2v zero = E ? h2v{(_Float16)-1536.0f, (_Float16)-1536.0f} : h2v{(_Float16)-1056.0f, (_Float16)-1056.0f};
        const uint32_t mask = mk.q[E], bits = mk.high[E];
        constexpr int up = 4 - 2 * (G & 1), down = 4 + 2 * (G & 1);
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            uint32_t a[4], b[4];
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const uint32_t w = ql[2 * kk + d], x = qh[2 * kk + d];
                const h2v t0 = __builtin_bit_cast(h2v, ((x << up) & bits) | ((w & mask) | mk.magic)) + zero;
                const h2v t1 = __builtin_bit_cast(h2v, ((x >> down) & bits) | (((w >> 8) & mask) | mk.magic)) + zero;
                a[2 * d] = __builtin_bit_cast(uint32_t, t0 * s);
                a[2 * d + 1] = __builtin_bit_cast(uint32_t, t1 * s);
                b[2 * d] = __builtin_bit_cast(uint32_t, t0 * p);
                b[2 * d + 1] = __builtin_bit_cast(uint32_t, t1 * p);
            }
            wf[0][kk] = __builtin_bit_cast(h8, u32x4{a[0], a[1], a[2], a[3]});
            wf[1][kk] = __builtin_bit_cast(h8, u32x4{b[0], b[1], b[2], b[3]});
        }
    }
};

template <class F, int MT, int RW, int KS, bool DEAL>
__global__ __launch_bounds__(64 * RW * KS) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_f16_kernel(
    const uint8_t *__restrict__ W, const uint8_t *__restrict__ A, float *__restrict__ out, uint32_t m, uint32_t n, uint32_t k,
    int accumulate, const float *__restrict__ bias, uint32_t m_tiles, uint32_t n_tiles, float *__restrict__ partial) {
    static_assert(MT * 2 == RW, "one 16-byte piece of a stage per thread");
    static_assert(!DEAL || KS == 1, "the deal is over whole work groups");
    static_assert(MT % KS == 0, "the parts of k share the token tiles out at the end");
    constexpr uint32_t TOK = 32 * MT, ROWS = 32 * RW, STAGE = TOK * 128;
    constexpr int NS = 8 * MT;  // steps of a super-block
    // per part of k: four stage buffers; token scales of the stages, fp32 [stage][e][token]; the bf16 pieces of P of two
    // super-blocks in turn [plane][token][8], plane 3 zero; the waves' tables, two super-blocks' in turn
    __shared__ __align__(16) uint8_t tok_all[KS][4][STAGE];
    __shared__ __align__(16) float das_all[KS][4][2][TOK];
    __shared__ __align__(16) uint8_t pl_all[KS][F::HAS_MIN ? 2 : 1][F::HAS_MIN ? 4 * TOK * 16 : 16];
    __shared__ __align__(16) uint8_t tab_all[KS][RW][2][F::T_BYTES];

    const uint32_t n_super = k / 256, nsb = k / 32;
    const uint32_t part = KS == 1 ? 0 : (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / (64 * RW)));
    const uint32_t tid = KS == 1 ? threadIdx.x : threadIdx.x % (64 * RW), lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    auto &tok = tok_all[part];
    auto &das = das_all[part];
    auto &pl = pl_all[part];
    auto &tab = tab_all[part];
    // this part's super-blocks, the first part's the longer run
    const uint32_t per_part = (n_super + KS - 1) / KS;
    uint32_t blk0 = part * per_part, nblk = min(blk0 + per_part, n_super);
    const uint32_t c = lane & 31, h = lane >> 5;

    uint32_t m_tile, n_tile;
    // DEAL: whole tiles first, as many to every work group, the rest of them as runs of super-blocks
    uint32_t tile = 0, whole = 0, unit = 0, unit_end = 0, slot = 0;
    bool dealt = false;
    if constexpr (DEAL) {
        const uint32_t rank = deal_rank(blockIdx.x, gridDim.x), rounds = m_tiles * n_tiles / gridDim.x;
        const DealRange r = deal_range(rank, gridDim.x, (m_tiles * n_tiles - rounds * gridDim.x) * n_super);
        tile = rank * rounds, whole = rounds, unit = r.begin, unit_end = r.end, slot = 2 * rank;
        if (whole == 0 && unit == unit_end) return;
    } else {
        if (!tile_run_at(blockIdx.x, gridDim.x, m_tiles, n_tiles, m_tile, n_tile)) return;  // the whole work group
    }
    do {  // (DEAL: the work group's run of a tile, then its run of the next one)
    if constexpr (DEAL) {
        uint32_t t = tile;
        if (whole) {
            blk0 = 0, nblk = n_super;
            tile++, whole--;
        } else {
            t = unit / n_super;
            blk0 = unit - t * n_super, nblk = min(n_super, blk0 + (unit_end - unit));
            unit += nblk - blk0;
            dealt = true;
            t += m_tiles * n_tiles / gridDim.x * gridDim.x;
        }
        n_tile = t / m_tiles, m_tile = t - n_tile * m_tiles;
    }
    const uint32_t m_wg = m_tile * TOK, n_wg = n_tile * ROWS, n_wave = n_wg + 32 * wave;

    const uint32_t row_bytes = n_super * F::BLOCK;
    const size_t w_left = (size_t)(n - n_wg) * row_bytes;
    const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(W + (size_t)n_wg * row_bytes), 0, (int)min(w_left, (size_t)0x7FFFFFFF), BUFFER_FLAGS);
    const uint32_t act_row = nsb * Q8_BLOCK_BYTES;
    const size_t a_left = (size_t)(m - m_wg) * act_row;
    const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(A + (size_t)m_wg * act_row), 0, (int)min(a_left, (size_t)0x7FFFFFFF), BUFFER_FLAGS);
    // the lane's weight row as A-operand supplier (rows past n re-read the last row; their results are not stored)
    const uint32_t wrow = (min(n_wave + c, n - 1) - n_wg) * row_bytes, wq_off = wrow + 16 * h;

    // ---- staging: thread (token tl, block pe of the stage's two, half ph of the block) ------------------------------
    const uint32_t tl = tid >> 2, pe = (tid >> 1) & 1, ph = tid & 1;
    const uint32_t act_off = min(tl, m - 1 - m_wg) * act_row + pe * F::E_STEP * Q8_BLOCK_BYTES;  // (tokens past m: the last one)
    const uint32_t frag_off = (((pe * MT + (tl >> 5)) * 2 + ph) * 2 * 32 + (tl & 31)) * 16;
    struct Staged {
        u32x4 q;
        uint32_t d;
    };
    auto stage_load = [&](uint32_t blk, uint32_t g) __attribute__((always_inline)) {
        const uint32_t so = (8 * min(blk, nblk - 1) + F::sub_block(g)) * Q8_BLOCK_BYTES;
        Staged s;
        s.q = __builtin_amdgcn_raw_buffer_load_b128(rs_a, act_off + 2 + 16 * ph, so, 0);
        s.d = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_a, act_off, so, 0);
        return s;
    };
    // g: the stage's place in its super-block, par: which of the two P buffers that super-block has
    auto stage_store = [&](const Staged &s, uint8_t *buf, int g, uint32_t par) __attribute__((always_inline)) {
        const h2v off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            uint32_t o[4];
#pragma unroll
            for (int d = 0; d < 2; d++) {  // pairs (0, 2) and (1, 3) of a dword's bytes: the order of pf_slot_byte
                const uint32_t x = s.q[2 * kk + d] ^ 0x80808080u;
                const h2v t0 = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, x, 0x04020400u));
                const h2v t1 = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, x, 0x04030401u));
                o[2 * d] = __builtin_bit_cast(uint32_t, t0 + off);
                o[2 * d + 1] = __builtin_bit_cast(uint32_t, t1 + off);
            }
            *reinterpret_cast<lds_u32x4 *>(buf + frag_off + kk * 512) = u32x4{o[0], o[1], o[2], o[3]};
        }
        const float d = h2f(s.d);
        das[g & 3][pe][tl] = d;  // (both halves: the same value)
        if constexpr (F::HAS_MIN) {
            int sum = 0;
            for (int i = 0; i < 4; i++) sum = sdot4(s.q[i], 0x01010101u, sum);
            sum += xor1_i(sum);
            // P = d * sum: at most 23 significant bits; three truncated bf16 pieces hold it exactly
            const float P = d * (float)sum;
            uint16_t piece[3];
            bf16_pieces(P, piece);
            uint8_t *at = pl[par] + tl * 16 + 2 * (2 * (g & 3) + pe);
            *reinterpret_cast<lds_u16 *>(at) = piece[0];
            *reinterpret_cast<lds_u16 *>(at + TOK * 16) = piece[1];
            *reinterpret_cast<lds_u16 *>(at + 2 * TOK * 16) = piece[2];
        }
    };
    // End of a stage: this wave's LDS traffic is done, then everybody's; loads to registers stay in flight.  It makes the
    // stage written during this one readable (from the end of the next one on) and frees this stage's buffer.
    auto stage_end = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto tokbuf = [&](int g) __attribute__((always_inline)) -> uint8_t * {
        return tok[g & 3];
    };
    auto tok_frag = [&](const uint8_t *buf, int ts, int kk) __attribute__((always_inline)) {
        return lds_h8(buf + (((ts * 2 + h) * 2 + kk) * 32 + c) * 16);
    };

    v16f y[MT], accblk[MT];
    for (int a = 0; a < MT; a++)
        for (int i = 0; i < 16; i++) y[a][i] = 0.0f, accblk[a][i] = 0.0f;
    v16f zero16;
    for (int i = 0; i < 16; i++) zero16[i] = 0.0f;
    Masks mk = {0x64006400u, {0x000F000Fu, 0x00F000F0u}, {F::HIGH[0], F::HIGH[1]}};
    asm volatile("" : "+v"(mk.magic), "+s"(mk.q[0]), "+s"(mk.q[1]));
    if constexpr (F::NQH) asm volatile("" : "+s"(mk.high[0]), "+s"(mk.high[1]));

    // ---- fill the pipeline -------------------------------------------------------------------------------------------
    u32x4 ql[2], qh[F::NQH ? F::NQH : 1];  // ql: slot g % 2, refilled two groups ahead
#pragma unroll
    for (int g = 0; g < 2; g++) ql[g] = F::fetch_ql(rs_w, wq_off, blk0, g);
#pragma unroll
    for (int i = 0; i < F::NQH; i++) qh[i] = F::fetch_qh(rs_w, wq_off, blk0, i);
    u32x4 qh_next = {0, 0, 0, 0};  // (one run of fifth bits for the whole super-block: the next one's waits here)
    if constexpr (F::NQH == 1) qh_next = F::fetch_qh(rs_w, wq_off, min(blk0 + 1, nblk - 1), 0);
    Staged st0 = stage_load(blk0, 0), st1 = stage_load(blk0, 1), st = stage_load(blk0, 2);
    F::decode(F::load_hdr(rs_w, wrow, blk0), tab[wave][blk0 & 1], c, h);
    if constexpr (F::HAS_MIN)
        for (uint32_t i = tid; i < TOK * 2; i += 64 * RW)
            *reinterpret_cast<lds_u32x4 *>(pl[i / TOK] + 3 * TOK * 16 + (i % TOK) * 16) = u32x4{0, 0, 0, 0};
    stage_store(st0, tok[0], 0, blk0 & 1);
    stage_store(st1, tok[1], 1, blk0 & 1);
    __syncthreads();
    h8 wf[F::PIECES][2], tf[2][2];
    v16f T[2];
    float da[2];
    typename F::Const ck = F::load_const(tab[wave][blk0 & 1], 0, 0, c, h);
    F::template unpack<0, 0>(ql[0], qh[0], ck, mk, wf);
    ck = F::load_const(tab[wave][blk0 & 1], 0, 1, c, h);
    auto mfma_chain = [&](const h8 (&t)[2]) __attribute__((always_inline)) {
        v16f r = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[0][0], t[0], zero16, 0, 0, 0);
        r = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[0][1], t[1], r, 0, 0, 0);
        if constexpr (F::PIECES == 2) {
            r = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[1][0], t[0], r, 0, 0, 0);
            r = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[1][1], t[1], r, 0, 0, 0);
        }
        return r;
    };
    // state carried from step to step (step q = 2 MT g + ts: sub-block ts / MT of group g against token tile ts % MT):
    //   wf     A operands of the sub-block that step q + 1 takes      tf[i]  token fragments of steps q + 1, q + 2
    //   da[i]  block scale of the lane's token for steps q, q + 1     T[i]   matrix-core results of steps q, q + 1
    da[0] = das[0][0][c];
    tf[0][0] = tok_frag(tok[0], 0, 0);
    tf[0][1] = tok_frag(tok[0], 0, 1);
    tf[1][0] = tok_frag(tok[0], 1, 0);
    tf[1][1] = tok_frag(tok[0], 1, 1);
    T[0] = mfma_chain(tf[0]);

    for (uint32_t blk = blk0; blk < nblk; blk++) {
        uint8_t *const tab_cur = tab[wave][blk & 1], *const tab_next = tab[wave][(blk + 1) & 1];
        typename F::Hdr hd_next;
        static_for(std::make_integer_sequence<int, NS>{}, [&](auto qc) __attribute__((always_inline)) {
            constexpr int q = decltype(qc)::value;
            constexpr int g = q / (2 * MT), ts = q % (2 * MT), mt = ts % MT;
            if constexpr (ts == 0) {
                // the stage after next goes to LDS, the one after that is requested
                stage_store(st, tokbuf(g + 2), g + 2, (blk + (g >= 2 ? 1 : 0)) & 1);
                st = stage_load(blk + (g >= 1 ? 1 : 0), (g + 3) & 3);
                if constexpr (g == 0) hd_next = F::load_hdr(rs_w, wrow, min(blk + 1, nblk - 1));
            }
            // operands of the sub-block that step q + 1 opens
            if constexpr (ts == MT - 1) F::template unpack<g, 1>(ql[g & 1], qh[F::NQH == 2 ? g >> 1 : 0], ck, mk, wf);
            if constexpr (ts == 2 * MT - 1) {
                if constexpr (F::NQH == 1 && g == 3) {
                    qh[0] = qh_next;
                    qh_next = F::fetch_qh(rs_w, wq_off, min(blk + 2, nblk - 1), 0);
                }
                constexpr int gn = (g + 1) & 3;
                F::template unpack<gn, 0>(ql[gn & 1], qh[F::NQH == 2 ? gn >> 1 : 0], ck, mk, wf);
            }
            {
                constexpr int q1 = q + 1;
                T[q1 & 1] = mfma_chain(tf[q1 & 1]);
            }
            {
                constexpr int q2 = q + 2;
                const uint8_t *const b2 = tokbuf(q2 / (2 * MT));
                tf[q & 1][0] = tok_frag(b2, q2 % (2 * MT), 0);
                tf[q & 1][1] = tok_frag(b2, q2 % (2 * MT), 1);
            }
            {
                constexpr int q1 = q + 1, t1 = q1 % (2 * MT);
                da[q1 & 1] = das[(q1 / (2 * MT)) & 3][t1 / MT][(t1 % MT) * 32 + c];
            }
            const float d = da[q & 1];
            const v16f t = T[q & 1];
#pragma unroll
            for (int i = 0; i < 16; i++) accblk[mt][i] = q < MT ? t[i] * d : fmaf(t[i], d, accblk[mt][i]);
            if constexpr (ts == MT - 1) ck = F::load_const(g == 3 ? tab_next : tab_cur, (g + 1) & 3, 0, c, h);
            if constexpr (ts == 2 * MT - 1) ck = F::load_const(g == 3 ? tab_next : tab_cur, (g + 1) & 3, 1, c, h);
            // (both sub-blocks of the group are unpacked: its slot takes the group after next)
            if constexpr (ts == MT) {
                ql[g & 1] = F::fetch_ql(rs_w, wq_off, g < 2 ? blk : min(blk + 1, nblk - 1), (g + 2) & 3);
                if constexpr (F::NQH == 2 && (g & 1) == 1) qh[g >> 1] = F::fetch_qh(rs_w, wq_off, min(blk + 1, nblk - 1), g >> 1);
                if constexpr (g == 1) F::decode(hd_next, tab_next, c, h);
            }
            if constexpr (q >= NS - MT) {
                // ---- the super-block's factors for token tile mt, whose last step this was:
                //      y += d * accblk - dmin * (mn . P) --------------------------------------------------------------
                v16f U;
                if constexpr (F::HAS_MIN) {
                    const uint8_t *const p = pl[blk & 1];
                    const b8 mn8 = lds_b8(tab_cur + F::T_MNB + c * 16);
                    const b8 pa = lds_b8(p + ((h * MT + mt) * 32 + c) * 16);
                    const b8 pb = lds_b8(p + (((2 + h) * MT + mt) * 32 + c) * 16);
                    U = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mn8, pa, zero16, 0, 0, 0);
                    U = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mn8, pb, U, 0, 0, 0);
                }
#pragma unroll
                for (int a = 0; a < 4; a++) {
                    const v4f dv = *reinterpret_cast<const lds_v4f *>(tab_cur + F::T_D + (8 * a + 4 * h) * 4);
                    v4f nv = {0.0f, 0.0f, 0.0f, 0.0f};
                    if constexpr (F::HAS_MIN) nv = *reinterpret_cast<const lds_v4f *>(tab_cur + F::T_NDM + (8 * a + 4 * h) * 4);
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        y[mt][4 * a + b] = fmaf(accblk[mt][4 * a + b], dv[b], y[mt][4 * a + b]);
                        if constexpr (F::HAS_MIN) y[mt][4 * a + b] = fmaf(U[4 * a + b], nv[b], y[mt][4 * a + b]);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ts == 2 * MT - 1) stage_end();
        });
    }

    uint32_t mt_first = 0, mt_last = MT;  // token tiles this wave stores
    if constexpr (KS > 1) {
        // a part with a super-block less: the barriers of the one it does not have
        for (uint32_t i = nblk - blk0; i < per_part; i++)
            for (int g = 0; g < 4; g++) stage_end();
        // The parts' sums meet in LDS (the stage buffers are free behind the last barrier): part p keeps token tiles
        // p MT / KS .. and gives the others away; sums are added in the order of k.
        constexpr int OWN = MT / KS;
        v4f *const red = reinterpret_cast<v4f *>(&tok_all[0][0][0]);  // [row wave][part][token tile][4][lane]
        static_assert(sizeof(tok_all) >= (size_t)RW * KS * MT * 4 * 64 * 16, "room for the parts' sums");
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int a = 0; a < 4; a++)
                red[(((wave * KS + part) * MT + mt) * 4 + a) * 64 + lane] =
                    v4f{y[mt][4 * a], y[mt][4 * a + 1], y[mt][4 * a + 2], y[mt][4 * a + 3]};
        __syncthreads();
        mt_first = part * OWN, mt_last = mt_first + OWN;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int a = 0; a < 4; a++) {
                if (mt < (int)mt_first || mt >= (int)mt_last) continue;
                v4f v = red[((wave * KS * MT + mt) * 4 + a) * 64 + lane];
#pragma unroll
                for (int p = 1; p < KS; p++) v = v + red[(((wave * KS + p) * MT + mt) * 4 + a) * 64 + lane];
                for (int b = 0; b < 4; b++) y[mt][4 * a + b] = v[b];
            }
    }

    if constexpr (DEAL) {
        if (nblk - blk0 != n_super) {  // a tile that others have runs of: the sums as they lie in the registers
            v4f *const to = reinterpret_cast<v4f *>(partial) + (size_t)slot * (TOK * ROWS / 4) + wave * (MT * 256) + lane;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int a = 0; a < 4 && m_wg + 32 * mt < m; a++)
                    to[(mt * 4 + a) * 64] = v4f{y[mt][4 * a], y[mt][4 * a + 1], y[mt][4 * a + 2], y[mt][4 * a + 3]};
            slot |= 1;
            continue;
        }
        if (dealt) slot |= 1;
    }
    // ---- store: lane (token c, half h) holds rows 8a + 4h + 0..3 of its wave's 32, for MT token tiles -----------------
    const bool vec4 = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 &&
                      (!bias || (reinterpret_cast<uintptr_t>(bias) & 15) == 0);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const uint32_t t = m_wg + mt * 32 + c;
        if (mt < (int)mt_first || mt >= (int)mt_last || t >= m) continue;
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const uint32_t row = n_wave + 8 * a + 4 * h;
            if (row >= n) continue;
            float *o = out + (size_t)t * n + row;
            if (vec4) {
                v4f v = {y[mt][4 * a], y[mt][4 * a + 1], y[mt][4 * a + 2], y[mt][4 * a + 3]};
                if (accumulate) {
                    const v4f old = *reinterpret_cast<const v4f *>(o);
                    v = old + v;
                } else if (bias) {
                    v = v + *reinterpret_cast<const v4f *>(bias + row);
                }
                *reinterpret_cast<v4f *>(o) = v;
            } else {
#pragma unroll
                for (int b = 0; b < 4; b++)
                    if (row + b < n)
                        o[b] = accumulate ? o[b] + y[mt][4 * a + b] : bias ? y[mt][4 * a + b] + bias[row + b] : y[mt][4 * a + b];
            }
        }
    }
    } while (DEAL && (whole || unit < unit_end));
}

// The sums of the tiles that several work groups had runs of, added in the order of k: a work group here takes the 32 rows
// of one wave against one token tile, a thread four rows of a token, so that a token's 128 bytes are stored together.
template <int MT, int RW>
__global__ __launch_bounds__(256) void gemm_f16_deal_sum(const float *__restrict__ partial, float *__restrict__ out, uint32_t m,
                                                         uint32_t n, uint32_t n_super, int accumulate,
                                                         const float *__restrict__ bias, uint32_t m_tiles, uint32_t n_tiles,
                                                         uint32_t groups) {
    constexpr uint32_t TOK = 32 * MT, ROWS = 32 * RW;
    const uint32_t tile = blockIdx.x / (RW * MT), at = blockIdx.x % (RW * MT), wave = at / MT, mt = at % MT;
    const uint32_t tile0 = m_tiles * n_tiles / groups * groups;  // the whole rounds before the deal
    const uint32_t units = (m_tiles * n_tiles - tile0) * n_super;
    const uint32_t first = deal_owner(tile * n_super, groups, units), last = deal_owner(tile * n_super + n_super - 1, groups, units);
    if (first == last) return;  // stored by the one work group that had all of it
    const uint32_t c = threadIdx.x >> 3, piece = threadIdx.x & 7;  // token c, rows 4 piece ..: register group piece / 2, half piece % 2
    const uint32_t n_tile = (tile0 + tile) / m_tiles, t = (tile0 + tile - n_tile * m_tiles) * TOK + mt * 32 + c, row = n_tile * ROWS + wave * 32 + piece * 4;
    if (t >= m || row >= n) return;
    const v4f *const p = reinterpret_cast<const v4f *>(partial) + (wave * MT + mt) * 256 + (piece >> 1) * 64 + (piece & 1) * 32 + c;
    v4f y = p[(size_t)deal_slot(first, tile * n_super, groups, units) * (TOK * ROWS / 4)];
    // (behind the first a work group's run began inside this tile: its first slot.  Four loads in flight, added in order)
    for (uint32_t w = first + 1; w <= last; w += 4) {
        v4f v[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) v[i] = p[(size_t)(2 * min(w + i, last)) * (TOK * ROWS / 4)];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++)
            if (w + i <= last) y = y + v[i];
    }
    float *const o = out + (size_t)t * n + row;
    if ((n & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 && (!bias || (reinterpret_cast<uintptr_t>(bias) & 15) == 0)) {
        if (accumulate)
            y = *reinterpret_cast<const v4f *>(o) + y;
        else if (bias)
            y = y + *reinterpret_cast<const v4f *>(bias + row);
        *reinterpret_cast<v4f *>(o) = y;
    } else {
        for (int b = 0; b < 4; b++)
            if (row + b < n) o[b] = accumulate ? o[b] + y[b] : bias ? y[b] + bias[row + b] : y[b];
    }
}

// One work group per compute unit, the same number on each XCD.
uint32_t f16_deal_groups() { return device_cus() < 16 ? 8 : device_cus() / 8 * 8; }

template <class F>
hipError_t launch_f16_deal(const GemmArgs &a, float *partial, hipStream_t stream) {
    constexpr int MT = 4, RW = 8;
    const uint32_t m_tiles = (a.m + 32 * MT - 1) / (32 * MT), n_tiles = (a.n + 32 * RW - 1) / (32 * RW), groups = f16_deal_groups();
    // (every run has a unit, so that the work groups between a tile's first and last have all left sums)
    const uint32_t rest = m_tiles * n_tiles % groups;
    if (rest && (uint64_t)rest * (a.k / 256) < groups) return hipErrorNotSupported;
    note_launch("gemm_f16_deal_kernel", F::TYPE, MT, RW, 1, 0, groups, 1, 64 * RW);
    hipLaunchKernelGGL((gemm_f16_kernel<F, MT, RW, 1, true>), dim3(groups), dim3(64 * RW), 0, stream, a.W, a.A, a.out, a.m, a.n,
                       a.k, a.accumulate, a.bias, m_tiles, n_tiles, partial);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || m_tiles * n_tiles % groups == 0) return e;
    hipLaunchKernelGGL((gemm_f16_deal_sum<MT, RW>), dim3(m_tiles * n_tiles % groups * MT * RW), dim3(256), 0, stream, partial, a.out, a.m,
                       a.n, a.k / 256, a.accumulate, a.bias, m_tiles, n_tiles, groups);
    return hipGetLastError();
}

template <class F, int MT, int RW, int KS>
hipError_t launch_f16_shape(const GemmArgs &a, hipStream_t stream) {
    const uint32_t m_tiles = (a.m + 32 * MT - 1) / (32 * MT), n_tiles = (a.n + 32 * RW - 1) / (32 * RW);
    const dim3 grid(tile_order_grid(m_tiles, n_tiles));
    note_launch("gemm_f16_kernel", F::TYPE, MT, RW, KS, 0, grid.x, 1, 64 * RW * KS);
    hipLaunchKernelGGL((gemm_f16_kernel<F, MT, RW, KS, false>), grid, dim3(64 * RW * KS), 0, stream, a.W, a.A, a.out, a.m, a.n, a.k,
                       a.accumulate, a.bias, m_tiles, n_tiles, nullptr);
    return hipGetLastError();
}

// (the large shape of Q4_K is for the fixed-shape knob alone: those calls go to the prefill kernel)
template <class F>
hipError_t launch_f16(const GemmArgs &a, int shape, hipStream_t stream) {
    return shape == 1 ? launch_f16_shape<F, 4, 8, 1>(a, stream) : launch_f16_shape<F, 2, 4, 2>(a, stream);
}

}  // namespace

bool gemm_f16_supported(uint32_t type, uint32_t m, uint32_t n, uint32_t k) {
    if ((type != OXQ_TYPE_Q4_K && type != OXQ_TYPE_Q5_K && type != OXQ_TYPE_Q6_K) || k == 0 || k % 256 != 0 || m == 0 || n == 0)
        return false;
    // 32-bit offsets inside a work group's rows and tokens
    return (size_t)k / 256 * 210 * 256 < 0x7FFFFFFFull && (size_t)k / 32 * 34 * 128 < 0x7FFFFFFFull;
}

// Which shape of this kernel a plain matmul takes; 0: the other kernels serve it better.  A work group takes its time
// whatever its neighbours do, so what counts is how the grid fills its rounds of the chip.  One round at k = 4096: Q6_K
// 110-130 us (large shape) and 47-54 (small), Q5_K 100-108 and 41-48, Q4_K 92-100 and 36-42; a round with rows and columns to
// spare costs as much as a full one.
// Q6_K, whose tile kernel takes four vector instructions per result where this one takes one: either shape once its
// grid is three quarters full (768 x 4096 x 4096 95 us against 103; in one round of the small shape 192 tiles are a tie, 51
// against 50, and 206 win, 52 against 62), the large one from 64 % on in a single round (333 x 14336 x 4096 115 against 145).
// Two rounds of the small shape up to 384 rows, where the tile kernel splits k inside work groups of 64 x 32 and keeps
// the chip full: from 82 % on (384 tiles: 256 x 12288 x 4096 93 against 82, 384 x 8192 x 8192 176 against 153, x 3072 72 against
// 66; 420 tiles, 333 x 8960 x 1536, 42 against 47; 432, 256 x 13824 x 5120, a tie).
// Q4_K and Q5_K, whose tile kernel is about as fast per result: only full rounds, the large shape of Q5_K (Q4_K has the
// prefill kernel there) and the small one in a single round (512 x 4096 x 4096, 256 tiles, Q4_K 40 against 45, Q5_K 44 against
// 50; with 208 to 240 tiles 39-40 against 40-41 and 43-44 against 45, with 192 it loses, 37 against 34; 264 tiles, two rounds,
// 72 against 62 and 80 against 73) of more than 384 rows: up to there the tile kernel's own tiles fill the chip as well (256
// tiles at k = 4096 / 8192, 128 rows Q4_K 41 / 77 against 41 / 75, Q5_K 45 / 89 against 46 / 89, 256 rows Q4_K 40 / 76 against 40 /
// 73, Q5_K 44 / 83 against 45 / 83; only on rows of 1024 columns this one wins, 16 against 19).
int gemm_f16_shape(uint32_t type, uint32_t m, uint32_t n, uint32_t k) {
    if (!gemm_f16_supported(type, m, n, k) || k < 1024) return 0;
    const uint64_t cus = device_cus();
    const uint64_t large = (uint64_t)((m + 127) / 128) * ((n + 255) / 256), small = (uint64_t)((m + 63) / 64) * ((n + 127) / 128);
    const uint64_t rl = (large + cus - 1) / cus, rs = (small + cus - 1) / cus;
    // (token tiles mostly in use: a work group costs the same with a few of its token rows)
    const bool large_ok = 100 * (uint64_t)m >= 70 * 128 * ((m + 127) / 128), small_ok = m > 64 && 100 * (uint64_t)m >= 80 * 64 * ((m + 63) / 64);
    if (type == OXQ_TYPE_Q6_K) {
        if (large_ok && rl * 130 <= rs * 54) return 100 * large >= (rl == 1 ? 64u : 72u) * rl * cus ? 1 : 0;
        return small_ok && 100 * small >= (rs == 1 ? 80u : rs == 2 && m <= 384 ? 82u : 74u) * rs * cus ? 2 : 0;
    }
    if (type == OXQ_TYPE_Q5_K && large_ok && 100 * large >= 96 * rl * cus && (rl == 1 || k >= 8192)) return 1;
    return small_ok && rs == 1 && 100 * small >= 96 * cus && m > 384 ? 2 : 0;
}

// Whether a call takes the even deal: where its time, estimated, is less than that of the kernel that the call would take
// otherwise.  Both are lines through measured times (294 calls with 40 to 2048 rows, 768 to 28672 weight rows and columns):
//   the deal     17 / 20 / 21 us (Q4_K / Q5_K / Q6_K) for the ramp, the exchange of up to 64 MB of sums and the second launch,
//                6.9 / 7.4 / 9.5 per super-block of the longest run, 8 where whole tiles go before the runs
//   the others   a time per round of the chip and 4096 columns, the least that was measured for the shape (the calls with
//                short rows and partly used tiles take up to a third more): the prefill kernel 90, this kernel's whole
//                tiles 100 / 122 (Q5_K / Q6_K) and 38 / 43 / 45.6 (small), the tile kernel 57 / 57 / 88 (128 x 128 tiles), 30 / 33
//                / 53 (128 x 64), 33 / 37.5 / 50 (64 x 128), 9.7 / 11.3 / 14.7 (64 x 32, k split)
// so that the line errs towards the kernels with whole tiles.  On 529 other calls (profiles/even_deal_against_other_kernels.txt) four
// estimates of the deal in five are within 10 %, the mean over the calls is 8 % less than without the deal, the best choice of
// each 9 % less, and the worst of the 208 calls that take it loses 5 % (Q4_K 200 x 14336 x 4096 64 us, 61).  us, without and with it: Q4_K
// 333 x 11008 x 4096 77 and 75, 1100 x 4096 x 14336 390 and 221, 512 x 4096 x 14336 121 and 102; Q5_K 333 x 11008 x 4096 92 and 81; Q6_K
// 333 x 4096 x 11008 127 and 96, 768 x 4096 x 14336 324 and 206, 1100 x 4096 x 4096 143 and 102.  Q4_K 333 x 4096 x 4096, where runs are three
// super-blocks, stays (33, 40).
bool gemm_f16_deal_pays(uint32_t type, uint32_t m, uint32_t n, uint32_t k) {
    // (a token tile half empty, against 32-token tiles.  Matrices narrower than a tile: not for the time, which the deal would
    // more than halve on long rows -- 333 x 128 x 28672 Q4_K 74 us against 32, 1024 x 192 x 14336 Q6_K 59 against 34 -- but because
    // there a call's fp32 sums are those of the integer sums' dump, bit for bit, and are held to it)
    if (!gemm_f16_supported(type, m, n, k) || m <= 64 || n < 256) return false;
    const int f = type == OXQ_TYPE_Q4_K ? 0 : type == OXQ_TYPE_Q5_K ? 1 : 2;
    const uint64_t groups = f16_deal_groups(), cus = device_cus(), n_super = k / 256;
    const uint64_t tiles = tile_count(m, n, 128, 256), whole = tiles / groups, rest = tiles % groups;
    if (rest * n_super < groups) return false;
    // tenths of a microsecond
    static constexpr uint32_t RAMP[3] = {175, 203, 209}, RUN[3] = {69, 74, 95};
    const uint64_t deal = RAMP[f] + RUN[f] * (whole * n_super + (rest * n_super + groups - 1) / groups) + (whole ? 80 : 0);
    static constexpr uint32_t PREFILL = 900, LARGE[3] = {0, 1000, 1220}, SMALL[3] = {380, 430, 456}, T128X128[3] = {570, 570, 880},
                              T128X64[3] = {300, 330, 530}, T64X128[3] = {330, 375, 500}, T64X32[3] = {97, 113, 147};
    uint64_t per_round, wgs;
    if (gemm_prefill_supported(type, m, n, k) && gemm_prefill_pays(m, n)) {
        per_round = PREFILL, wgs = tiles;
    } else if (const int shape = gemm_f16_shape(type, m, n, k)) {
        per_round = shape == 1 ? LARGE[f] : SMALL[f], wgs = shape == 1 ? tiles : tile_count(m, n, 64, 128);
    } else if (tile_big(m, n, k, 1, cus)) {
        const bool square = tile_square(type, tile_count(m, n, 128, 128), k, cus);
        per_round = square ? T128X128[f] : T128X64[f], wgs = tile_count(m, n, 128, square ? 128 : 64);
    } else if (tile_scales_fit(k, 64)) {
        const bool wide = !tile_narrow(m, n, k, 1, cus) && tile_mid_wide(32 * tile_count(m, n, 64, 128), cus);
        per_round = wide ? T64X128[f] : T64X32[f], wgs = tile_count(m, n, 64, wide ? 128 : 32);
    } else {
        return false;
    }
    return deal * 4096 < per_round * ((wgs + cus - 1) / cus) * k;
}

size_t gemm_f16_deal_bytes() { return (size_t)2 * f16_deal_groups() * (128 * 256 * sizeof(float)); }

hipError_t launch_gemm_f16_deal(uint32_t type, const GemmArgs &a, float *partial, hipStream_t stream) {
    if (!gemm_f16_supported(type, a.m, a.n, a.k) || a.offsets || a.sums) return hipErrorNotSupported;
    switch (type) {
    case OXQ_TYPE_Q4_K: return launch_f16_deal<F16Q4K>(a, partial, stream);
    case OXQ_TYPE_Q5_K: return launch_f16_deal<F16Q5K>(a, partial, stream);
    default: return launch_f16_deal<F16Q6K>(a, partial, stream);
    }
}

hipError_t launch_gemm_f16(uint32_t type, const GemmArgs &a, int shape, hipStream_t stream) {
    if (!gemm_f16_supported(type, a.m, a.n, a.k) || a.offsets || a.sums) return hipErrorNotSupported;
    switch (type) {
    case OXQ_TYPE_Q4_K: return launch_f16<F16Q4K>(a, shape, stream);
    case OXQ_TYPE_Q5_K: return launch_f16<F16Q5K>(a, shape, stream);
    default: return launch_f16<F16Q6K>(a, shape, stream);
    }
}

}  // namespace oxq
