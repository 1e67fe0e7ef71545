// Few tokens per weight matrix, weights straight from memory into the matrix core's registers: the batched fused matvec
//   out[m x n] (+)= A_q8[m rows of Q8_0 blocks] x W[n x k]^T
// (the reference's gemm loop over matvec_q8_fused, crates/oxillama-quant/src/reference/q4_k.rs:186-201, :218-333) for a
// decode batch or a short prompt on one matrix, where its few tiles of 16 rows x 16 tokens make the launch's ramp and the
// chain along k the time (77 rows of Q4_0: 1536 x 1536 12.2 us on the tile kernel, 5.6 here; 8960 x 1536 22.3 / 12.2).
//
//  * k is dealt to the waves of a work group, PB super-blocks each, and a wave keeps its part of the tokens in registers, in
//    operand order, for as long as the work group walks tiles of 16 weight rows: nothing about the tokens is read again.
//    The parts' sums meet in LDS, in the order of k, so there is no reduction launch.
//  * A work group takes TT tiles of 16 tokens: the weights are unpacked once for them.  More tokens are further work groups' (grid y).
//  * Weights: four lanes share a row; a lane loads 16 bytes of each 64 of a super-block.  Those are 16 weights of one or two
//    sub-blocks where the operand needs 8 of every sub-block from each of the four: two or four v_permlane{32,16}_swap
//    per 16 bytes put them there.  No LDS on the way.
//  * v_mfma_i32_16x16x32_i8 with the weights as the A operand: lane (c = l % 16, q = l / 16) supplies k-slots 8q..8q+7 of
//    row c and of token c and receives rows 4q..4q+3 against token c.  A token's scale is one register per sub-block;
//    the rows' factors, decoded by lane (c, q) for row c, reach the lanes that need them through a small LDS table.
// Arithmetic per result as in the tile kernel (oxq_gemm_tile.hpp): fl(dsc * isum) by the 1.5 * 2^23 trick, then one fma with the token's
// scale, so that an infinite one keeps its infinities (the trick on the token's side, one constant per token instead of
// four per lane and sub-block, makes them NaN: inf - inf; a decode batch of 16 rows through an 8B model's layer 74.3 us that way, 75.3 this way);
// the zero-point term as a 16 x 16 x 4 fp32 MFMA per four sub-blocks.
#pragma once
#include "oxq_gemm_tile.hpp"
#include "oxq_direct_window.hpp"

namespace oxq {

#define OXQ_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))
typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef float v4f32 __attribute__((ext_vector_type(4)));

// a = (a of lanes 0..31, b of lanes 0..31), b = (a of lanes 32..63, b of lanes 32..63)
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
// the same inside each half of the wave: a = (row 0 of a, row 0 of b, row 2 of a, row 2 of b), b the odd rows
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}
// Lanes q = 0, 1 hold the halves of one run of 32 bytes, q = 2, 3 those of the next: afterwards w[0], w[1] are 8 bytes of the
// first run in every lane (bytes 0, 16, 8, 24 on for q = 0 .. 3), w[2], w[3] of the second.
__device__ __forceinline__ void spread_runs(u32x4 &w) {
    uint32_t a = w[0], b = w[1], c = w[2], d = w[3];
    swap32(a, c), swap32(b, d);
    w = u32x4{a, b, c, d};
}
// Lane q holds the 16 bytes of piece q: afterwards w[j] is dword q of piece j.
__device__ __forceinline__ void transpose_pieces(u32x4 &w) {
    uint32_t a = w[0], b = w[1], c = w[2], d = w[3];
    swap32(a, c), swap32(b, d);
    swap16(a, b), swap16(c, d);
    w = u32x4{a, b, c, d};
}
__device__ __forceinline__ long i8x8(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

// Per format:
//   BLOCK      bytes of 256 weights
//   KS         scale factors per sub-block (two: of 16 weights each)
//   HAS_MIN    a zero-point term
//   TIMES      what the operand is a multiple of (a power of two that the factors take out again)
//   OFFSET     what the dump of the integer sums has added to every weight
//   ORDER      which of a block's token bytes the k-slots of lane q hold: 0 the eight from 8 * {0, 2, 1, 3}[q] on; 1 the eight
//              from 8 q on, even ones first
//   W, load    the lane's bytes of a super-block (at byte `so` of the row that starts at `row`): lane q's share, LOADS
//              buffer loads
//   arrange    the exchange between the lanes that share a row
//   operand    8 int8 weights of sub-block s
//   factors    KS = 1: the scale factors of sub-blocks q and q + 4 of row c and (HAS_MIN) their zero-point factors
//              KS = 2: the factors 4 q .. 4 q + 3 of the row's sixteen
template <class F>
struct Direct {
    static constexpr bool OK = false;
};

template <>
struct Direct<TileQ4K> {  // reference/q4_k.rs:27-99
    static constexpr bool OK = true, HAS_MIN = true;
    static constexpr uint32_t BLOCK = 144, LOADS = 3;
    static constexpr int KS = 1, ORDER = 0, TIMES = 1, OFFSET = 0;
    struct W {
        u32x4 hdr, qs[2];
    };
    static __device__ __forceinline__ void load(W &w, __amdgpu_buffer_rsrc_t rs, uint32_t row, uint32_t q, uint32_t so) {
#pragma unroll
        for (int i = 0; i < 2; i++) w.qs[i] = buf16(rs, row + 16 * q, so + 16 + 64 * i);
        w.hdr = buf16(rs, row, so);
    }
    static __device__ __forceinline__ void arrange(W &w, uint32_t) { spread_runs(w.qs[0]), spread_runs(w.qs[1]); }
    static __device__ __forceinline__ long operand(const W &w, int s) {
        const u32x4 v = w.qs[s >> 2];
        const uint32_t a = v[s & 2], b = v[(s & 2) + 1];
        return (s & 1) ? i8x8((a >> 4) & 0x0F0F0F0Fu, (b >> 4) & 0x0F0F0F0Fu) : i8x8(a & 0x0F0F0F0Fu, b & 0x0F0F0F0Fu);
    }
    static __device__ __forceinline__ void factors(const W &w, uint32_t q, float (&f)[2], float (&z)[2]) {
        const uint32_t a = w.hdr[1] >> (8 * q), b = w.hdr[2] >> (8 * q), c = w.hdr[3] >> (8 * q);
        const float d = h2f(w.hdr[0] & 0xFFFF), ndmin = -h2f(w.hdr[0] >> 16);
        f[0] = d * (float)(a & 63);
        f[1] = d * (float)((c & 15) | ((a >> 2) & 48));
        z[0] = ndmin * (float)(b & 63);
        z[1] = ndmin * (float)(((c >> 4) & 15) | ((b >> 2) & 48));
    }
};

// The 32-weight formats' blocks of 18 and 34 bytes, and Q6_K's of 210, start on a dword in turn.  Loads start on the dword at or
// below the first byte (a 16-byte load off a dword takes 48 cycles of a compute unit's texture unit where an aligned one of this
// pattern takes 24: 57344 x 4096 of Q6_K, sixteen rows, 62 us, and 49 with the same bytes on dwords), the bytes are moved
// down by shift / 8 afterwards.  next: the dword behind the 16 bytes.
__device__ __forceinline__ u32x4 from_dword(const u32x4 w, uint32_t next, uint32_t shift) {
    return u32x4{__builtin_amdgcn_alignbit(w[1], w[0], shift), __builtin_amdgcn_alignbit(w[2], w[1], shift),
                 __builtin_amdgcn_alignbit(w[3], w[2], shift), __builtin_amdgcn_alignbit(next, w[3], shift)};
}
// s[i] in rows 0 .. 3 of the wave, x behind them, as one sequence of seventeen: every element replaced by its successor.
__device__ __forceinline__ void successors(uint32_t (&s)[4], uint32_t x) {
    swap32(s[0], s[2]), swap32(s[1], s[3]), swap16(s[0], s[1]), swap16(s[2], s[3]);  // row i of s[j]: row j of s[i]
    uint32_t a = s[0], b = s[0], c = s[0];
    swap16(a, b);  // b: rows 1, 1, 3, 3
    swap32(c, x);  // x: rows 2, 3, x, x
    swap16(b, x);  // b: rows 1, 2, 3, x
    s[0] = s[1], s[1] = s[2], s[2] = s[3], s[3] = b;
    swap32(s[0], s[2]), swap32(s[1], s[3]), swap16(s[0], s[1]), swap16(s[2], s[3]);
}

// Q6_K (reference/q6_k.rs:25-75): the operand is 4 (q - 32), which fits a byte with its sign: the low nibble at bits 2 .. 5,
// the upper two bits at 6 and 7, the topmost inverted; a quarter of the scale takes the 4 out again (both exact).  Each half of
// 16 weights has its scale, so each is an MFMA of its own with the other half's lanes (q even: the first half) supplying zeros.
template <>
struct Direct<TileQ6K> {
    static constexpr bool OK = true, HAS_MIN = false;
    static constexpr uint32_t BLOCK = 210, LOADS = 5;
    static constexpr int KS = 2, ORDER = 0, TIMES = 4, OFFSET = 0;
    struct W {
        u32x4 ql[2], qh;
        uint32_t sc, d, shift;
    };
    static __device__ __forceinline__ void load(W &w, __amdgpu_buffer_rsrc_t rs, uint32_t row, uint32_t q, uint32_t so) {
        const uint32_t at = (row + so) & ~3u;
        w.shift = ((row + so) & 2) * 8;
#pragma unroll
        for (int i = 0; i < 2; i++) w.ql[i] = buf16(rs, at + 16 * q, 64 * i);
        w.qh = buf16(rs, at + 16 * q, 128);
        w.sc = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, at + 4 * q, 192, 0);
        w.d = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, at, 208, 0);  // its low half, or with the scales' last two before it the upper
    }
    static __device__ __forceinline__ void arrange(W &w, uint32_t) {
        uint32_t next[4] = {w.ql[0][0], w.ql[1][0], w.qh[0], w.sc};
        successors(next, w.d);
        w.ql[0] = from_dword(w.ql[0], next[0], w.shift), w.ql[1] = from_dword(w.ql[1], next[1], w.shift);
        w.qh = from_dword(w.qh, next[2], w.shift);
        w.sc = __builtin_amdgcn_alignbit(next[3], w.sc, w.shift);
        w.d >>= w.shift;
        spread_runs(w.ql[0]), spread_runs(w.ql[1]), spread_runs(w.qh);
        for (int i = 0; i < 4; i++) w.qh[i] ^= 0xAAAAAAAAu;  // the topmost bit of every field
    }
    static __device__ __forceinline__ long operand(const W &w, int s) {
        const int hh = s >> 2, p = s & 1, e = (s >> 1) & 1, sh = 2 * p + 4 * e;
        uint32_t v[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t l = w.ql[hh][2 * p + i], h = w.qh[2 * hh + i];
            v[i] = ((e ? l >> 2 : l << 2) & 0x3C3C3C3Cu) | ((h << (6 - sh)) & 0xC0C0C0C0u);
        }
        return i8x8(v[0], v[1]);
    }
    static __device__ __forceinline__ void factors(const W &w, float (&f)[4]) {
        const float d = 0.25f * h2f(w.d & 0xFFFF);
#pragma unroll
        for (int b = 0; b < 4; b++) f[b] = d * (float)(int)(int8_t)((w.sc >> (8 * b)) & 0xFF);
    }
};

// IQ4_XS (reference/iq4_xs.rs:47-97): a lane takes the 16 bytes of sub-blocks q and q + 4.
template <>
struct Direct<TileIQ4XS> {
    static constexpr bool OK = true, HAS_MIN = false;
    static constexpr uint32_t BLOCK = 136, LOADS = 3;
    static constexpr int KS = 1, ORDER = 1, TIMES = 1, OFFSET = 0;
    struct W {
        u32x4 qs[2];
        u32x2 hdr;
    };
    static __device__ __forceinline__ void load(W &w, __amdgpu_buffer_rsrc_t rs, uint32_t row, uint32_t q, uint32_t so) {
#pragma unroll
        for (int i = 0; i < 2; i++) w.qs[i] = buf16(rs, row + 16 * q, so + 8 + 64 * i);
        w.hdr = __builtin_amdgcn_raw_buffer_load_b64(rs, row, so, 0);
    }
    static __device__ __forceinline__ void arrange(W &w, uint32_t) { transpose_pieces(w.qs[0]), transpose_pieces(w.qs[1]); }
    static __device__ __forceinline__ long operand(const W &w, int s) {
        const uint32_t v = w.qs[s >> 2][s & 3];
        return i8x8(FmtIQ4XS::lut4(v & 0x0F0F0F0Fu), FmtIQ4XS::lut4((v >> 4) & 0x0F0F0F0Fu));
    }
    static __device__ __forceinline__ void factors(const W &w, uint32_t q, float (&f)[2], float (&)[2]) {
        const float d = h2f(w.hdr[0] & 0xFFFF);
#pragma unroll
        for (uint32_t i = 0; i < 2; i++) {
            const uint32_t s = q + 4 * i;
            const uint32_t low = (w.hdr[1] >> (4 * s)) & 15, high = (w.hdr[0] >> (16 + 2 * s)) & 3;
            f[i] = d * (float)((int)(low | (high << 4)) - 32);
        }
    }
};

struct DirectQ5K {
    static constexpr uint32_t TYPE = OXQ_TYPE_Q5_K;
};
// Q5_K (reference/q5_k.rs): Q4_K's header, 32 bytes of fifth bits (bit g of byte l: weight l of run g's low nibbles, bit g + 4:
// of its high ones), four runs of nibbles.
template <>
struct Direct<DirectQ5K> {
    static constexpr bool OK = true, HAS_MIN = true;
    static constexpr uint32_t BLOCK = 176, LOADS = 4;
    static constexpr int KS = 1, ORDER = 0, TIMES = 1, OFFSET = 0;
    struct W {
        u32x4 hdr, qs[2];
        u32x2 qh;
    };
    static __device__ __forceinline__ void load(W &w, __amdgpu_buffer_rsrc_t rs, uint32_t row, uint32_t q, uint32_t so) {
#pragma unroll
        for (int i = 0; i < 2; i++) w.qs[i] = buf16(rs, row + 16 * q, so + 48 + 64 * i);
        w.hdr = buf16(rs, row, so);
        w.qh = __builtin_amdgcn_raw_buffer_load_b64(rs, row + 16 * (q & 1) + 8 * (q >> 1), so + 16, 0);  // its share of every run
    }
    static __device__ __forceinline__ void arrange(W &w, uint32_t) { spread_runs(w.qs[0]), spread_runs(w.qs[1]); }
    static __device__ __forceinline__ long operand(const W &w, int s) {
        const int bit = (s >> 1) + 4 * (s & 1);
        uint32_t v[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t l = w.qs[s >> 2][(s & 2) + i], h = w.qh[i];
            v[i] = ((s & 1 ? l >> 4 : l) & 0x0F0F0F0Fu) | ((bit <= 4 ? h << (4 - bit) : h >> (bit - 4)) & 0x10101010u);
        }
        return i8x8(v[0], v[1]);
    }
    static __device__ __forceinline__ void factors(const W &w, uint32_t q, float (&f)[2], float (&z)[2]) {
        Direct<TileQ4K>::W k;
        k.hdr = w.hdr;
        Direct<TileQ4K>::factors(k, q, f, z);
    }
};

// (Blocks of 18 and 34 bytes: with an even block, whose payload starts two bytes into a dword, and the odd one behind it, whose
// payload starts on one, the dword in which the even block ends also holds the odd one's scale.)

// Q4_0 (reference/q4_0.rs:22-49): eight blocks of 18 bytes stand for a super-block; a lane takes the nibbles of blocks q and
// q + 4.  The operand is 16 (n - 8), the nibble at bits 4 .. 7 with the topmost inverted: no zero-point term, which would cost an
// infinite token its infinities (the GEMV that serves fewer rows has them) and sums as exact as integers are.  The dump is
// the other kernels', of the unsigned nibbles.
template <>
struct Direct<TileQ4_0> {
    static constexpr bool OK = true, HAS_MIN = false;
    static constexpr uint32_t BLOCK = 144, LOADS = 4;
    static constexpr int KS = 1, ORDER = 1, TIMES = 16, OFFSET = 8;
    struct W {
        u32x4 qs[2];
        uint32_t x[2];
        uint32_t d[2];
    };
    static __device__ __forceinline__ void load(W &w, __amdgpu_buffer_rsrc_t rs, uint32_t row, uint32_t q, uint32_t so) {
        const uint32_t pair = row + 36 * (q >> 1);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            w.qs[i] = buf16(rs, pair + 20 * (q & 1), so + 72 * i);
            w.x[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, pair, so + 72 * i + 16, 0);
        }
    }
    static __device__ __forceinline__ void arrange(W &w, uint32_t q) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            w.d[i] = q & 1 ? w.x[i] >> 16 : w.qs[i][0] & 0xFFFF;
            w.qs[i] = from_dword(w.qs[i], w.x[i], q & 1 ? 0 : 16);
            transpose_pieces(w.qs[i]);
            for (int j = 0; j < 4; j++) w.qs[i][j] ^= 0x88888888u;
        }
    }
    static __device__ __forceinline__ long operand(const W &w, int s) {
        const uint32_t v = w.qs[s >> 2][s & 3];
        return i8x8((v << 4) & 0xF0F0F0F0u, v & 0xF0F0F0F0u);
    }
    static __device__ __forceinline__ void factors(const W &w, uint32_t, float (&f)[2], float (&)[2]) {
#pragma unroll
        for (int i = 0; i < 2; i++) f[i] = 0.0625f * h2f(w.d[i]);
    }
};

// Q8_0 weights (reference/q8_0.rs:22-47): 34 bytes a block; four lanes take the halves of two blocks at a time.
template <>
struct Direct<TileQ8_0> {
    static constexpr bool OK = true, HAS_MIN = false;
    static constexpr uint32_t BLOCK = 272, LOADS = 8;
    static constexpr int KS = 1, ORDER = 0, TIMES = 1, OFFSET = 0;
    struct W {
        u32x4 qs[4];
        uint32_t x[4];
        uint32_t d[2];
    };
    static __device__ __forceinline__ void load(W &w, __amdgpu_buffer_rsrc_t rs, uint32_t row, uint32_t q, uint32_t so) {
        const uint32_t at = row + 16 * (q & 1) + 36 * (q >> 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            w.qs[i] = buf16(rs, at, so + 68 * i);
            w.x[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, row, so + 68 * i + 32, 0);
        }
    }
    static __device__ __forceinline__ void arrange(W &w, uint32_t q) {
        // the scales of blocks q and q + 4: an odd block's is in the dword between the two, an even one's where lane q = 0 loaded
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t a = w.qs[2 * i][0], b = w.qs[2 * i + 1][0];
            swap32(a, b);  // a: that of pair 2 i in row 0, of pair 2 i + 1 in row 2
            const uint32_t x0 = w.x[2 * i], x1 = w.x[2 * i + 1], odd = q & 2 ? x1 : x0;
            w.d[i] = q & 1 ? odd >> 16 : a & 0xFFFF;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // behind the first half lies the second's first dword, behind that the one between the blocks
            uint32_t a = w.qs[i][0], next = w.x[i];
            swap16(a, next);
            w.qs[i] = from_dword(w.qs[i], next, q & 2 ? 0 : 16);
            spread_runs(w.qs[i]);
        }
    }
    static __device__ __forceinline__ long operand(const W &w, int s) {
        return i8x8(w.qs[s >> 1][2 * (s & 1)], w.qs[s >> 1][2 * (s & 1) + 1]);
    }
    static __device__ __forceinline__ void factors(const W &w, uint32_t, float (&f)[2], float (&)[2]) {
#pragma unroll
        for (int i = 0; i < 2; i++) f[i] = h2f(w.d[i]);
    }
};

// LDS floats of an exchanged 16 x 16 tile: rows 4q .. 4q + 3 against token c at q * EX_Q + 4 c
constexpr uint32_t EX_Q = 80, EX_TILE = 4 * EX_Q;
// LDS of a work group: the waves' factor tables (two super-blocks' in turn), their tokens' strips, the exchange (twice, in turn),
// which lies over the strips where there is no room beside them
template <class F, int WAVES>
constexpr uint32_t direct_tables() { return WAVES * 2 * 8 * Direct<F>::KS * 16 * 4; }
template <int PB, int TT, int WAVES>
constexpr uint32_t direct_strips() { return WAVES * 1024 * ((17 * PB * 16 * TT + 63) / 64); }
// row tiles of a wave whose sums are exchanged at once (what a barrier costs is shared), as LDS and registers allow
template <int TT, int WAVES>
constexpr int direct_turn() { return TT <= 2 && WAVES == 8 ? 2 : 1; }
template <int TT, int XT, int WAVES>
constexpr uint32_t direct_exchange() { return 2 * WAVES * TT * XT * EX_TILE * 4; }
template <class F, int PB, int TT, int WAVES>
constexpr bool direct_exchange_apart() {
    return direct_tables<F, WAVES>() + direct_strips<PB, TT, WAVES>() + direct_exchange<TT, direct_turn<TT, WAVES>(), WAVES>() <= 160 * 1024;
}
template <class F, int TT, int WAVES>
constexpr bool direct_streamed_apart() {
    return direct_tables<F, WAVES>() + direct_strips<1, TT, WAVES>() + direct_exchange<TT, 1, WAVES>() <= 160 * 1024;
}
template <class F, int TT, int WAVES>
constexpr uint32_t direct_streamed_lds() {
    constexpr uint32_t s = direct_strips<1, TT, WAVES>(), e = direct_exchange<TT, 1, WAVES>();
    return direct_tables<F, WAVES>() + (direct_streamed_apart<F, TT, WAVES>() ? s + e : s > e ? s : e);
}
template <class F, int PB, int TT, int WAVES>
constexpr uint32_t direct_lds() {
    constexpr uint32_t s = direct_strips<PB, TT, WAVES>(), e = direct_exchange<TT, direct_turn<TT, WAVES>(), WAVES>();
    return direct_tables<F, WAVES>() + (direct_exchange_apart<F, PB, TT, WAVES>() ? s + e : s > e ? s : e);
}

struct __attribute__((may_alias)) lds_f1 { float v; };
struct __attribute__((may_alias)) lds_f4 { v4f32 v; };
struct __attribute__((may_alias)) lds_q4 { u32x4 v; };
struct __attribute__((packed, aligned(4), may_alias)) lds_d2 { u32x2 v; };
struct __attribute__((packed, aligned(4), may_alias)) lds_d1 { uint32_t v; };
struct __attribute__((packed, aligned(2), may_alias)) lds_h1 { uint16_t v; };

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave's tokens of PB super-blocks, TT tiles of 16: operands, block scales, and P = d * sum(q) of sub-blocks q and q + 4
template <class F, int PB, int TT>
struct DirectTokens {
    u32x2 a[PB][TT][8];
    float d[PB][TT][8];
    float p[PB][TT][2];
};

// 16-byte pieces, consecutive lanes consecutive ones of a token's PB super-blocks (272 bytes each), straight to LDS.  Tokens past
// the last lie past the end of the buffer and become zeros, those past the tiles among them: the strip is whole KB long.  (No
// branch: behind one the compiler moves the fmas of a super-block that was begun before it, and spills the matrix core's results.)
template <int PB, int TT>
constexpr uint32_t direct_pieces() { return 17 * PB * 16 * TT; }
template <int PB, int TT>
constexpr uint32_t direct_dma() { return (direct_pieces<PB, TT>() + 63) / 64; }
template <int PB, int TT>
__device__ __forceinline__ void direct_token_loads(__amdgpu_buffer_rsrc_t rs, uint32_t arow, uint32_t blk0, uint8_t *strip, uint32_t lane) {
    constexpr uint32_t PIECES = 17 * PB;
    uint32_t tok = PB == 1 ? (lane * 241) >> 12 : (lane * 241) >> 13, piece = lane - tok * PIECES;  // lane / 17, lane / 34
    static_assert(PB == 1 || PB == 2, "the division above");
#pragma unroll
    for (uint32_t i = 0; i < direct_dma<PB, TT>(); i++) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, OXQ_LDS_PTR(strip + 1024 * i), 16, __umul24(tok, arow) + 16 * piece, blk0 * 272, 0, 0);
        tok += 64 / PIECES, piece += 64 % PIECES;
        if (piece >= PIECES) piece -= PIECES, tok++;
    }
}
template <class F, int PB, int TT>
__device__ __forceinline__ void direct_tokens(DirectTokens<F, PB, TT> &tk, const uint8_t *strip, uint32_t live, uint32_t lane) {
    using D = Direct<F>;
    constexpr uint32_t TS = 272 * PB;
    const uint32_t c = lane & 15, q = lane >> 4, oct = D::ORDER == 0 ? ((q & 1) << 1) | (q >> 1) : q;
#pragma unroll
    for (int t = 0; t < TT; t++) {
        const uint8_t *const head = strip + (16 * t + c) * TS, *const mine = head + 8 * oct, *const scale = head + 34 * q;
#pragma unroll
        for (int b = 0; b < PB; b++) {
            int sum[8];
#pragma unroll
            for (int s = 0; s < 8; s++) {
                // a pair of blocks is 17 dwords: the first payload two bytes into one, the second on a dword
                const uint8_t *at = mine + 272 * b + 68 * (s >> 1);
                uint32_t v0, v1;
                if (s & 1) {
                    const u32x2 x = reinterpret_cast<const lds_d2 *>(at + 36)->v;
                    v0 = x[0], v1 = x[1];
                } else {
                    const u32x2 x = reinterpret_cast<const lds_d2 *>(at)->v;
                    const uint32_t y = reinterpret_cast<const lds_d1 *>(at + 8)->v;
                    v0 = __builtin_amdgcn_alignbit(x[1], x[0], 16), v1 = __builtin_amdgcn_alignbit(y, x[1], 16);
                }
                if (D::HAS_MIN) sum[s] = sdot4(v0, 0x01010101u, sdot4(v1, 0x01010101u, 0));
                tk.a[b][t][s] = D::ORDER == 1 ? u32x2{__builtin_amdgcn_perm(v1, v0, 0x06040200u), __builtin_amdgcn_perm(v1, v0, 0x07050301u)}
                                              : u32x2{v0, v1};
            }
#pragma unroll
            for (int g = 0; g < 2; g++) {
                // lane q reads the scale of sub-block 4g + q; every lane needs all four
                // (a super-block past the last: the next token's bytes were staged, or zeros; neither counts)
                const float d = (uint32_t)b < live ? h2f(reinterpret_cast<const lds_h1 *>(scale + 272 * b + 136 * g)->v) : 0.0f;
                uint32_t d0 = __builtin_bit_cast(uint32_t, d), d1 = d0;
                swap16(d0, d1);
                uint32_t d2 = d0, d3 = d1;
                swap32(d0, d2), swap32(d1, d3);
                tk.d[b][t][4 * g] = __builtin_bit_cast(float, d0), tk.d[b][t][4 * g + 1] = __builtin_bit_cast(float, d1);
                tk.d[b][t][4 * g + 2] = __builtin_bit_cast(float, d2), tk.d[b][t][4 * g + 3] = __builtin_bit_cast(float, d3);
                if constexpr (D::HAS_MIN) {
                    // the four lanes' parts of four sub-blocks' sums: lane q ends up with that of sub-block 4g + q
                    uint32_t s0 = sum[4 * g], s1 = sum[4 * g + 1], s2 = sum[4 * g + 2], s3 = sum[4 * g + 3];
                    swap32(s0, s2), swap32(s1, s3);
                    s0 += s2, s1 += s3;
                    swap16(s0, s1);
                    tk.p[b][t][g] = d * (float)(int)(s0 + s1);
                }
            }
        }
    }
}

// The factors of a super-block of the wave's rows to the table [sub-block (, half)][row]; z: this lane's zero-point factors
template <class F>
__device__ __forceinline__ void direct_factors(const typename Direct<F>::W &w, uint8_t *tab, bool live, uint32_t c, uint32_t q, float (&z)[2]) {
    using D = Direct<F>;
    if constexpr (D::KS == 1) {
        float f[2];
        D::factors(w, q, f, z);
        if (!live) f[0] = f[1] = z[0] = z[1] = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < 2; i++) reinterpret_cast<lds_f1 *>(tab + ((q + 4 * i) * 16 + c) * 4)->v = f[i];
    } else {
        float f[4];
        D::factors(w, f);
        if (!live) f[0] = f[1] = f[2] = f[3] = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) reinterpret_cast<lds_f1 *>(tab + ((4 * q + i) * 16 + c) * 4)->v = f[i];
    }
}

// One super-block of the wave's rows (arranged; factors in the table) against its tokens.
// sink(t, v, s, is, sum): every integer sum, as the MFMA left it (for the dump, with OFFSET times the token's).
template <class F, int TT, bool DUMP, class Sink>
__device__ __forceinline__ void direct_block(const typename Direct<F>::W &w, const uint8_t *tab, const float (&z)[2],
                                             const u32x2 (&ta)[TT][8], const float (&td)[TT][8], const float (&tp)[TT][2], uint32_t q,
                                             const v4i32 magic, v4f32 (&acc)[TT], const Sink &sink) {
    using D = Direct<F>;
    constexpr float MAGIC = 12582912.0f;  // 1.5 * 2^23
    constexpr int KS = D::KS;
    const uint64_t half = (q & 1) ? 0ull : ~0ull;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        if constexpr (D::HAS_MIN) {
            // Between the products of its four sub-blocks, which it mostly takes back: partial sums stay small.  (All of them first:
            // 1.3 to 1.6 times the error against 64 bits on 1024 columns of Q4_K, Q5_K, Q4_0.)
            if (s % 4 == 2)
#pragma unroll
                for (int t = 0; t < TT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(z[s / 4], tp[t][s / 4], acc[t], 0, 0, 0);
        }
        const long op = D::operand(w, s);
#pragma unroll
        for (int is = 0; is < KS; is++) {
            const v4f32 dsc = reinterpret_cast<const lds_f4 *>(tab + ((s * KS + is) * 16 + 4 * q) * 4)->v, corr = -(MAGIC * dsc);  // (exact)
            const long o = KS == 1 ? op : (long)((uint64_t)op & (is == 0 ? half : ~half));
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const u32x2 a = ta[t][s];
                const float da = td[t][s];
                const v4i32 r = __builtin_amdgcn_mfma_i32_16x16x32_i8(o, i8x8(a[0], a[1]), magic, 0, 0, 0);
                v4i32 token = {0, 0, 0, 0};
                if constexpr (DUMP && D::OFFSET) token = __builtin_amdgcn_mfma_i32_16x16x32_i8(0x0101010101010101l, i8x8(a[0], a[1]), token, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    int ri = r[v];
                    const float x = fmaf(__builtin_bit_cast(float, ri), dsc[v], corr[v]);  // fl(dsc * isum)
                    acc[t][v] = fmaf(x, da, acc[t][v]);
                    if constexpr (DUMP) ri += D::TIMES * D::OFFSET * token[v];
                    sink(t, v, s, is, ri);
                }
            }
        }
    }
}

// What a work group works on: row tiles of the matrix, at most 16 * TT token rows.
struct DirectJob {
    const uint8_t *W, *A;  // the matrix; the first token's blocks
    float *out;            // the first token's row
    int32_t *sums;
    const float *bias;
    uint32_t rows, n, k;
    int accumulate;
    uint32_t first, end, step;  // sets of RG row tiles (streamed: one): first, first + step, ..., below end
};

template <int N, int TT>
__device__ __forceinline__ void zero_sums(v4f32 (&acc)[N][TT]) {
#pragma unroll
    for (int x = 0; x < N; x++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[x][t] = v4f32{0.0f, 0.0f, 0.0f, 0.0f};
}

// The integer sum of (weight row, token, sub-block or half of one) to the debug dump.
template <class F>
__device__ __forceinline__ void direct_dump(const DirectJob &j, int ri, uint32_t row, uint32_t tok, uint32_t blk, int s, int is, bool live) {
    using D = Direct<F>;
    if (row < j.n && tok < j.rows && live)
        j.sums[((size_t)tok * j.n + row) * (j.k / 32 * D::KS) + (blk * 8 + s) * D::KS + is] = (ri - 0x4B400000) / D::TIMES;
}

// Where the parts' sums of XT sets of WAVES / KP row tiles meet, [turn][wave][set][token tile] in LDS: thread e of each 256 takes row
// e % 16 against token e / 16 of one (row tile, token tile), adds the parts in the order of k and stores.  One barrier: the
// next sets' sums go to the other buffer.
template <int KP, int TT, int XT, int WAVES>
struct DirectExchange {
    static constexpr uint32_t RG = WAVES / KP, TILES = XT * RG * TT, THREADS = 64 * WAVES;
    static constexpr int NE = (TILES * 256 + THREADS - 1) / THREADS;
    const DirectJob &j;
    uint8_t *ex;
    uint32_t turn;
    __device__ __forceinline__ bool at(int i, uint32_t set, uint32_t &row, uint32_t &tok, uint32_t &slot) const {
        const uint32_t e = threadIdx.x + THREADS * i, t = (e >> 8) % TT, g = (e >> 8) / TT % RG, x = (e >> 8) / TT / RG;
        row = 16 * ((set + x * j.step) * RG + g) + (e & 15), tok = 16 * t + ((e >> 4) & 15);
        slot = (g * KP * XT + x) * TT + t;
        return e < TILES * 256 && set + x * j.step < j.end && row < j.n && tok < j.rows;
    }
    // what the sums are added to, requested before they are formed
    __device__ __forceinline__ void request(float (&old)[NE], uint32_t set) const {
        if (j.accumulate || j.bias)
#pragma unroll
            for (int i = 0; i < NE; i++) {
                uint32_t row, tok, slot;
                if (at(i, set, row, tok, slot)) old[i] = j.accumulate ? j.out[(size_t)tok * j.n + row] : j.bias[row];
            }
    }
    __device__ __forceinline__ void finish(const v4f32 (&acc)[XT][TT], const float (&old)[NE], uint32_t set) {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        uint8_t *const buf = ex + turn * (WAVES * XT * TT * EX_TILE * 4);
        turn ^= 1;
#pragma unroll
        for (int x = 0; x < XT; x++)
#pragma unroll
            for (int t = 0; t < TT; t++)
                reinterpret_cast<lds_f4 *>(buf + (((wave * XT + x) * TT + t) * EX_TILE + (lane >> 4) * EX_Q + 4 * (lane & 15)) * 4)->v = acc[x][t];
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NE; i++) {
            uint32_t row, tok, slot;
            if (at(i, set, row, tok, slot)) {
                const uint32_t r = row & 15;
                const uint8_t *p = buf + (slot * EX_TILE + (r >> 2) * EX_Q + 4 * (tok & 15) + (r & 3)) * 4;
                float y = reinterpret_cast<const lds_f1 *>(p)->v;
#pragma unroll
                for (int k = 1; k < KP; k++) y += reinterpret_cast<const lds_f1 *>(p + k * (XT * TT * EX_TILE * 4))->v;
                j.out[(size_t)tok * j.n + row] = j.accumulate || j.bias ? old[i] + y : y;
            }
        }
    }
};

// KP parts of k, PB super-blocks each, on WAVES / KP row tiles at a time; the tokens stay in registers.
template <class F, int PB, int KP, int TT, int WAVES, bool DUMP>
__device__ __forceinline__ void direct_resident(const DirectJob j, uint8_t *lds) {
    using D = Direct<F>;
    constexpr uint32_t RG = WAVES / KP;
    constexpr int U = 2, XT = direct_turn<TT, WAVES>();  // row tiles whose weights are in flight; that are exchanged at once
    const uint32_t lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), part = wave % KP, rg = wave / KP;
    const uint32_t nb = j.k / 256, blk0 = part * PB, sets = j.end;
    const uint32_t live = nb > blk0 ? min((uint32_t)PB, nb - blk0) : 0;  // super-blocks of this part
    const uint32_t row_bytes = nb * D::BLOCK, arow = nb * 272;
    constexpr bool APART = direct_exchange_apart<F, PB, TT, WAVES>();
    uint8_t *const tab = lds + wave * (direct_tables<F, WAVES>() / WAVES);
    uint8_t *const strips = lds + direct_tables<F, WAVES>(), *const strip = strips + wave * (direct_strips<PB, TT, WAVES>() / WAVES);
    uint8_t *const ex = APART ? strips + direct_strips<PB, TT, WAVES>() : strips;

    const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(j.A), 0, (int)(j.rows * arow), BUFFER_FLAGS);
    if (live) direct_token_loads<PB, TT>(rs_a, arow, blk0, strip, lane);
    const uint32_t wrow = c * row_bytes;
    typename D::W ring[U][PB];
    auto load = [&](int u, int b, uint32_t set) __attribute__((always_inline)) {
        // (rows past the last lie past the end of the buffer: zeros)
        const DirectWindow win = direct_window(set, sets, rg, RG, j.n, row_bytes);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(j.W + (size_t)win.row0 * row_bytes), 0, (int)win.records, BUFFER_FLAGS);
        D::load(ring[u][b], rs, wrow, q, direct_super_block(blk0 + b, nb) * D::BLOCK);
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int b = 0; b < PB; b++) {  // (in the order of use, as in the loop: a wait counts what was requested after)
            load(u, b, j.first + u * j.step);
            __builtin_amdgcn_sched_barrier(0);
        }
    // the tokens are there when no more than the weights' loads are outstanding
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(U * PB * D::LOADS) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    DirectTokens<F, PB, TT> tk;
    direct_tokens<F, PB, TT>(tk, strip, live, lane);

    v4i32 magic;
    asm volatile("v_mov_b32 %0, 0x4b400000\n\tv_mov_b32 %1, 0x4b400000\n\tv_mov_b32 %2, 0x4b400000\n\tv_mov_b32 %3, 0x4b400000"
                 : "=v"(magic[0]), "=v"(magic[1]), "=v"(magic[2]), "=v"(magic[3]));
    if constexpr (!APART) __syncthreads();  // every wave has its tokens in registers
    DirectExchange<KP, TT, XT, WAVES> xc{j, ex, 0};
    if (live == 0) {  // a part past the last super-block: zeros
        v4f32 none[XT][TT];
        zero_sums<XT, TT>(none);
        for (uint32_t set = j.first; set < sets; set += XT * j.step) {
            float old[xc.NE];
            xc.request(old, set);
            xc.finish(none, old, set);
        }
        return;
    }
    auto row_tile = [&](int u, uint32_t set, v4f32 (&acc)[TT]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < PB; b++) {
            D::arrange(ring[u][b], q);
            float z[2];
            uint8_t *const tb = tab + (b & 1) * 8 * D::KS * 64;
            direct_factors<F>(ring[u][b], tb, (uint32_t)b < live, c, q, z);
            wave_lds_fence();
            auto sink = [&](int t, int v, int s, int is, int ri) __attribute__((always_inline)) {
                if (DUMP) direct_dump<F>(j, ri, 16 * (set * RG + rg) + 4 * q + v, 16 * t + c, blk0 + b, s, is, (uint32_t)b < live);
            };
            direct_block<F, TT, DUMP>(ring[u][b], tb, z, tk.a[b], tk.d[b], tk.p[b], q, magic, acc, sink);
            wave_lds_fence();
            // (only now: a load while the slot is still in use would go to other registers and be copied when it arrives)
            load(u, b, set + U * j.step);
        }
    };
    uint32_t set = j.first;
#pragma clang loop unroll(disable)
    for (; set + j.step < sets; set += 2 * j.step) {
        v4f32 acc[2][TT];
        zero_sums<2, TT>(acc);
        if constexpr (XT == 2) {
            float old[xc.NE];
            xc.request(old, set);
            row_tile(0, set, acc[0]), row_tile(1, set + j.step, acc[1]);
            xc.finish(acc, old, set);
        } else {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                float old[xc.NE];
                xc.request(old, set + u * j.step);
                row_tile(u, set + u * j.step, acc[u]);
                xc.finish(reinterpret_cast<v4f32(&)[1][TT]>(acc[u]), old, set + u * j.step);
            }
        }
    }
    if (set < sets) {
        v4f32 acc[XT][TT];
        zero_sums<XT, TT>(acc);
        float old[xc.NE];
        xc.request(old, set);
        row_tile(0, set, acc[0]);
        xc.finish(acc, old, set);
    }
}

// One row tile at a time over a k of any length: each wave goes through its own run of super-blocks, the next one's tokens and the
// next two's weights in flight.
template <class F, int TT, int WAVES, bool DUMP>
__device__ __forceinline__ void direct_streamed(const DirectJob j, uint8_t *lds) {
    using D = Direct<F>;
    const uint32_t lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nb = j.k / 256, tiles = j.end;
    const uint32_t blk0 = wave * (nb / WAVES) + min(wave, nb % WAVES), run = nb / WAVES + (wave < nb % WAVES ? 1 : 0);  // (nb >= WAVES: no empty run)
    const uint32_t row_bytes = nb * D::BLOCK, arow = nb * 272, wrow = c * row_bytes;
    uint8_t *const tab = lds + wave * (direct_tables<F, WAVES>() / WAVES);
    uint8_t *const strips = lds + direct_tables<F, WAVES>(), *const strip = strips + wave * (direct_strips<1, TT, WAVES>() / WAVES);
    constexpr bool APART = direct_streamed_apart<F, TT, WAVES>();
    uint8_t *const ex = APART ? strips + direct_strips<1, TT, WAVES>() : strips;
    const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(j.A), 0, (int)(j.rows * arow), BUFFER_FLAGS);
    v4i32 magic;
    asm volatile("v_mov_b32 %0, 0x4b400000\n\tv_mov_b32 %1, 0x4b400000\n\tv_mov_b32 %2, 0x4b400000\n\tv_mov_b32 %3, 0x4b400000"
                 : "=v"(magic[0]), "=v"(magic[1]), "=v"(magic[2]), "=v"(magic[3]));
    DirectExchange<WAVES, TT, 1, WAVES> xc{j, ex, 0};
#pragma clang loop unroll(disable)
    for (uint32_t tile = j.first; tile < tiles; tile += j.step) {
        const DirectWindow win = direct_window(tile, tiles, 0, 1, j.n, row_bytes);
        const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t *>(j.W + (size_t)win.row0 * row_bytes), 0, (int)win.records, BUFFER_FLAGS);
        typename D::W ring[2];
        // super-block i of the run (past its end: the last one again, not used)
        auto request_tokens = [&](uint32_t i) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            direct_token_loads<1, TT>(rs_a, arow, blk0 + min(i, run - 1), strip, lane);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto request_weights = [&](int u, uint32_t i) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            D::load(ring[u], rs_w, wrow, q, (blk0 + min(i, run - 1)) * D::BLOCK);
            __builtin_amdgcn_sched_barrier(0);
        };
        // One token tile: the run's even and odd super-blocks apart, which halves the length of the chain (one chain: 1.2 times the
        // error against 64 bits of the few-token kernel's split of k, Q6_K 4096 x 14336).  More: no registers left, nor is their error larger than the tile kernel's.
        constexpr int CHAINS = TT == 1 ? 2 : 1;
        v4f32 acc[CHAINS][TT];
        zero_sums<CHAINS, TT>(acc);
        float old[xc.NE];
        xc.request(old, tile);
        request_tokens(0), request_weights(0, 0), request_weights(1, 1);
        auto super_block = [&](int u, uint32_t i) __attribute__((always_inline)) {
            // its tokens are there when no more is outstanding than the next super-block's weights
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D::LOADS) : "memory");
            __builtin_amdgcn_sched_barrier(0);
            DirectTokens<F, 1, TT> tk;
            direct_tokens<F, 1, TT>(tk, strip, 1, lane);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the strip has been read
            request_tokens(i + 1);
            D::arrange(ring[u], q);
            float z[2];
            direct_factors<F>(ring[u], tab, true, c, q, z);
            wave_lds_fence();
            auto sink = [&](int t, int v, int s, int is, int ri) __attribute__((always_inline)) {
                if (DUMP) direct_dump<F>(j, ri, 16 * tile + 4 * q + v, 16 * t + c, blk0 + i, s, is, true);
            };
            direct_block<F, TT, DUMP>(ring[u], tab, z, tk.a[0], tk.d[0], tk.p[0], q, magic, acc[u % CHAINS], sink);
            wave_lds_fence();
            request_weights(u, i + 2);
        };
        uint32_t i = 0;
#pragma clang loop unroll(disable)
        for (; i + 1 < run; i += 2) super_block(0, i), super_block(1, i + 1);
        if (i < run) super_block(0, i);
        if constexpr (CHAINS == 2) acc[0][0] += acc[1][0];
        if constexpr (APART) {
            xc.finish(reinterpret_cast<v4f32(&)[1][TT]>(acc[0]), old, tile);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (what was requested past the run's end: the strip is written again)
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();  // nothing is on its way to a strip and none is read any more
            xc.finish(reinterpret_cast<v4f32(&)[1][TT]>(acc[0]), old, tile);
            if (tile + j.step < tiles) __syncthreads();  // the sums have been read
        }
    }
}

// The kernels.  KP == 0: k streamed.
// blockIdx.y: a run of 16 * TT token rows
template <class F, int PB, int KP, int TT, int WAVES, bool DUMP>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(WAVES / 4, WAVES / 4))) void gemm_direct_kernel(
    const uint8_t *__restrict__ W, const uint8_t *__restrict__ A, float *__restrict__ out, int32_t *__restrict__ sums, uint32_t m,
    uint32_t n, uint32_t k, int accumulate, const float *__restrict__ bias) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t t0 = blockIdx.y * (16 * TT), nb = k / 256, tiles = (n + 15) / 16;
    constexpr uint32_t RG = KP ? WAVES / (KP ? KP : 1) : 1;
    const DirectJob j = {W, A + (size_t)t0 * nb * 272, out + (size_t)t0 * n, DUMP ? sums + (size_t)t0 * n * (nb * 8 * Direct<F>::KS) : nullptr, bias,
                         min(m - t0, (uint32_t)(16 * TT)), n, k, accumulate, blockIdx.x, (tiles + RG - 1) / RG, gridDim.x};
    if constexpr (KP == 0) direct_streamed<F, TT, WAVES, DUMP>(j, lds);
    else direct_resident<F, PB, KP, TT, WAVES, DUMP>(j, lds);
}

}  // namespace oxq
