// The few-token kernel that keeps its tokens in registers (oxq_gemm_direct.hpp), instantiated for its formats.
#include "oxq_gemm_direct.hpp"
#include "oxq_gemm_skinny.hpp"

namespace oxq {

// KP == 0: the streamed form
template <class F, int PB, int KP, int TT, int WAVES = 8>
static hipError_t launch_direct_shape(const GemmArgs &a, hipStream_t stream) {
    auto kern = a.sums ? &gemm_direct_kernel<F, PB, KP, TT, WAVES, true> : &gemm_direct_kernel<F, PB, KP, TT, WAVES, false>;
    constexpr size_t lds = KP ? direct_lds<F, PB, TT, WAVES>() : direct_streamed_lds<F, TT, WAVES>();
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    const hipError_t e = allow_lds(reinterpret_cast<const void *>(kern), lds);
    if (e != hipSuccess) return e;
    constexpr uint32_t RG = KP ? WAVES / KP : 1;
    const uint32_t sets = ((a.n + 15) / 16 + RG - 1) / RG;
    const dim3 grid(sets < device_cus() ? sets : device_cus());
    // (named by what the call would take otherwise)
    note_launch(TT == 1 && a.workspace && !a.by_rows && skinny_whole_pays(F::TYPE, a.n, a.k, skinny_splits(a.n, a.k) >= 2) ? "gemm_skinny_whole_kernel_direct"
                                                                                            : "gemm_skinny_kernel_direct",
                F::TYPE, PB, KP, TT, WAVES, grid.x, 1, 64 * WAVES);
    hipLaunchKernelGGL(kern, grid, dim3(64 * WAVES), lds, stream, a.W, a.A, a.out, a.sums, a.m, a.n, a.k, a.accumulate, a.bias);
    return hipGetLastError();
}
template <class F, int TT>
static hipError_t launch_direct(const GemmArgs &a, hipStream_t stream) {
    const uint32_t nb = a.k / 256;
    if constexpr (TT == 1) {
        if (nb > 16) return launch_direct_shape<F, 1, 0, 1>(a, stream);
        if (nb > 8) return launch_direct_shape<F, 1, 16, 1, 16>(a, stream);
    } else {
        if (nb > 8) return launch_direct_shape<F, 2, 8, 2>(a, stream);
    }
    if (nb > 4) return launch_direct_shape<F, 1, 8, TT>(a, stream);
    return launch_direct_shape<F, 1, 4, TT>(a, stream);
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
bool gemm_direct_pays(uint32_t type, uint32_t m, uint32_t n, uint32_t k) {
    if (!direct_format(type) || m == 0 || m > 32 || k % 256 != 0 || k < 512) return false;
    if (k > 4096) return m <= 16 && n <= 16 * device_cus() && k <= 32768 && (type != OXQ_TYPE_Q8_0 || n >= 1536);
    return type != OXQ_TYPE_Q8_0 || n < 256 * device_cus();
}

hipError_t launch_gemm_direct(uint32_t type, const GemmArgs &a, hipStream_t stream) {
    if (a.offsets || a.m == 0 || a.m > 32 || a.k % 256 != 0 || a.k < 512 || (a.m > 16 && a.k > 4096) ||
        (size_t)a.m * (a.k / 32) * Q8_BLOCK_BYTES > 0x7FFFFFFF || (reinterpret_cast<uintptr_t>(a.W) & 3) ||
        (reinterpret_cast<uintptr_t>(a.A) & 15))  // (what loads straight to LDS and the dword-wise loads were built for)
        return hipErrorNotSupported;
#define OXQ_DIRECT(T, F) \
    if (type == T) return a.m <= 16 ? launch_direct<F, 1>(a, stream) : launch_direct<F, 2>(a, stream);
    OXQ_DIRECT(OXQ_TYPE_Q4_K, TileQ4K)
    OXQ_DIRECT(OXQ_TYPE_Q5_K, DirectQ5K)
    OXQ_DIRECT(OXQ_TYPE_Q6_K, TileQ6K)
    OXQ_DIRECT(OXQ_TYPE_IQ4_XS, TileIQ4XS)
    OXQ_DIRECT(OXQ_TYPE_Q4_0, TileQ4_0)
    OXQ_DIRECT(OXQ_TYPE_Q8_0, TileQ8_0)
#undef OXQ_DIRECT
    return hipErrorNotSupported;
}

}  // namespace oxq
