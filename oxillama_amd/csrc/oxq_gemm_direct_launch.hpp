// Launches of the kernel in oxq_gemm_direct.hpp.
#pragma once
#include "oxq_gemm_direct.hpp"
#include "oxq_gemm_skinny.hpp"

namespace oxq {

// KP == 0: the streamed form.  A call's tokens go in `chunks` runs of 16 * TT rows, each with its own work groups; where there are more
// row tiles than work groups for them, all walk the same number.
template <class F, int PB, int KP, int TT, int WAVES = 8>
hipError_t launch_direct_shape(const GemmArgs &a, hipStream_t stream) {
    auto kern = &gemm_direct_kernel<F, PB, KP, TT, WAVES, false>;
    if constexpr (TT <= 2) {
        if (a.sums) kern = &gemm_direct_kernel<F, PB, KP, TT, WAVES, true>;
    } else if (a.sums) {
        return hipErrorNotSupported;
    }
    constexpr size_t lds = KP ? direct_lds<F, PB, TT, WAVES>() : direct_streamed_lds<F, TT, WAVES>();
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    const hipError_t e = allow_lds(reinterpret_cast<const void *>(kern), lds);
    if (e != hipSuccess) return e;
    constexpr uint32_t RG = KP ? WAVES / (KP ? KP : 1) : 1;
    const uint32_t sets = ((a.n + 15) / 16 + RG - 1) / RG, chunks = (a.m + 16 * TT - 1) / (16 * TT);
    const uint32_t room = device_cus() > chunks ? device_cus() / chunks : 1, walk = (sets + room - 1) / room;
    const dim3 grid(chunks == 1 ? (sets < room ? sets : room) : (sets + walk - 1) / walk, chunks);
    note_launch("gemm_direct_kernel", F::TYPE, PB, KP, TT, WAVES, grid.x, grid.y, 64 * WAVES);
    hipLaunchKernelGGL(kern, grid, dim3(64 * WAVES), lds, stream, a.W, a.A, a.out, a.sums, a.m, a.n, a.k, a.accumulate, a.bias);
    return hipGetLastError();
}
template <class F, int TT>
hipError_t launch_direct(const GemmArgs &a, hipStream_t stream) {
    const uint32_t nb = a.k / 256;
    if constexpr (TT == 1) {
        if (nb > 16) return launch_direct_shape<F, 1, 0, 1>(a, stream);
        if (nb > 8) return launch_direct_shape<F, 1, 16, 1, 16>(a, stream);
    } else {
        if (nb > 16) return launch_direct_shape<F, 1, 0, TT>(a, stream);
        if (nb > 8) {
            if constexpr (TT == 2) return launch_direct_shape<F, 2, 8, 2>(a, stream);
            else return hipErrorNotSupported;
        }
    }
    if (nb > 4) return launch_direct_shape<F, 1, 8, TT>(a, stream);
    return launch_direct_shape<F, 1, 4, TT>(a, stream);
}
// One or the other number of token tiles.
template <int T0, int T1>
hipError_t launch_direct_of(uint32_t type, uint32_t tt, const GemmArgs &a, hipStream_t stream) {
#define OXQ_DIRECT(T, F) \
    if (type == T) return tt == T0 ? launch_direct<F, T0>(a, stream) : launch_direct<F, T1>(a, stream);
    OXQ_DIRECT(OXQ_TYPE_Q4_K, TileQ4K)
    OXQ_DIRECT(OXQ_TYPE_Q5_K, DirectQ5K)
    OXQ_DIRECT(OXQ_TYPE_Q6_K, TileQ6K)
    OXQ_DIRECT(OXQ_TYPE_IQ4_XS, TileIQ4XS)
    OXQ_DIRECT(OXQ_TYPE_Q4_0, TileQ4_0)
    OXQ_DIRECT(OXQ_TYPE_Q8_0, TileQ8_0)
#undef OXQ_DIRECT
    return hipErrorNotSupported;
}
hipError_t launch_direct_wide(uint32_t type, uint32_t tt, const GemmArgs &a, hipStream_t stream);  // three and four token tiles
constexpr uint32_t DIRECT_MAX_ROWS = 512;

}  // namespace oxq
