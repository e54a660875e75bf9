// Launches of the streamed routed-expert kernels (moe_stream.hpp).
#include "moe_stream.hpp"

namespace hm {

void launch_moe_front(int bm, const RouteParams& R, const TokenQuant& Q, hipStream_t s) {
    const dim3 grid(1 + (Q.rows + FRONT_THREADS / 64 - 1) / (FRONT_THREADS / 64)), block(FRONT_THREADS);
    if (bm == 16)
        hipLaunchKernelGGL(moe_front_kernel<16>, grid, block, 0, s, R, Q);
    else
        hipLaunchKernelGGL(moe_front_kernel<48>, grid, block, 0, s, R, Q);
}

template <int BITS, int EPI, int RTM, bool AQ>
static void launch_windows(const MoeStreamParams& P, int grid, hipStream_t s) {
    const int units = (P.K_pad / (BITS == 8 ? 16 : 32) + 3) / 4;
    const int per_wave = (units + STREAM_NWV - 1) / STREAM_NWV;
    const size_t lds = AQ ? (size_t)P.K_pad * 16 : 0;
    const dim3 g(grid), b(STREAM_NT);
    if (per_wave <= 2)
        hipLaunchKernelGGL((moe_stream_kernel<BITS, EPI, RTM, 2, false, AQ>), g, b, lds, s, P);
    else if (per_wave <= 3)
        hipLaunchKernelGGL((moe_stream_kernel<BITS, EPI, RTM, 3, false, AQ>), g, b, lds, s, P);
    else if (per_wave <= 4)
        hipLaunchKernelGGL((moe_stream_kernel<BITS, EPI, RTM, 4, false, AQ>), g, b, lds, s, P);
    else if constexpr (RTM == 1)  // (longer K takes 16-row tiles only)
        hipLaunchKernelGGL((moe_stream_kernel<BITS, EPI, RTM, 4, true, AQ>), g, b, lds, s, P);
}

void launch_moe_stream(int bits, int epi, int bm, bool aq, const MoeStreamParams& P, int tiles, hipStream_t s) {
    const int grid = (tiles + 7) / 8 * 8 * P.tiles_n;
    if (epi != EPI_PLAIN) {  // gate/up are W4
        if (bm == 16)
            launch_windows<4, EPI_SWIGLU_MAX, 1, false>(P, grid, s);
        else
            launch_windows<4, EPI_SWIGLU_MAX, 3, false>(P, grid, s);
    } else if (bits == 8) {
        if (aq)
            launch_windows<8, EPI_PLAIN, 1, true>(P, grid, s);
        else if (bm == 16)
            launch_windows<8, EPI_PLAIN, 1, false>(P, grid, s);
        else
            launch_windows<8, EPI_PLAIN, 3, false>(P, grid, s);
    } else {
        if (aq)
            launch_windows<4, EPI_PLAIN, 1, true>(P, grid, s);
        else if (bm == 16)
            launch_windows<4, EPI_PLAIN, 1, false>(P, grid, s);
        else
            launch_windows<4, EPI_PLAIN, 3, false>(P, grid, s);
    }
}

}  // namespace hm
