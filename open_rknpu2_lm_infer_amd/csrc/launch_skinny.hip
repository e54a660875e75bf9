// Launches of skinny_kernel (both weight widths, both epilogues).
#include "launch.hpp"
#include "skinny.hpp"

namespace hm {

// Weight window: all of a wave's units when there are at most 5 (K up to 2560),
// else 8 of them, reloaded as they are used.
template <int BITS, int RT, int CT, int EPI>
static void launch_one(const SkinnyParams& S, int blocks_n, hipStream_t s) {
    constexpr int NWV = BITS == 4 ? 4 : 8;
    const int units = (S.g.K_pad / (BITS == 8 ? 16 : 32) + 3) / 4;
    const dim3 grid(blocks_n, (S.g.M + 16 * RT - 1) / (16 * RT));
    if (units <= 5 * NWV)
        hipLaunchKernelGGL((skinny_kernel<BITS, RT, CT, EPI, NWV, 5>), grid, dim3(64 * NWV), 0, s, S);
    else
        hipLaunchKernelGGL((skinny_kernel<BITS, RT, CT, EPI, NWV, 8>), grid, dim3(64 * NWV), 0, s, S);
}

template <int BITS, int CT, int EPI>
static void launch_rows(int row_tiles, const SkinnyParams& S, int blocks_n, hipStream_t s) {
    if (row_tiles <= 1)
        launch_one<BITS, 1, CT, EPI>(S, blocks_n, s);
    else if (row_tiles <= 2)
        launch_one<BITS, 2, CT, EPI>(S, blocks_n, s);
    else if (row_tiles <= 4)
        launch_one<BITS, 4, CT, EPI>(S, blocks_n, s);
    else
        launch_one<BITS, 8, CT, EPI>(S, blocks_n, s);
}

template <int BITS>
static void launch_epi(int epi, const SkinnyPlan& p, const SkinnyParams& S, hipStream_t s) {
    if (epi != EPI_PLAIN)
        launch_rows<BITS, 2, EPI_SWIGLU_MAX>(p.row_tiles, S, p.blocks_n, s);
    else if (p.col_tiles == 2)
        launch_rows<BITS, 2, EPI_PLAIN>(p.row_tiles, S, p.blocks_n, s);
    else
        launch_rows<BITS, 1, EPI_PLAIN>(p.row_tiles, S, p.blocks_n, s);
}

void launch_skinny(int bits, int epi, const SkinnyPlan& p, bool staged, const GemmParams& G, float* part,
                   hipStream_t s) {
    const SkinnyParams S{G, part, staged ? 1 : 0};
    if (bits == 8)
        launch_epi<8>(epi, p, S, s);
    else
        launch_epi<4>(epi, p, S, s);
}

}  // namespace hm
