// Instantiations and launcher of the 128 x 128, 128 x 64 and 64 x 64 FP8 GEMM tiles (gemm_mid.h); the choice between them and the
// 256-wide ones is made in gemm.hip.
#include "gemm_common.h"
#include "gemm_big.h"
#include "gemm_mid.h"

namespace ntfp8 {

template <int FA, int FB>
static int launch_fmt(const BigLaunch& L, int tile_m, int tile_n, bool fp8_out, int tiles, hipStream_t st) {
    (void)hipGetLastError();   // an error left behind by an unrelated earlier call is not this launch's
    auto go = [&](auto m_tag, auto n_tag) {
        constexpr int TM = decltype(m_tag)::value, TN = decltype(n_tag)::value;
        if (fp8_out) hipLaunchKernelGGL((gemm_mid_kernel<FA, FB, TM, TN, true>), dim3(tiles), dim3(kBigThreads), 0, st, L);
        else hipLaunchKernelGGL((gemm_mid_kernel<FA, FB, TM, TN, false>), dim3(tiles), dim3(kBigThreads), 0, st, L);
    };
    typedef std::integral_constant<int, 128> Wide;
    typedef std::integral_constant<int, 64> Narrow;
    if (tile_n == 128) go(Wide{}, Wide{});
    else if (tile_m == 128) go(Wide{}, Narrow{});
    else go(Narrow{}, Narrow{});
    return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}

int launch_mid(const BigLaunch& L, int fa, int fb, int tile_m, int tile_n, bool fp8_out, int tiles, hipStream_t st) {
    if (fa == kE4M3)
        return fb == kE4M3 ? launch_fmt<kE4M3, kE4M3>(L, tile_m, tile_n, fp8_out, tiles, st) : launch_fmt<kE4M3, kE5M2>(L, tile_m, tile_n, fp8_out, tiles, st);
    return fb == kE4M3 ? launch_fmt<kE5M2, kE4M3>(L, tile_m, tile_n, fp8_out, tiles, st) : launch_fmt<kE5M2, kE5M2>(L, tile_m, tile_n, fp8_out, tiles, st);
}

}  // namespace ntfp8
