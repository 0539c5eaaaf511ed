// Instantiations and launcher of the 128- and 64-wide FP8 GEMM tiles (gemm_mid.h); the choice between them and the
// 256-wide ones is made in gemm.hip.
#include "gemm_common.h"
#include "gemm_big.h"
#include "gemm_mid.h"

namespace ntfp8 {

template <int FA, int FB>
static int launch_fmt(const BigLaunch& L, int tile, bool fp8_out, int tiles, hipStream_t st) {
    (void)hipGetLastError();   // an error left behind by an unrelated earlier call is not this launch's
    if (tile == 128) {
        if (fp8_out) hipLaunchKernelGGL((gemm_mid_kernel<FA, FB, 128, true>), dim3(tiles), dim3(kBigThreads), 0, st, L);
        else hipLaunchKernelGGL((gemm_mid_kernel<FA, FB, 128, false>), dim3(tiles), dim3(kBigThreads), 0, st, L);
    } else {
        if (fp8_out) hipLaunchKernelGGL((gemm_mid_kernel<FA, FB, 64, true>), dim3(tiles), dim3(kBigThreads), 0, st, L);
        else hipLaunchKernelGGL((gemm_mid_kernel<FA, FB, 64, false>), dim3(tiles), dim3(kBigThreads), 0, st, L);
    }
    return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}

int launch_mid(const BigLaunch& L, int fa, int fb, int tile, bool fp8_out, int tiles, hipStream_t st) {
    if (fa == kE4M3)
        return fb == kE4M3 ? launch_fmt<kE4M3, kE4M3>(L, tile, fp8_out, tiles, st) : launch_fmt<kE4M3, kE5M2>(L, tile, fp8_out, tiles, st);
    return fb == kE4M3 ? launch_fmt<kE5M2, kE4M3>(L, tile, fp8_out, tiles, st) : launch_fmt<kE5M2, kE5M2>(L, tile, fp8_out, tiles, st);
}

}  // namespace ntfp8
