// Instantiations and launcher of the FP8 GEMM for a few rows of A (gemm_few.h); gemm.hip decides when it serves.
#include "gemm_common.h"
#include "gemm_big.h"
#include "gemm_few.h"

namespace ntfp8 {

template <int FA, int FB>
static int launch_fmt(const BigProblem& p, hipStream_t st) {
    const bool narrow = (p.N - 1) / 16 + 1 <= cu_count();   // one workgroup per CU
    const dim3 grid((p.N - 1) / (narrow ? 16 : 32) + 1), block(kFewThreads);
    (void)hipGetLastError();   // an error left behind by an unrelated earlier call is not this launch's
    if (p.M > 16) hipLaunchKernelGGL((gemm_few_kernel<FA, FB, 2, 1>), dim3((p.N - 1) / 16 + 1), block, 0, st, p);
    else if (narrow) hipLaunchKernelGGL((gemm_few_kernel<FA, FB, 1, 1>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((gemm_few_kernel<FA, FB, 1, 2>), grid, block, 0, st, p);
    return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}

int launch_few(const BigProblem& p, int fa, int fb, hipStream_t st) {
    if (fa == kE4M3) return fb == kE4M3 ? launch_fmt<kE4M3, kE4M3>(p, st) : launch_fmt<kE4M3, kE5M2>(p, st);
    return fb == kE4M3 ? launch_fmt<kE5M2, kE4M3>(p, st) : launch_fmt<kE5M2, kE5M2>(p, st);
}

}  // namespace ntfp8
