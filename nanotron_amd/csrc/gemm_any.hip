// Instantiations and launchers of the GEMM kernels off the main path: any K and alignment (gemm_any.h), and fp8 outputs
// whose rows or columns do not come in whole words or large results of few K-tiles.  The choice is made in gemm.hip.
#include "gemm_common.h"
#include "gemm_big.h"
#include "gemm_any.h"

namespace ntfp8 {

template <int FA, int FB>
static int launch_fmt(const BigLaunch& L, int tile, bool fp8_out, int tiles, hipStream_t st) {
    (void)hipGetLastError();   // an error left behind by an unrelated earlier call is not this launch's
    if (tile == 128) {
        if (fp8_out) hipLaunchKernelGGL((gemm_any_kernel<FA, FB, 2, true>), dim3(tiles), dim3(kAnyThreads), 0, st, L);
        else hipLaunchKernelGGL((gemm_any_kernel<FA, FB, 2, false>), dim3(tiles), dim3(kAnyThreads), 0, st, L);
    } else {
        if (fp8_out) hipLaunchKernelGGL((gemm_any_kernel<FA, FB, 1, true>), dim3(tiles), dim3(kAnyThreads), 0, st, L);
        else hipLaunchKernelGGL((gemm_any_kernel<FA, FB, 1, false>), dim3(tiles), dim3(kAnyThreads), 0, st, L);
    }
    return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}

int launch_any(const BigLaunch& L, int fa, int fb, int tile, bool fp8_out, int tiles, hipStream_t st) {
    if (fa == kE4M3)
        return fb == kE4M3 ? launch_fmt<kE4M3, kE4M3>(L, tile, fp8_out, tiles, st) : launch_fmt<kE4M3, kE5M2>(L, tile, fp8_out, tiles, st);
    return fb == kE4M3 ? launch_fmt<kE5M2, kE4M3>(L, tile, fp8_out, tiles, st) : launch_fmt<kE5M2, kE5M2>(L, tile, fp8_out, tiles, st);
}

// ---------------------------------------------------------------------------------------------
// One output per thread, for the smallest products (gemm.hip has the line): bound by the latency of a launch, not by the
// K loads of each thread, while a tile's trip through LDS and its code cost 2 us more.  128 x 62 x 22 6.6 -> 4.2 us.
constexpr int kTinyThreads = 256;
template <int FA, int FB>
__global__ __launch_bounds__(kTinyThreads) void gemm_tiny_kernel(const BigProblem P) {
    const int M = P.M, N = P.N, K = P.K;
    const uint32_t idx = blockIdx.x * kTinyThreads + threadIdx.x;
    const bool live = idx < (uint32_t)M * N;   // (whole waves stay: the amax reduction runs over all lanes)
    const int m = live ? idx / N : 0, n = live ? idx % N : 0;
    float acc = 0.0f;
    for (int k = 0; live && k < K; ++k) {
        const int a = P.A[(int64_t)m * K + k], b = P.B[(int64_t)n * K + k];
        acc += (FA == kE4M3 ? __builtin_amdgcn_cvt_f32_fp8(a, 0) : __builtin_amdgcn_cvt_f32_bf8(a, 0)) *
               (FB == kE4M3 ? __builtin_amdgcn_cvt_f32_fp8(b, 0) : __builtin_amdgcn_cvt_f32_bf8(b, 0));
    }
    float v = acc * descale_factor(P.scale_a, P.scale_b, P.ex.scale_inv);
    if (P.ex.bias && live) v += bias_at(P.ex.bias, P.ex.bias_dtype, n);
    if (P.d_dtype == NTFP8_OUT_E4M3 || P.d_dtype == NTFP8_OUT_E5M2) {   // uniform
        uint32_t amax = 0;
        const uint32_t w = P.d_dtype == NTFP8_OUT_E4M3 ? quant4<kE4M3>(v, 0.f, 0.f, 0.f, *P.fp8.scale, true, amax)
                                                       : quant4<kE5M2>(v, 0.f, 0.f, 0.f, *P.fp8.scale, true, amax);
        if (live) {
            static_cast<uint8_t*>(P.D)[idx] = (uint8_t)w;
            if (P.fp8.Dt) P.fp8.Dt[(int64_t)n * M + m] = (uint8_t)w;
        }
        publish_amax(live ? amax : 0u, P.fp8.ws);
    } else if (live) {
        if (P.d_dtype == NTFP8_BF16) static_cast<uint16_t*>(P.D)[idx] = OutT<NTFP8_BF16>::cvt(v);
        else if (P.d_dtype == NTFP8_F16) static_cast<uint16_t*>(P.D)[idx] = OutT<NTFP8_F16>::cvt(v);
        else if (P.accumulate) static_cast<float*>(P.D)[idx] += v;
        else static_cast<float*>(P.D)[idx] = v;
    }
}

int launch_tiny(const BigProblem& p, int fa, int fb, hipStream_t st) {
    (void)hipGetLastError();
    const dim3 grid((unsigned)(((int64_t)p.M * p.N + kTinyThreads - 1) / kTinyThreads)), block(kTinyThreads);
    if (fa == kE4M3) {
        if (fb == kE4M3) hipLaunchKernelGGL((gemm_tiny_kernel<kE4M3, kE4M3>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((gemm_tiny_kernel<kE4M3, kE5M2>), grid, block, 0, st, p);
    } else {
        if (fb == kE4M3) hipLaunchKernelGGL((gemm_tiny_kernel<kE5M2, kE4M3>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((gemm_tiny_kernel<kE5M2, kE5M2>), grid, block, 0, st, p);
    }
    return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------------------------
// 128 x 128 x 128, 4 waves (2 x 2, each 64 x 64), loads staged through registers.  Bound by HBM on the shapes it serves
// (mostly output): its prologues and epilogues overlap in the three workgroups that a CU holds (168 registers: two more and it is two).
constexpr int kBM = 128, kBN = 128;
constexpr int kGemmThreads = 256;

// DT: an fp8 output type, or NTFP8_F32 for every other (`d_dtype` and `accumulate` at run time).
template <int FA, int FB, int DT>
__global__ __launch_bounds__(kGemmThreads, 3) void gemm_nt_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                               void* __restrict__ Dv, const float* __restrict__ scale_a,
                                                               const float* __restrict__ scale_b, int M, int N, int K,
                                                               int tiles_m, int tiles_n, Fp8Out fp8, GemmExtras ex,
                                                               int d_dtype, int accumulate, uint32_t magic) {
    __shared__ __attribute__((aligned(16))) uint8_t sA[kBM * kBK];
    __shared__ __attribute__((aligned(16))) uint8_t sB[kBN * kBK];

    int pid_m, pid_n;
    tile_of_block(tiles_m, tiles_n, magic, pid_m, pid_n);
    const int m0 = pid_m * kBM, n0 = pid_n * kBN;

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;

    // global -> LDS assignment: 1024 16-byte chunks per operand tile, 4 per thread
    int ld_row[4], ld_kc[4];
    const uint8_t* a_ptr[4];
    const uint8_t* b_ptr[4];
    bool a_ok[4], b_ok[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = t + kGemmThreads * i;
        ld_row[i] = c >> 3;
        ld_kc[i] = c & 7;
        a_ok[i] = m0 + ld_row[i] < M;
        b_ok[i] = n0 + ld_row[i] < N;
        a_ptr[i] = A + (int64_t)(a_ok[i] ? m0 + ld_row[i] : 0) * K + ld_kc[i] * 16;
        b_ptr[i] = B + (int64_t)(b_ok[i] ? n0 + ld_row[i] : 0) * K + ld_kc[i] * 16;
    }

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    v4i ra[4], rb[4];
    const v4i zero = {0, 0, 0, 0};
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool kin = k0 + ld_kc[i] * 16 < K;
            ra[i] = (a_ok[i] && kin) ? *reinterpret_cast<const v4i*>(a_ptr[i] + k0) : zero;
            rb[i] = (b_ok[i] && kin) ? *reinterpret_cast<const v4i*>(b_ptr[i] + k0) : zero;
        }
    };

    const int frow = lane & 31;
    const int fk = (lane >> 5) * 2;

    fetch(0);
    for (int k0 = 0; k0 < K; k0 += kBK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<v4i*>(&sA[lds_off(ld_row[i], ld_kc[i])]) = ra[i];
            *reinterpret_cast<v4i*>(&sB[lds_off(ld_row[i], ld_kc[i])]) = rb[i];
        }
        __syncthreads();
        if (k0 + kBK < K) fetch(k0 + kBK);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            v8i fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ra_row = wm + i * 32 + frow, rb_row = wn + i * 32 + frow;
                const v4i a0 = *reinterpret_cast<const v4i*>(&sA[lds_off(ra_row, ks * 4 + fk)]);
                const v4i a1 = *reinterpret_cast<const v4i*>(&sA[lds_off(ra_row, ks * 4 + fk + 1)]);
                const v4i b0 = *reinterpret_cast<const v4i*>(&sB[lds_off(rb_row, ks * 4 + fk)]);
                const v4i b1 = *reinterpret_cast<const v4i*>(&sB[lds_off(rb_row, ks * 4 + fk + 1)]);
                fa[i] = (v8i){a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
                fb[i] = (v8i){b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma_32x32x64<FA, FB>(fb[j], fa[i], acc[i][j]);
        }
    }

    float alpha = descale_factor(scale_a, scale_b, ex.scale_inv);
    if (ex.bias) {   // uniform
        add_bias32<2, 2>(acc, alpha, ex.bias, ex.bias_dtype, N, n0 + wn, lane);
        alpha = 1.0f;
    }
    const int mb = m0 + wm, nb = n0 + wn;
    if constexpr (DT != NTFP8_F32) {
        constexpr int F = DT == NTFP8_OUT_E4M3 ? kE4M3 : kE5M2;
        const float scale_d = *fp8.scale;
        const uint32_t amax = store_wave_tile_fp8<F, 2, 2>(acc, static_cast<uint8_t*>(Dv), fp8.Dt, alpha, scale_d,
                                                           scale_is_degenerate(scale_d), M, N, mb, nb, lane);
        publish_amax(amax, fp8.ws);
    } else if (d_dtype == NTFP8_BF16) {
        store_wave_tile<NTFP8_BF16, false, 2, 2>(acc, Dv, alpha, M, N, mb, nb, lane);
    } else if (d_dtype == NTFP8_F16) {
        store_wave_tile<NTFP8_F16, false, 2, 2>(acc, Dv, alpha, M, N, mb, nb, lane);
    } else if (accumulate) {
        store_wave_tile<NTFP8_F32, true, 2, 2>(acc, Dv, alpha, M, N, mb, nb, lane);
    } else {
        store_wave_tile<NTFP8_F32, false, 2, 2>(acc, Dv, alpha, M, N, mb, nb, lane);
    }
}

template <int FA, int FB>
static void launch_plain_fmt(const GemmDesc& g, hipStream_t st) {
    const int tm = (g.M + kBM - 1) / kBM, tn = (g.N + kBN - 1) / kBN;
    const uint8_t* a = static_cast<const uint8_t*>(g.A);
    const uint8_t* b = static_cast<const uint8_t*>(g.B);
    const Fp8Out fp8 = {g.sd, static_cast<uint8_t*>(g.Dt), static_cast<Workspace*>(g.ws)};
    const GemmExtras ex = {g.bias, g.bias_dtype, g.scale_inv};
    auto go = [&](auto dt) {
        hipLaunchKernelGGL((gemm_nt_kernel<FA, FB, decltype(dt)::value>), dim3(tm * tn), dim3(kGemmThreads), 0, st, a, b, g.D, g.sa, g.sb,
                           g.M, g.N, g.K, tm, tn, fp8, ex, g.d_dtype, g.accumulate, magic_of((uint32_t)kGroupM * (uint32_t)tn));
    };
    if (g.d_dtype == NTFP8_OUT_E4M3) go(std::integral_constant<int, NTFP8_OUT_E4M3>{});
    else if (g.d_dtype == NTFP8_OUT_E5M2) go(std::integral_constant<int, NTFP8_OUT_E5M2>{});
    else go(std::integral_constant<int, NTFP8_F32>{});
}

int launch_plain(const GemmDesc& g, hipStream_t st) {
    (void)hipGetLastError();
    if (g.fmt_a == kE4M3) {
        if (g.fmt_b == kE4M3) launch_plain_fmt<kE4M3, kE4M3>(g, st);
        else launch_plain_fmt<kE4M3, kE5M2>(g, st);
    } else {
        if (g.fmt_b == kE4M3) launch_plain_fmt<kE5M2, kE4M3>(g, st);
        else launch_plain_fmt<kE5M2, kE5M2>(g, st);
    }
    return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}

}  // namespace ntfp8
