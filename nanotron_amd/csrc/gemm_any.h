// FP8 GEMM for any K and any pointer alignment (gfx950); included by gemm_any.hip.
//
// What the other kernels do not take: rows of A and B that start on no 16-byte boundary, because K is not a multiple
// of 16 (a weight gradient reduces over the tokens of the batch, and those are a multiple of nothing) or because a
// pointer is a view into the middle of something.
//
// The products run on V_MFMA_F32_32X32X16_BF16: every e4m3 and e5m2 value is exact in bf16, and the accumulated sum
// differs from the exact one by 7e-8 at K = 4096, as a chain of fp32 FMAs does (the fp8 instructions align the
// products of a step before they add them: 1.5e-5).  The conversion, one V_CVT_SCALEF32_PK_BF16_* per two values,
// issues beside the MFMAs.  Tile: (64 MB) x (64 MB) x 128 bytes of K, four waves of (32 MB) x (32 MB); two LDS stages
// with the next K-tile in registers and one barrier per K-tile.  Bound by the latency of a K-tile (load, deposit,
// barrier) on small shapes, by the LDS reads on large ones.  Against one output per thread, which this kernel replaced:
// 2304 x 1024 x 1021 6124 -> 18.5 us (261 TFLOP/s), 333 x 601 x 515 222 -> 7.9 us; 4096 x 4096 x 4095 767 TFLOP/s.
//
// Global loads are 16 bytes wide whatever the address (gfx950 serves misaligned ones); a chunk that reaches past its
// row is masked, one that reaches past the tensor is put together from bytes.
#pragma once

namespace ntfp8 {

constexpr int kAnyThreads = 256;
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef v4i v4i_any __attribute__((aligned(1)));

template <int F>
__device__ __forceinline__ v8bf fp8x8_to_bf16(uint32_t lo, uint32_t hi) {
    v2bf r[4];
    if constexpr (F == kE4M3) {
        r[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
        r[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
        r[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
        r[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    } else {
        r[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(lo, 1.0f, false);
        r[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(lo, 1.0f, true);
        r[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(hi, 1.0f, false);
        r[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(hi, 1.0f, true);
    }
    return (v8bf){r[0].x, r[0].y, r[1].x, r[1].y, r[2].x, r[2].y, r[3].x, r[3].y};
}

__device__ __forceinline__ v16f mfma_32x32x16_bf16(v8bf b_frag, v8bf a_frag, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(b_frag, a_frag, c, 0, 0, 0);   // result indexed [n][m]
}

// bytes k .. k + 15 of row `row` of an [R, K] operand; zero past the row or the operand.  `whole`: k + 16 <= K for
// every lane (uniform).
__device__ __forceinline__ v4i any_chunk(const uint8_t* __restrict__ P, int64_t R, int64_t K, int64_t row, int64_t k, bool whole) {
    v4i v = {0, 0, 0, 0};
    if (row >= R || k >= K) return v;
    const uint8_t* p = P + row * K + k;
    if (whole || k + 16 <= K) return *reinterpret_cast<const v4i_any*>(p);
    const int valid = (int)(K - k);   // 1 .. 15
    if (row * K + k + 16 <= R * K) {  // the bytes past the row belong to the next one: read and masked
        v = *reinterpret_cast<const v4i_any*>(p);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int nb = valid - 4 * w;
            v[w] &= nb >= 4 ? -1 : (nb <= 0 ? 0 : (int)((1u << (8 * nb)) - 1u));
        }
    } else {
#pragma unroll
        for (int b = 0; b < 15; ++b)
            if (b < valid) v[b >> 2] |= (int)p[b] << (8 * (b & 3));
    }
    return v;
}

// Output type and accumulation are run-time properties of a problem and a launch takes up to kBigMaxProblems of the same
// operand formats, as in the other tile kernels (BigLaunch, gemm_big.h): the two GEMMs of a small layer's backward share
// one launch.
template <int FA, int FB, int MB, bool kFp8Out>
__global__ __launch_bounds__(kAnyThreads) void gemm_any_kernel(const BigLaunch L) {
    constexpr int kT = 64 * MB;             // tile edge
    constexpr int kC = kT * 8 / kAnyThreads;   // 16-byte chunks per operand and thread
    __shared__ __attribute__((aligned(16))) uint8_t sA[2][kT * kBK];
    __shared__ __attribute__((aligned(16))) uint8_t sB[2][kT * kBK];

    int pid = blockIdx.x;
    if (gridDim.x % kXcds == 0) pid = (pid % kXcds) * (gridDim.x / kXcds) + pid / kXcds;   // an XCD works on a run of tiles
    const Picked G = pick_problem(L, pid);
    const BigProblem& P = L.p[G.which];
    const uint8_t* __restrict__ A = G.A;
    const uint8_t* __restrict__ B = G.B;
    const int M = G.M, N = G.N, K = G.K;
    pid -= G.tile_begin;
    int pid_m, pid_n;
    tile_in_group(pid, G.tiles_m, G.tiles_n, G.magic, pid_m, pid_n);
    const int m0 = pid_m * kT, n0 = pid_n * kT;
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wm = (wave >> 1) * (32 * MB), wn = (wave & 1) * (32 * MB);

    v16f acc[MB][MB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    v4i ra[kC], rb[kC];
    auto fetch = [&](int64_t k0) {
        const bool whole = k0 + kBK <= K;
#pragma unroll
        for (int i = 0; i < kC; ++i) {
            const int c = t + kAnyThreads * i;
            ra[i] = any_chunk(A, M, K, (int64_t)m0 + (c >> 3), k0 + (c & 7) * 16, whole);
            rb[i] = any_chunk(B, N, K, (int64_t)n0 + (c >> 3), k0 + (c & 7) * 16, whole);
        }
    };
    fetch(0);
    int s = 0;
    for (int64_t k0 = 0; k0 < K; k0 += kBK, s ^= 1) {
#pragma unroll
        for (int i = 0; i < kC; ++i) {
            const int c = t + kAnyThreads * i;
            *reinterpret_cast<v4i*>(&sA[s][lds_off(c >> 3, c & 7)]) = ra[i];
            *reinterpret_cast<v4i*>(&sB[s][lds_off(c >> 3, c & 7)]) = rb[i];
        }
        // one barrier per K-tile: the stage written in the next trip was last read before this barrier
        __syncthreads();
        if (k0 + kBK < K) fetch(k0 + kBK);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            // a lane's 16 bytes feed two MFMAs of 16 k each; which k an MFMA step covers does not matter as long as
            // both operands agree
            const int kc = ks * 2 + (lane >> 5);
            v4i a[MB], b[MB];
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                a[i] = *reinterpret_cast<const v4i*>(&sA[s][lds_off(wm + i * 32 + (lane & 31), kc)]);
                b[i] = *reinterpret_cast<const v4i*>(&sB[s][lds_off(wn + i * 32 + (lane & 31), kc)]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v8bf fa[MB], fb[MB];
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    fa[i] = fp8x8_to_bf16<FA>((uint32_t)a[i][2 * h], (uint32_t)a[i][2 * h + 1]);
                    fb[i] = fp8x8_to_bf16<FB>((uint32_t)b[i][2 * h], (uint32_t)b[i][2 * h + 1]);
                }
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < MB; ++j) acc[i][j] = mfma_32x32x16_bf16(fb[j], fa[i], acc[i][j]);
            }
        }
    }

    float alpha = descale_factor(P.scale_a, P.scale_b, P.ex.scale_inv);
    if (P.ex.bias) {   // uniform
        add_bias32<MB, MB>(acc, alpha, P.ex.bias, P.ex.bias_dtype, N, n0 + wn, lane);
        alpha = 1.0f;
    }
    const bool d_aligned = (reinterpret_cast<uintptr_t>(P.D) & 15) == 0;
    const int mb = m0 + wm, nb = n0 + wn;
    if constexpr (kFp8Out) {
        const float scale_d = *P.fp8.scale;
        const bool slow = scale_is_degenerate(scale_d);
        uint8_t* D = static_cast<uint8_t*>(P.D);
        const uint32_t amax = P.d_dtype == NTFP8_OUT_E4M3
                                  ? store_wave_tile_fp8<kE4M3, MB, MB>(acc, D, P.fp8.Dt, alpha, scale_d, slow, M, N, mb, nb, lane, d_aligned)
                                  : store_wave_tile_fp8<kE5M2, MB, MB>(acc, D, P.fp8.Dt, alpha, scale_d, slow, M, N, mb, nb, lane, d_aligned);
        publish_amax(amax, P.fp8.ws);
        finish_fp8(L, P.fp8.ws, blockIdx.x);
    } else if (P.d_dtype == NTFP8_BF16) {
        store_wave_tile<NTFP8_BF16, false, MB, MB>(acc, P.D, alpha, M, N, mb, nb, lane, d_aligned);
    } else if (P.d_dtype == NTFP8_F16) {
        store_wave_tile<NTFP8_F16, false, MB, MB>(acc, P.D, alpha, M, N, mb, nb, lane, d_aligned);
    } else if (P.accumulate) {
        store_wave_tile<NTFP8_F32, true, MB, MB>(acc, P.D, alpha, M, N, mb, nb, lane, d_aligned);
    } else {
        store_wave_tile<NTFP8_F32, false, MB, MB>(acc, P.D, alpha, M, N, mb, nb, lane, d_aligned);
    }
}

}  // namespace ntfp8
