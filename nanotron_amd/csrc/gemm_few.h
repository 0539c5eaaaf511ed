// FP8 GEMM for a few rows of A (tokens) against a full-size B (weight), gfx950.  Included by gemm_few.hip.
//
// Bound by the latency of reading the weight: a 64-wide tile gives 4096 columns to 64 of 256 CUs, each walking all of K
// in turn behind barriers.  Here a workgroup computes 16 or 32 columns of D (256 workgroups for 4096), its eight waves take
// the K-tiles in turn, straight from memory into registers with four K-tiles in flight per wave, and their sums meet
// in LDS, added in the order of the waves.  16 rows, weight not in a cache, 64-wide tiles -> here, us: 4096 x 4096
// 11.3 -> 7.6, 4096 x 14336 31.1 -> 19.6, 1040 x 14336 30.2 -> 16.6, 6144 x 4096 11.9 -> 11.0, 8192 x 8192 23.2 -> 19.3
// (3.5 TB/s; every workgroup reads all of A, which is what the time grows with: one row of 4096 x 14336 takes 14.6).
#pragma once

namespace ntfp8 {

constexpr int kFewWaves = 8, kFewThreads = 64 * kFewWaves;

// MI: blocks of 16 rows of A (M <= 16 MI).  NJ: blocks of 16 columns of a workgroup.
template <int FA, int FB, int MI, int NJ>
__global__ __launch_bounds__(kFewThreads) void gemm_few_kernel(const BigProblem P) {
    constexpr int kAhead = 4;   // K-tiles a wave has in flight: 64 KB (NJ = 1) or 128 KB of B per workgroup
    constexpr int kColumns = 16 * NJ;
    __shared__ __attribute__((aligned(16))) float s_part[kFewWaves][16 * MI][kColumns + 4];
    const int M = P.M, N = P.N, K = P.K;
    const int n0 = blockIdx.x * kColumns;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, q = lane >> 4;

    // Rows past the end fall behind the descriptors and read as zeros; so do chunks at k >= K.  A lane's 32 bytes of a
    // K-tile are chunks q and q + 4 of its row, the same in A and B (the order of k inside a product is free), so that
    // a load takes 64 contiguous bytes of each row.
    const int KT = (K + kBK - 1) / kBK;
    constexpr uint32_t kNowhere = 0xfffffff0u;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(P.A, (uint32_t)M * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(P.B + (int64_t)n0 * K, (uint32_t)min(N - n0, kColumns) * (uint32_t)K);
    v4i fa[kAhead][MI][2], fb[kAhead][NJ][2];
    auto request = [&](int slot, int kt) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t k = (uint32_t)kt * kBK + h * 64 + q * 16;
            const bool in = k < (uint32_t)K;
#pragma unroll
            for (int j = 0; j < NJ; ++j) fb[slot][j][h] = reg_load16(rb, in ? (row + 16 * j) * (uint32_t)K + k : kNowhere, 0);
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[slot][i][h] = reg_load16(ra, in ? (row + 16 * i) * (uint32_t)K + k : kNowhere, 0);
        }
    };
    auto frag = [](const v4i (&x)[2]) -> v8i { return (v8i){x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w}; };

    v4f acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kAhead; ++s) request(s, wave + s * kFewWaves);
    for (int kt = wave; kt < KT; kt += kAhead * kFewWaves) {
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {   // (tiles past the end add zeros)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = mfma_16x16x128<FA, FB>(frag(fb[s][j]), frag(fa[s][i]), acc[i][j]);
            request(s, kt + (s + kAhead) * kFewWaves);
        }
    }

#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) *reinterpret_cast<v4f*>(&s_part[wave][16 * i + row][16 * j + 4 * q]) = acc[i][j];
    __syncthreads();
    const float alpha = descale_factor(P.scale_a, P.scale_b, P.ex.scale_inv);
    const int c = threadIdx.x % kColumns, n = n0 + c;
    if (n >= N) return;
    const float bias = P.ex.bias ? bias_at(P.ex.bias, P.ex.bias_dtype, n) : 0.0f;
    for (int m = threadIdx.x / kColumns; m < M; m += kFewThreads / kColumns) {
        float sum = s_part[0][m][c];
#pragma unroll
        for (int w = 1; w < kFewWaves; ++w) sum += s_part[w][m][c];
        float r = sum * alpha;
        if (P.ex.bias) r += bias;
        const int64_t at = (int64_t)m * N + n;
        if (P.d_dtype == NTFP8_BF16) static_cast<uint16_t*>(P.D)[at] = OutT<NTFP8_BF16>::cvt(r);
        else if (P.d_dtype == NTFP8_F16) static_cast<uint16_t*>(P.D)[at] = OutT<NTFP8_F16>::cvt(r);
        else if (P.accumulate) static_cast<float*>(P.D)[at] += r;
        else static_cast<float*>(P.D)[at] = r;
    }
}

}  // namespace ntfp8
