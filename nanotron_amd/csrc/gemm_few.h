// FP8 GEMM for a few rows of A (tokens) against a full-size B (weight), gfx950.  Included by gemm_few.hip.
//
// Bound by reading the weight: a 64-wide tile gives 4096 columns to 64 of 256 CUs, each walking all of K in turn behind
// barriers.  Here a workgroup computes 16 or 32 columns of D (256 workgroups for 4096), its eight waves take the K-tiles in
// turn with four in flight per wave, and their sums meet in LDS, added in the order of the waves.  The weight goes straight
// into LDS, 8 rows of 128 bytes a load; as fragments into registers a load was 16 rows of 64 bytes, half a line each (a
// kernel that only reads a 4096 x 14336 weight: 15.0 / 19.8 us).  16 rows, weight not in a cache, through registers / LDS, us:
// 6144 x 4096 10.3 / 8.7, 4096 x 4096 7.6 / 7.1, 4096 x 14336 17.2 / 15.1 (3.9 TB/s), 8192 x 4096 11.1 / 9.8; in the memory-side
// cache 8.6 / 6.2, 6.6 / 5.3, 15.8 / 12.0, 8.8 / 7.0.  (Streaming loads: 5 % less from memory, 8 to 14 % more from the cache.)
// Every workgroup reads all of A, which is what the time grows with.
#pragma once

namespace ntfp8 {

constexpr int kFewWaves = 8, kFewThreads = 64 * kFewWaves;

// MI: blocks of 16 rows of A (M <= 16 MI).  NJ: blocks of 16 columns of a workgroup.
template <int FA, int FB, int MI, int NJ>
__global__ __launch_bounds__(kFewThreads) void gemm_few_kernel(const BigProblem P) {
    constexpr int kAhead = 4;   // K-tiles a wave has in flight: 64 KB (NJ = 1) or 128 KB of B per workgroup
    constexpr int kColumns = 16 * NJ;
    constexpr int kLoads = 2 * NJ + 2 * MI;   // of a K-tile
    __shared__ __attribute__((aligned(1024))) uint8_t s_b[kFewWaves][kAhead][kColumns * kBK];
    __shared__ __attribute__((aligned(16))) float s_part[kFewWaves][16 * MI][kColumns + 4];
    const int M = P.M, N = P.N, K = P.K;
    const int n0 = blockIdx.x * kColumns;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, q = lane >> 4;

    // Rows past the end fall behind the descriptors and read as zeros; so do chunks at k >= K.  A lane's 32 bytes of a
    // K-tile are chunks q and q + 4 of its row, the same in A and B (the order of k inside a product is free).  B passes
    // through LDS (swizzled as in gemm_big.h), 8 whole lines of 128 bytes a load; a wave's stages are its own, so nothing
    // but its memory counter stands between a load and the reads of it.
    const int KT = (K + kBK - 1) / kBK;
    constexpr uint32_t kNowhere = 0xfffffff0u;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(P.A, (uint32_t)M * (uint32_t)K);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(P.B + (int64_t)n0 * K, (uint32_t)min(N - n0, kColumns) * (uint32_t)K);
    v4i fa[kAhead][MI][2];
    auto request = [&](int slot, int kt) {
#pragma unroll
        for (int i = 0; i < 2 * NJ; ++i) {   // rows 8 i + lane / 8: position p of a row receives chunk p ^ swz16(row)
            const uint32_t k = (uint32_t)kt * kBK + (((lane & 7) ^ (lane >> 3) ^ (i & 1)) << 4);
            lds_load16(rb, (lds_ptr)(uintptr_t)&s_b[wave][slot][i * 1024], k < (uint32_t)K ? (8 * i + (lane >> 3)) * (uint32_t)K + k : kNowhere, 0);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t k = (uint32_t)kt * kBK + h * 64 + q * 16;
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[slot][i][h] = reg_load16(ra, k < (uint32_t)K ? (row + 16 * i) * (uint32_t)K + k : kNowhere, 0);
        }
    };
    auto frag = [](const v4i (&x)[2]) -> v8i { return (v8i){x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w}; };

    v4f acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        request(s, wave + s * kFewWaves);
        sched_fence();   // the wait below counts loads: those of a slot have to be older than the next slot's
    }
    const float alpha = descale_factor(P.scale_a, P.scale_b, P.ex.scale_inv);   // (behind the first requests)
    const int rd0 = lds_off16(row, q), rd1 = lds_off16(row, q + 4);
    for (int kt = wave; kt < KT; kt += kAhead * kFewWaves) {
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {   // (tiles past the end add zeros)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kAhead - 1) * kLoads) : "memory");   // all but the tiles requested since
            v4i fb[NJ][2];
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                fb[j][0] = *reinterpret_cast<const v4i*>(&s_b[wave][s][rd0 + j * 2048]);
                fb[j][1] = *reinterpret_cast<const v4i*>(&s_b[wave][s][rd1 + j * 2048]);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = mfma_16x16x128<FA, FB>(frag(fb[j]), frag(fa[s][i]), acc[i][j]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage has been read
            sched_fence();
            request(s, kt + (s + kAhead) * kFewWaves);
            sched_fence();
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last requests write zeros into stages nobody reads again)

#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) *reinterpret_cast<v4f*>(&s_part[wave][16 * i + row][16 * j + 4 * q]) = acc[i][j];
    __syncthreads();
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
