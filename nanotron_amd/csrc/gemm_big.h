// Large-tile FP8 GEMM kernel for gfx950; included by gemm.hip after the shared helpers.
//
// Block tile (32 MI) x 256 x 128 bytes of K, four waves in a 2 x 2 arrangement, one wave per
// SIMD.  Each wave owns (16 MI) x 128 outputs as MI x 8 accumulator blocks of V_MFMA_F32_16X16X128_F8F6F4
// (MI = 8: 256-row block tile, 256 accumulator registers per lane; MI = 4: 128-row block tile).
//
// Data movement per K-tile: every wave brings a quarter of the A and B tiles from global memory into
// LDS (16 bytes per lane, XOR-swizzled), reads its MI A fragments from LDS once and keeps them in
// registers, and reads its 8 B fragments ahead of their use (below).  One MFMA
// group = the MI MFMAs that share one B fragment.
//
// Loads go straight from memory into LDS.  Whole tiles (MI = 8): two LDS stages and two workgroup barriers per K-tile.
//   * all B fragments of a tile have registers of their own and are read during its first 24 MFMAs; the first barrier
//     (behind MFMA 26 of 64) so releases the stage early, and the loads of tile kt + 2 have the rest of this K-tile and most
//     of the next to arrive;
//   * the second barrier (behind group 5) publishes tile kt + 1, whose A fragments are read during groups 6 and 7: these
//     are issued interleaved, two MFMAs per A fragment, and the fragment register, dead after them, is refilled with the
//     same fragment of tile kt + 1, so one set of A registers suffices.
// Bound by the package power limit and by issue slots: 191 instructions per K-tile of 64 MFMAs became 161, and no operand
// byte passes through a register on its way to LDS.  us, loads kept in registers for a K-tile / straight into LDS:
// 4096 x 4096 x 4096 50.6 / 48.5, 4096 x 14336 x 4096 179 / 173, 4096 x 4096 x 14336 165 / 160; both operands transposed
// beside dgrad, 4096 tokens: 4096 -> 4096 110 / 104, 4096 -> 14336 384 / 362, 14336 -> 4096 387 / 372.
// Half tiles (MI = 4): three stages, one barrier behind group 5 that releases the stage of tile kt and publishes tile kt + 1;
// B fragments in a ring of four, read three groups ahead.
//
// Instantiations beside the operand formats and MI: kFp8Out (the outputs are fp8 bytes, cast in the
// epilogue, with an optional transposed copy and the amax of the results) and kBT (the B operands are
// given as their transposes, [K, N] tensors, and gathered from LDS with the transposing read).
#pragma once
#include "reduce.h"

namespace ntfp8 {

// Profiling build (-DNTFP8_STAMPS, libntfp8_stamps.so): every workgroup of gemm_nt_big_kernel leaves five readings of
// the 100 MHz wall clock (kernel entry, first tile published, end of the K loop, last store issued, stores drained), the
// shader-clock cycle counter at both ends of the K loop and the identity of its CU in a table that
// ntfp8_debug_stamps() copies out.  The product library is built without it.
#ifdef NTFP8_STAMPS
constexpr int kStampSlots = 16384;
__device__ unsigned long long g_stamps[kStampSlots * 8];
// 1: workgroups take the tiles in launch order, i.e. every XCD gets every eighth tile and touches all operand panels
// (what the fetch traffic costs; set with ntfp8_debug_set_tile_order)
__device__ int g_plain_tile_order = 0;
#define NTFP8_STAMP(var) var = wall_clock64()
#define NTFP8_CYCLES(var) var = __builtin_readcyclecounter()
#else
#define NTFP8_STAMP(var) (void)0
#define NTFP8_CYCLES(var) (void)0
#endif

constexpr int kBigN = 256;
constexpr int kBigWaves = 4, kBigThreads = kBigWaves * 64;
constexpr int kBigNJ = 8;              // 16-column accumulator blocks per wave: 128 columns
constexpr int kBigLB = kBigN / 8 / kBigWaves;   // 1 KB wave-level loads of the B tile per wave per stage

// Swizzle for 16-row fragments: the 16 lanes that read chunk c of rows r .. r + 15 hit 16 distinct
// 16-byte bank groups when the chunk index is XORed with (row mod 8) ^ (bit 3 of row).
__device__ __forceinline__ int swz16(int row) { return (row & 7) ^ ((row >> 3) & 1); }
__device__ __forceinline__ int lds_off16(int row, int kc) { return row * kBK + ((kc ^ swz16(row)) << 4); }

template <int FA, int FB>
__device__ __forceinline__ v4f mfma_16x16x128(v8i b_frag, v8i a_frag, v4f c) {
    // B fragment first: the 16 x 16 result block is indexed [n][m], so a lane owns 4 consecutive n
    // (n = 4 (lane / 16) + r) of one output row m = lane % 16.
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b_frag, a_frag, c, FB, FA, 0, 0, 0, 0);
}
// rows (groups of 16 lanes) 1 and 3 of x <-> rows 0 and 2 of y (V_PERMLANE16_SWAP)
__device__ __forceinline__ void swap_rows16(uint32_t& x, uint32_t& y) {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    const v2u r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r.x;
    y = r.y;
}
// 16 bytes per lane from global memory into registers; offsets past the descriptor read as zero
template <int kPolicy = 0>
__device__ __forceinline__ v4i reg_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kPolicy));
}
__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }
// 16 bytes of output to global memory, written through to memory as they are issued (sc0 sc1) and marked streaming
// (nt).  An ordinary store leaves its line dirty in the XCD's L2; a tile's worth of output per CU then fills that L2,
// and the lines are written back in one burst when the kernel ends.  Written through, the output drains while the
// other waves still compute: 2.5 us less per round of tiles (4096^3: 58.0 -> 55.5 us; `nt` alone changes nothing).
// The two wait states belong to the store: its data registers are still being read then, and the compiler, which keeps such
// a distance behind stores of its own, does not see this one (without them the next block's first product overwrote a word
// of four lanes now and then).
__device__ __forceinline__ void store16_through(void* p, v4i v) {
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

// 16 / 4 bytes per lane to global memory through a buffer descriptor; offsets past its size are dropped.  Cache policy
// of the builtin's last argument on gfx950: bit 0 = sc0, bit 1 = nt, bit 4 = sc1 (written through, as store16_through).
constexpr int kStoreThrough = 1 | 2 | 16, kStreaming = 2;
template <int kPolicy = kStoreThrough>
__device__ __forceinline__ void reg_store16(__amdgpu_buffer_rsrc_t r, uint32_t voff, v4i data) {
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, data), r, voff, 0, kPolicy);
}
__device__ __forceinline__ void reg_store4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t data) {
    __builtin_amdgcn_raw_buffer_store_b32(data, r, voff, 0, kStoreThrough);
}
constexpr uint32_t kDropped = 0xfffffff0u;   // past every descriptor
// within groups of 16 lanes: lanes 8 .. 15 of x <-> lanes 0 .. 7 of y
__device__ __forceinline__ void swap_octets(uint32_t& x, uint32_t& y) {
    const int a = (int)x, b = (int)y;
    x = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false);   // row_ror:8 into banks 2, 3
    y = (uint32_t)__builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false);   // row_ror:8 into banks 0, 1
}

// `count` rows from m_base on of a row-major M x N output: rows past its end fall behind the descriptor
constexpr int kMaxColumns = 1 << 22;   // 128 rows within reach of 32-bit offsets
template <typename O>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(O* D, int M, int N, int m_base, int count) {
    // (a clamp is a vector instruction, and through a descriptor in vector registers the compiler accesses in a loop)
    const uint32_t rows = (uint32_t)__builtin_amdgcn_readfirstlane(max(0, min(M - m_base, count)));
    return make_rsrc(D + (int64_t)m_base * N, rows * (uint32_t)N * (uint32_t)sizeof(O));
}

// Epilogue of one wave: MI x NJ accumulator blocks of 16 x 16, block (i, j) at rows m_base + 16 i,
// columns n_base + 16 j.  Descale, optional fp32 accumulate, one rounding, store.
// kBias: bv[j][e] = bias of column n_base + 16 j + 4 (lane / 16) + e, added to the descaled value before the rounding.
template <int DT, bool kAcc, int MI, int NJ, bool kBias = false>
__device__ __forceinline__ void store_wave_tile16(const v4f (&acc)[MI][NJ], void* __restrict__ Dv, float alpha, int M,
                                                  int N, int m_base, int n_base, int lane, const float (*bv)[4] = nullptr) {
    typedef typename OutT<DT>::type O;
    O* D = static_cast<O*>(Dv);
    const int mrow = lane & 15, q = lane >> 4;
    // element e of block (i, j): descaled, plus bias if there is one (two separately rounded fp32 operations)
    auto val = [&](int i, int j, int e) -> float {
        if constexpr (kBias) return acc[i][j][e] * alpha + bv[j][e];
        else return acc[i][j][e] * alpha;
    };
    if constexpr (DT != NTFP8_F32 && NJ != 4) {
        // 16-bit outputs: a lane's 4 consecutive n are only 8 bytes.  Exchanging registers of two
        // neighbouring blocks between lane rows gives every lane 8 consecutive n (16 bytes) of one
        // block, and lane rows r / r + 2 together a full 32-byte sector per output row, which the
        // memory side writes without read-modify-write traffic.
        if ((N & 7) == 0) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int m = m_base + i * 16 + mrow;
#pragma unroll
                for (int j = 0; j < NJ; j += 2) {
                    uint32_t x0 = OutT<DT>::pack2(val(i, j, 0), val(i, j, 1));
                    uint32_t x1 = OutT<DT>::pack2(val(i, j, 2), val(i, j, 3));
                    uint32_t y0 = OutT<DT>::pack2(val(i, j + 1, 0), val(i, j + 1, 1));
                    uint32_t y1 = OutT<DT>::pack2(val(i, j + 1, 2), val(i, j + 1, 3));
                    swap_rows16(x0, y0);
                    swap_rows16(x1, y1);
                    // lane row q now holds n 8 (q / 2) .. + 7 of block j + (q & 1): x = first four, y = last four
                    const int n = n_base + (j + (q & 1)) * 16 + (q >> 1) * 8;
                    if (m < M && n < N)
                        store16_through(D + (int64_t)m * N + n, (v4i){(int)x0, (int)x1, (int)y0, (int)y1});
                }
            }
            return;
        }
    }
    if constexpr (DT != NTFP8_F32 && NJ == 4) {
        // The same, and exchanging words between lanes l and l ^ 8 of two such pairs, a store covers 64 columns, a whole line, of 8 rows.
        // (us, half lines of 16 rows / this: bf16 1021 x 2304 x 1024 with bias 9.5 / 8.9, 3000 x 1000 x 1024 10.7 / 9.6,
        // most shapes the same; the 256-wide tiles the same everywhere)
        if ((N & 7) == 0 && N < kMaxColumns) {
            const __amdgpu_buffer_rsrc_t rd = rows_rsrc(D, M, N, m_base, 16 * MI);
            // lane row q holds n 8 (q / 2) .. + 7 of block j + (q & 1), lanes 8 .. 15 of it those of the pair behind
            const int col = n_base + ((mrow >> 3) * 2 + (q & 1)) * 16 + (q >> 1) * 8;
            const uint32_t step = 8u * (uint32_t)N * 2u;
            uint32_t at = ((uint32_t)(mrow & 7) * (uint32_t)N + (uint32_t)col) * 2u;
#pragma unroll
            for (int i = 0; i < MI; ++i, at += 2 * step) {
#pragma unroll
                for (int j0 = 0; j0 < NJ; j0 += 4) {
                    uint32_t w[2][4];
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const int j = j0 + 2 * p;
                        uint32_t x0 = OutT<DT>::pack2(val(i, j, 0), val(i, j, 1));
                        uint32_t x1 = OutT<DT>::pack2(val(i, j, 2), val(i, j, 3));
                        uint32_t y0 = OutT<DT>::pack2(val(i, j + 1, 0), val(i, j + 1, 1));
                        uint32_t y1 = OutT<DT>::pack2(val(i, j + 1, 2), val(i, j + 1, 3));
                        swap_rows16(x0, y0);
                        swap_rows16(x1, y1);
                        w[p][0] = x0, w[p][1] = x1, w[p][2] = y0, w[p][3] = y1;
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) swap_octets(w[0][e], w[1][e]);
                    const bool in = col + j0 * 16 < N;
                    reg_store16(rd, in ? at + j0 * 32 : kDropped, (v4i){(int)w[0][0], (int)w[0][1], (int)w[0][2], (int)w[0][3]});
                    reg_store16(rd, in ? at + step + j0 * 32 : kDropped, (v4i){(int)w[1][0], (int)w[1][1], (int)w[1][2], (int)w[1][3]});
                }
                sched_fence();
            }
            return;
        }
    }
    if constexpr (DT == NTFP8_F32) {
        // A lane's 4 consecutive n are 16 bytes, the four lane rows together 64 bytes of an output row, half a line.
        // Exchanging words between lanes l and l ^ 8 of two neighbouring blocks, a store (or the load of the accumulator)
        // covers 32 columns, a whole line, of 8 rows.  Rows of whole 64-byte pieces are written through as 16-bit outputs are,
        // or, where the line has just been read for the accumulation, read and written with the streaming hint alone; others
        // keep ordinary accesses, which put the pieces together in the L2.  us, half lines and ordinary accesses / here:
        //   2048 x 2048 x 2048  14.3 / 12.7     14336 x 4096 x 4096, both transposed  211 / 195, accumulated  257 / 232
        //   4096 x 4096 x 14336 with that weight gradient  369 / 358, accumulated  413 / 386
        //   rows of 64-byte pieces  4096 x 4112 x 512  32.6 / 28.0, accumulated  57.7 / 48.0 (written through 56.8)
        //   others  4096 x 4104 x 512  32.3 / 31.4 (written through 43.6)
        if ((N & (NJ == 4 ? 3 : 15)) == 0 && N < kMaxColumns) {   // (NJ = 8: no registers for two kinds of accesses)
            const __amdgpu_buffer_rsrc_t rd = rows_rsrc(D, M, N, m_base, 16 * MI);
            const int col = n_base + (mrow >> 3) * 16 + q * 4;
            const uint32_t step = 8u * (uint32_t)N * 4u;
            auto rows = [&](auto policy_tag) {
                constexpr int kPolicy = decltype(policy_tag)::value;
                uint32_t at = ((uint32_t)(mrow & 7) * (uint32_t)N + (uint32_t)col) * 4u;
#pragma unroll
                for (int i = 0; i < MI; ++i, at += 2 * step) {
                    v4f old[NJ];   // all of a row block's old values are requested before the first one is needed
                    if constexpr (kAcc) {
#pragma unroll
                        for (int j = 0; j < NJ; ++j)
                            old[j] = __builtin_bit_cast(v4f, reg_load16<kPolicy>(rd, col + (j & ~1) * 16 < N ? at + (j & 1) * step + (j & ~1) * 64 : kDropped, 0));
                    }
#pragma unroll
                    for (int j = 0; j < NJ; j += 2) {
                        v4f x, y;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            uint32_t a = __float_as_uint(val(i, j, e)), b = __float_as_uint(val(i, j + 1, e));
                            swap_octets(a, b);
                            x[e] = __uint_as_float(a), y[e] = __uint_as_float(b);
                        }
                        if constexpr (kAcc) x = x + old[j], y = y + old[j + 1];
                        const bool in = col + j * 16 < N;
                        reg_store16<kPolicy>(rd, in ? at + j * 64 : kDropped, __builtin_bit_cast(v4i, x));
                        reg_store16<kPolicy>(rd, in ? at + step + j * 64 : kDropped, __builtin_bit_cast(v4i, y));
                        sched_fence();
                    }
                    // (values of several row blocks at once do not fit the registers)
                }
            };
            if (NJ != 4 || (N & 15) == 0) rows(std::integral_constant<int, kAcc ? kStreaming : kStoreThrough>{});   // uniform
            else rows(std::integral_constant<int, 0>{});
            return;
        }
    }
    const bool vec_ok = (N & 3) == 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m_base + i * 16 + mrow;
        if (m >= M) continue;
        // accumulate: all of a row block's old values are requested before the first one is needed
        v4f old[NJ];
        if constexpr (kAcc) {
            if (vec_ok) {
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int n = n_base + j * 16 + q * 4;
                    old[j] = n + 3 < N ? *reinterpret_cast<const v4f*>(static_cast<const float*>(Dv) + (int64_t)m * N + n)
                                       : (v4f){0.f, 0.f, 0.f, 0.f};
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int n = n_base + j * 16 + q * 4;
            if (n >= N) continue;
            O* dp = D + (int64_t)m * N + n;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = val(i, j, e);
            if (vec_ok && n + 3 < N) {
                if constexpr (DT == NTFP8_F32) {
                    v4f o = {v[0], v[1], v[2], v[3]};
                    if constexpr (kAcc) o = o + old[j];
                    // (rows that end inside a 64-byte piece, and rows too wide for the descriptors above: ordinary stores, as there)
                    *reinterpret_cast<v4f*>(dp) = o;
                } else {
                    *reinterpret_cast<uint2*>(dp) = make_uint2(OutT<DT>::pack2(v[0], v[1]), OutT<DT>::pack2(v[2], v[3]));
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (n + e < N) {
                        if constexpr (DT == NTFP8_F32) {
                            float o = v[e];
                            if constexpr (kAcc) o = o + dp[e];
                            dp[e] = o;
                        } else {
                            dp[e] = OutT<DT>::cvt(v[e]);
                        }
                    }
                }
            }
        }
    }
}

// fp8 epilogue of one wave (layout as store_wave_tile16); returns the lane's max|r| as a bit pattern.
// Shapes: N a multiple of 16, M a multiple of 4, M N < 2^32 (the launcher sends other shapes to the small kernel).
// A lane's 4 consecutive n of a block are one word of D.  Row-major bytes: a 4 x 4 exchange of words between the
// four lane rows and four neighbouring blocks gives lane row q the 16 consecutive n of block j0 + q, one 16-byte
// store per lane and 64 contiguous bytes per output row and instruction.  Transposed bytes: a 4 x 4 byte transpose
// inside each quad of lanes (4 consecutive m) turns the word into 4 consecutive m of one n.
// All stores go through buffer descriptors of M N bytes: rows and columns past the end get an offset that falls outside
// and are dropped.  (Their own offsets would not do: they run past M N by up to 255 rows, and past 2^32, to the first rows
// again, where M N is close to it.)  Nothing is predicated, which keeps the scalar registers of the epilogue (and with
// them the register budget of the K loop before it) small.
// Accumulators past M and past N stay out of the amax: they hold zeros times whatever the other operand holds (NaN
// against an infinite code), plus the bias, or, where an operand is read through the transposing loads and wraps
// into its next row, arbitrary values.  N is a multiple of 16, so a block's columns are in or out together, uniformly
// for the wave; rows are masked lane by lane.  (By selects: with a branch per block 41 shapes of 256 to 512 256-wide tiles
// took 65.2 us on average, with these 64.1, without a mask about the same.)
template <int F, int MI, int NJ, bool kBias = false>
__device__ __forceinline__ uint32_t store_wave_tile16_fp8(const v4f (&acc)[MI][NJ], uint8_t* __restrict__ D,
                                                          uint8_t* __restrict__ Dt, float alpha, float scale_d, bool slow,
                                                          int M, int N, int m_base, int n_base, int lane,
                                                          const float (*bv)[4] = nullptr) {
    auto val = [&](int i, int j, int e) -> float {
        if constexpr (kBias) return acc[i][j][e] * alpha + bv[j][e];
        else return acc[i][j][e] * alpha;
    };
    static_assert(NJ % 4 == 0, "blocks are exchanged four at a time");
    const int mrow = lane & 15, q = lane >> 4;
    uint32_t amax = 0;
    const uint32_t bytes = (uint32_t)M * (uint32_t)N;
    const __amdgpu_buffer_rsrc_t rd = make_rsrc(D, bytes);
    const __amdgpu_buffer_rsrc_t rt = make_rsrc(Dt, Dt ? bytes : 0u);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m_base + i * 16 + mrow;
        const int mq = m & ~3;
        uint32_t w[NJ], row_max = 0;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            uint32_t a = 0;
            w[j] = quant4<F>(val(i, j, 0), val(i, j, 1), val(i, j, 2), val(i, j, 3), scale_d, slow, a);
            row_max = max(row_max, a & (n_base + j * 16 < N ? ~0u : 0u));
        }
        amax = max(amax, m < M ? row_max : 0u);
        if (Dt) {   // uniform
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const uint32_t t = quad_transpose_bytes(w[j], lane);
                const int nt = n_base + j * 16 + q * 4 + (lane & 3);
                reg_store4(rt, m < M && n_base + j * 16 < N ? (uint32_t)nt * (uint32_t)M + (uint32_t)mq : kDropped, t);
            }
        }
#pragma unroll
        for (int j0 = 0; j0 < NJ; j0 += 4) {
            uint32_t x0 = w[j0], x1 = w[j0 + 1], x2 = w[j0 + 2], x3 = w[j0 + 3];
            swap_rows16(x0, x1);   // lane rows 1, 3 of a word <-> rows 0, 2 of the next block's word
            swap_rows16(x2, x3);
            swap_halves(x0, x2);   // lane rows 2, 3 <-> rows 0, 1 two blocks further on
            swap_halves(x1, x3);
            // lane row q now holds n 0-3, 4-7, 8-11, 12-15 of block j0 + q
            const int n = n_base + (j0 + q) * 16;
            reg_store16(rd, m < M && n < N ? (uint32_t)m * (uint32_t)N + (uint32_t)n : kDropped, (v4i){(int)x0, (int)x1, (int)x2, (int)x3});
        }
    }
    return amax;
}

// Launch geometry, computed on the host.  The first `full_blocks` tiles (in grouped order) are computed
// whole by the MI = 8 kernel.  If the tile count leaves a partial last round over the CUs, the
// remaining `tail_tiles` tiles are computed in parts by a second launch, so that the last round is shorter: two 128-row halves
// each by the MI = 4 kernel, or four or eight parts by the tiles of gemm_mid.h.
//
// One launch can carry several independent GEMMs of the same operand formats (the dgrad and wgrad of a
// layer, say): their tiles form one list, longest K first, so that the rounds of one problem fill up
// with tiles of the next instead of ending in a partial round and a kernel boundary each.
struct BigProblem {
    // what a workgroup needs before its first load (pick_problem)
    const uint8_t* A;
    const uint8_t* B;
    const float* scale_a;
    const float* scale_b;
    int M, N, K;
    int tiles_m, tiles_n;   // in the launch's tile size
    uint32_t magic;         // magic_of(kGroupM tiles_n)
    int tile_begin;         // position of this problem's first tile in the launch's tile list
    int at;                 // A is given as [K, M] row-major (its transpose); only together with bt
    int bt;                 // B is given as [K, N] row-major (its transpose)
    // and behind its K loop
    int d_dtype;            // NTFP8_F32 / NTFP8_F16 / NTFP8_BF16 / NTFP8_OUT_E4M3 / NTFP8_OUT_E5M2
    int accumulate;         // fp32 outputs only: D += result
    void* D;
    Fp8Out fp8;             // fp8 outputs only
    GemmExtras ex;          // bias, inverse-scale flag
};
constexpr int kBigMaxProblems = 4;
struct BigLaunch {
    BigProblem p[kBigMaxProblems];
    int count;
    int full_blocks;        // tiles (of the whole list) computed whole
    int tail_tiles;         // tiles at the end of the list computed in parts
    int round_size;         // workgroups resident at once
    uint32_t round_magic;   // magic_of(round_size)
    // a launch of one problem with fp8 outputs: the workgroup that finishes last (of fin_blocks, over both launches of a
    // call with a tail) turns the collected maxima into the output role's bookkeeping (0: left in the workspace)
    int fin_blocks;
    ScalarIO fin;
};

// The problem that tile `pid` of the launch's list belongs to, as far as a workgroup needs it before its first load.  The fields
// of the first two problems are read at once and chosen from: looked up by number they come in three dependent trips (which
// problem, its sizes, its pointers) to a launch's arguments, which are in no cache.  us, looked up and tiles found by
// divisions / here: 512 x 512 x 512 3.97 / 3.65, 2048 x 1024 x 1024 5.89 / 5.56, 1021 x 2304 x 1024 7.78 / 7.40, 4096 x 4096 x 4096
// 47.5 / 46.8, dgrad and wgrad of 256 x 256 x 256 4.05 / 3.68.
struct Picked {
    const uint8_t *A, *B;
    const float *scale_a, *scale_b;
    int M, N, K, tiles_m, tiles_n, tile_begin, at, bt, which;
    uint32_t magic;
};
__device__ __forceinline__ Picked pick_problem(const BigLaunch& L, int pid) {
    Picked r = {};
    auto look = [&](int i, bool take) {
        const BigProblem& p = L.p[i];
        r.A = take ? p.A : r.A, r.B = take ? p.B : r.B;
        r.scale_a = take ? p.scale_a : r.scale_a, r.scale_b = take ? p.scale_b : r.scale_b;
        r.M = take ? p.M : r.M, r.N = take ? p.N : r.N, r.K = take ? p.K : r.K;
        r.tiles_m = take ? p.tiles_m : r.tiles_m, r.tiles_n = take ? p.tiles_n : r.tiles_n;
        r.magic = take ? p.magic : r.magic, r.tile_begin = take ? p.tile_begin : r.tile_begin;
        r.at = take ? p.at : r.at, r.bt = take ? p.bt : r.bt;
        r.which = take ? i : r.which;
    };
    look(0, true);
    look(1, L.count > 1 && pid >= L.p[1].tile_begin);
    if (L.count > 2)   // (no registers for the fields of all of them at once)
        for (int i = 2; i < L.count; ++i) look(i, pid >= L.p[i].tile_begin);
    return r;
}

// End of a workgroup with fp8 outputs, its maxima published: `bid` of L.fin_blocks.  Replaces a one-wave kernel behind the
// GEMM (4.3 us of GPU and 3 us of host time).
__device__ __forceinline__ void finish_fp8(const BigLaunch& L, Workspace* ws, uint32_t bid) {
    if (L.fin_blocks == 0) return;   // uniform
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every wave's maximum is in place ...
    __syncthreads();
    if (threadIdx.x >= 64) return;
    uint32_t last = 0;
    if (threadIdx.x == 0) last = draw_ticket(ws, bid, (uint32_t)L.fin_blocks) ? 1u : 0u;   // ... before the ticket is drawn
    if (__builtin_amdgcn_readfirstlane(last) == 0) return;
    finalize_wave(ws, L.fin, kModeDelayed, prefetch_epilogue(L.fin, kModeDelayed));
}

// MI = 8 needs the whole register file of a SIMD for one wave (256 accumulators + fragments).  The
// MI = 4 variant is held to half of it by declaring a launch bound of twice its real workgroup
// size: given more registers than it needs, the compiler keeps its accumulators in a second
// register set and copies them back and forth inside the K loop.
// kFp8Out: every problem of the launch has an fp8 output (a kernel of its own: the other outputs' code stays as
// the register allocator likes it).
// kBT: the B operands are given transposed, as [K, N] row-major bytes (what a caller has when the reduction index is
// the row index of its tensor: W for dgrad, X for wgrad).  A K-tile of such an operand lies in LDS as it lies in
// memory, 128 rows of k with 256 bytes of n each, and the 16 x 128 fragments are gathered with the transposing
// LDS read DS_READ_B64_TR_B8: within 16 lanes, lane 2 u supplies the address of 8 bytes that lanes 0-7 receive one
// byte each of (byte i to lane i, as their byte u), lane 2 u + 1 the same for lanes 8-15.  With lane 2 u on row
// k0 + u, columns c .. c + 7, and lane 2 u + 1 on the same row, columns c + 8 .. c + 15, lane r receives k0 .. k0 + 7
// of column c + r: a quarter of its fragment.  16-byte chunk c of row k is stored at chunk
// c ^ ((k mod 8) | 8 (k / 32 mod 2)), so that the 8 rows one read touches (and the two 16-lane groups that go
// through LDS together) use different banks.
template <int FA, int FB, int MI, bool kFp8Out = false, bool kBT = false>
__global__ __launch_bounds__(MI == 8 ? kBigThreads : 2 * kBigThreads)
void gemm_nt_big_kernel(const BigLaunch L) {
    // whole tiles: 2 stages of 64 KB; half tiles: 3 stages of 48 KB (their K-tiles are half as long)
    constexpr int NS = MI == 8 ? 2 : 3;
    __shared__ __attribute__((aligned(1024))) uint8_t sA[NS][32 * MI * kBK];
    __shared__ __attribute__((aligned(1024))) uint8_t sB[NS][kBigN * kBK];

    // ---- which tile (or half tile) of which problem is this workgroup's ----------------------------
    [[maybe_unused]] unsigned long long st_entry = 0, st_first = 0, st_loop = 0, cy_first = 0, cy_loop = 0;
    NTFP8_STAMP(st_entry);
    int pid = blockIdx.x;
    int half = 0;
    if constexpr (MI == 8) {
        // Workgroups are dealt to the XCDs round robin.  Within each round of `round_size` workgroups (one per
        // CU) an XCD gets a contiguous run of the tile list, so its L2 sees few operand panels; across rounds
        // the list is walked in order, so that the long tiles at its head start together on the whole chip.
        const int round0 = quotient(pid, L.round_size, L.round_magic) * L.round_size;
        const int in_round = min(L.round_size, L.full_blocks - round0);
        const int local = pid - round0;
#ifdef NTFP8_STAMPS
        if (g_plain_tile_order) {
        } else
#endif
        pid = round0 + run_of_xcd(local, in_round);
    } else {
        const int nb = 2 * L.tail_tiles;
        pid = run_of_xcd(pid, nb);
        half = pid & 1;
        pid = L.full_blocks + (pid >> 1);
    }
    const Picked G = pick_problem(L, pid);
    const BigProblem& P = L.p[G.which];
    const uint8_t* __restrict__ A = G.A;
    const uint8_t* __restrict__ B = G.B;
    const int M = G.M, N = G.N, K = G.K;
    const float scale_a = *G.scale_a, scale_b = *G.scale_b;
    pid -= G.tile_begin;
    int pid_m, pid_n;
    tile_in_group(pid, G.tiles_m, G.tiles_n, G.magic, pid_m, pid_n);
    const int n0 = pid_n * kBigN;
    const int m0 = pid_m * 256 + half * 128;
    // this workgroup's place among all of the call
    [[maybe_unused]] const uint32_t bid = MI == 8 ? blockIdx.x : (uint32_t)L.full_blocks + blockIdx.x;
    if (m0 >= M) {   // second half of a bottom-edge tile with nothing in it (uniform for the workgroup)
        if constexpr (kFp8Out) finish_fp8(L, P.fp8.ws, bid);
        return;
    }

    const int t = threadIdx.x;
    const int lane = t & 63;
    // the wave index as a scalar: LDS destinations of the loads (M0) and every other per-wave offset then
    // live in scalar registers
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(A, (uint32_t)((int64_t)M * K));
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(B, (uint32_t)((int64_t)N * K));
    const int KT = (K + kBK - 1) / kBK;   // >= 2 (host)
    // A wave-level load fills 8 tile rows (1 KB of LDS, lane i at byte 16 i); the lane landing on
    // chunk position p of row r fetches global chunk p ^ swz16(r).  For the rows a lane serves
    // (8 (wave + 4 i) + lane / 8) that is the same chunk for every i.
    const int ld_kc = ((lane & 7) ^ (lane >> 3) ^ (wave & 1)) << 4;
    // chunks of the last K-tile at k >= K must read as zero, not as the start of the next row
    const bool tail_dead = (KT - 1) * kBK + ld_kc >= K;
    float alpha = 0.0f;

    constexpr int LA = MI * 2 * 16 / 8 / kBigWaves;  // wave-level loads of the A tile per wave per stage
    constexpr int LB = kBigLB;
    constexpr int NL = LA + LB;                      // loads per wave per K-tile
    const int wm = (wave >> 1) * (MI * 16), wn = (wave & 1) * 128;

    v4f acc[MI][kBigNJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < kBigNJ; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
    auto mma = [&](int i, int j, const v8i b, const v8i a) { acc[i][j] = mfma_16x16x128<FA, FB>(b, a, acc[i][j]); };

    // The K loop.  kAT: the A operand is given as its transpose, a [K, M] tensor (what wgrad has of dY: its reduction
    // index, the token, is the row index).  Its K-tiles lie in LDS as they lie in memory, 128 rows of k with 256 (whole
    // tiles) or 128 (half tiles) bytes of m each, and the 16 x 128 fragments are gathered with the transposing LDS read,
    // exactly as for a transposed B operand.  Operand layout is a property of the problem, decided per workgroup: a
    // launch mixes dgrad (A plain) and wgrad (A transposed) tiles.
    auto kloop = [&](auto at_tag) {
        constexpr bool kAT = decltype(at_tag)::value;
        uint32_t a_off[LA], b_off[LB];
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            if constexpr (kAT && MI == 8) {
                // as the transposed B below: 4 rows of k per wave-level load, 16 chunks of m each
                const int k = (wave + kBigWaves * i) * 4 + (lane >> 4);
                const int chunk = (lane & 15) ^ ((k & 7) | (((k >> 5) & 1) << 3));
                a_off[i] = (uint32_t)k * (uint32_t)M + (uint32_t)(m0 + chunk * 16);
            } else if constexpr (kAT) {
                // half tiles: 128 bytes of m per row of k, 8 rows of k per wave-level load; chunk c of row k is stored
                // at chunk c ^ ((k / 2 mod 4) | 4 (k / 32 mod 2)): the 8 rows one transposing read touches, and the
                // two 16-lane groups that go through LDS together, then use 16 different 16-byte bank groups
                const int k = (wave + kBigWaves * i) * 8 + (lane >> 3);
                const int chunk = (lane & 7) ^ (((k >> 1) & 3) | (((k >> 5) & 1) << 2));
                a_off[i] = (uint32_t)k * (uint32_t)M + (uint32_t)(m0 + chunk * 16);
            } else {
                // rows >= M fall past the descriptor: zeros
                a_off[i] = (uint32_t)(m0 + (wave + kBigWaves * i) * 8 + (lane >> 3)) * (uint32_t)K + ld_kc;
            }
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            if constexpr (kBT) {
                // a wave-level load fills 4 rows of k (lane / 16) with 16 chunks of n (lane % 16) each; rows k >= K fall
                // past the descriptor (zeros); chunks past N wrap into the next row and only reach outputs that are
                // never stored
                const int k = (wave + kBigWaves * i) * 4 + (lane >> 4);
                const int chunk = (lane & 15) ^ ((k & 7) | (((k >> 5) & 1) << 3));
                b_off[i] = (uint32_t)k * (uint32_t)N + (uint32_t)(n0 + chunk * 16);
            } else {
                b_off[i] = (uint32_t)(n0 + (wave + kBigWaves * i) * 8 + (lane >> 3)) * (uint32_t)K + ld_kc;
            }
        }
        // byte distance between K-tiles in memory
        const int a_step = kAT ? kBK * M : kBK, b_step = kBT ? kBK * N : kBK;

        // load number `l` (0 .. NL-1, A loads first) of K-tile `ktile` straight into its LDS stage, ktile mod NS
        auto issue = [&](int ktile, int l) {
            const int s = ktile % NS;
            if (l < LA)
                lds_load16(ra, (lds_ptr)(uintptr_t)&sA[s][(wave + kBigWaves * l) * 1024], a_off[l], ktile * a_step);
            else
                lds_load16(rb, (lds_ptr)(uintptr_t)&sB[s][(wave + kBigWaves * (l - LA)) * 1024], b_off[l - LA], ktile * b_step);
        };
        // Called once, before the first load of the last K-tile is queued (no other tile is loaded after it):
        // lanes whose chunk lies at k >= K get an offset past the descriptor and so read zeros.
        auto poison_tail = [&]() {
            if (tail_dead) {
                if constexpr (!kAT) {   // (rows k >= K of a transposed operand fall past its descriptor by themselves)
#pragma unroll
                    for (int i = 0; i < LA; ++i) a_off[i] = 0xfffffff0u;
                }
                if constexpr (!kBT) {
#pragma unroll
                    for (int i = 0; i < LB; ++i) b_off[i] = 0xfffffff0u;
                }
            }
        };

        // fragment reads: lane -> row (lane % 16) of a 16-row block, two 16-byte chunks 2 (lane / 16) + {0, 1};
        // block i of the wave is 16 i rows = 2048 i bytes further on (the swizzle only looks at row bits 0-3)
        const int frow = lane & 15;
        const int fk = (lane >> 4) * 2;
        const int a_rd0 = lds_off16(wm + frow, fk), a_rd1 = lds_off16(wm + frow, fk + 1);
        const int b_rd0 = lds_off16(wn + frow, fk), b_rd1 = lds_off16(wn + frow, fk + 1);
        // transposed operands: lane u of a 16-lane group (which serves k 32 (lane / 16) .. + 31) addresses row k0 + u / 2,
        // half u % 2 of the block's 16-byte chunk; quarter t of the fragment is k0 = 32 (lane / 16) + 8 t
        const int bt_row = (lane & 15) >> 1;
        const int bt_base = ((lane >> 4) * 32 + bt_row) * 256 + ((((wave & 1) ^ ((lane >> 4) & 1))) << 7) + (lane & 1) * 8;
        const int bt_x = bt_row << 4;
        // the same for A: the wave's blocks are chunks 8 (wave / 2) + i of a 256-byte row (whole tiles), chunks
        // 4 (wave / 2) + i of a 128-byte row (half tiles, swizzle (k / 2 mod 4) | 4 (k / 32 mod 2))
        const int at_base = MI == 8 ? ((lane >> 4) * 32 + bt_row) * 256 + ((((wave >> 1) ^ ((lane >> 4) & 1))) << 7) + (lane & 1) * 8
                                    : ((lane >> 4) * 32 + bt_row) * 128 + ((((wave >> 1) ^ ((lane >> 4) & 1))) << 6) + (lane & 1) * 8;
        const int at_x = MI == 8 ? bt_row << 4 : ((bt_row >> 1) & 3) << 4;
        constexpr int at_pitch = MI == 8 ? 256 : 128;
        // half h (0 / 1) of a fragment = one 128-bit LDS read, or two transposing 64-bit reads
        auto rd_a = [&](int s, int i, int h) -> v4i {
            if constexpr (kAT) {
                typedef int v2i __attribute__((ext_vector_type(2)));
                typedef __attribute__((address_space(3))) v2i* tr_ptr;
                int x = at_x;
                if constexpr (MI == 4) asm volatile("" : "+v"(x));
                uint8_t* p = &sA[s][at_base + ((i << 4) ^ x) + h * (2 * 8 * at_pitch)];
                const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)p);
                const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)(p + 8 * at_pitch));
                return (v4i){lo.x, lo.y, hi.x, hi.y};
            } else {
                return *reinterpret_cast<const v4i*>(&sA[s][(h ? a_rd1 : a_rd0) + i * 2048]);
            }
        };
        auto rd_b = [&](int s, int j, int h) -> v4i {
            if constexpr (kBT) {
                typedef int v2i __attribute__((ext_vector_type(2)));
                typedef __attribute__((address_space(3))) v2i* tr_ptr;
                // (address-space cast, not a round trip through an integer: the compiler must see that these reads
                // come from sB, or it waits for every direct-to-LDS load in flight before each of them)
                int x = bt_x;
                // half tiles: recomputed at every use, eight block offsets kept across the K loop do not fit their
                // register budget; whole tiles keep them (1 % faster than recomputing)
                if constexpr (MI == 4) asm volatile("" : "+v"(x));
                uint8_t* p = &sB[s][bt_base + ((j << 4) ^ x) + h * (2 * 8 * 256)];
                const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)p);
                const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)(p + 8 * 256));
                return (v4i){lo.x, lo.y, hi.x, hi.y};
            } else {
                return *reinterpret_cast<const v4i*>(&sB[s][(h ? b_rd1 : b_rd0) + j * 2048]);
            }
        };
        auto frag = [](const v4i (&x)[2]) -> v8i { return (v8i){x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w}; };

        v4i fa[MI][2];

        // A K-tile kt lives in LDS stage kt mod NS and is computed in two parts, front(kt) = MFMA groups 0-5 and back(kt) =
        // groups 6-7.  The K loop runs back(kt); front(kt + 1), so that its back edge sits right behind the barrier at
        // the end of front(), where no LDS read is outstanding.
        //
        // An MFMA occupies the matrix pipe for 32 cycles and the wave issues in order, so whatever stands between
        // two MFMAs must issue within that time or the pipe idles.  The code below therefore puts at most one
        // memory instruction (two LDS reads at most) behind each MFMA, and a scheduling fence behind each such
        // pair keeps the compiler from regrouping them.
        using Yes = std::true_type;
        using No = std::false_type;

        if constexpr (MI == 8) {
            // ---- whole tiles ---------------------------------------------------------------------------
            // Two stages.  front(f), MFMA groups 0-5 of tile f, in slots of one MFMA each (8 per group): the B
            // fragments 2-7 are read behind every other one of the first 24, a barrier then releases the stage, and the
            // loads of tile f + 2 go into it, one behind every third MFMA up to the end of back(f): spread out, because
            // sixteen in a row cost more than they gain (us, 4096 x 4096 x 4096 and x 14336: behind every MFMA 51.3 and
            // 184, every second 48.8 and 162, every third 48.5 and 160, every fourth 49.5 and 165; through registers,
            // deposited in LDS a K-tile later, 50.6 and 165).  The barrier at the end of front(f) publishes tile f + 1,
            // whose loads have had at least 48 MFMAs of time.
            constexpr int kRelease = 25;              // slot of the first barrier
            constexpr int kEvery = 3;                 // slots from load to load
            constexpr int kFront = (MI * 6 - 1 - kRelease) / kEvery;   // loads in front(), the others in back()
            constexpr int kReads = 4 * (kBigNJ - 2);  // B fragments 2-7 are read behind every other of so many slots
            static_assert(kRelease > kReads - 2 && kRelease < MI * 6, "the stage is released behind the last read of it, within front()");
            static_assert(kFront > 0 && kFront <= NL, "front() requests the first loads of a tile, back() the others");
            v4i fw[kBigNJ][2];   // all B fragments of a tile
            auto front_w = [&](auto l_tag, auto b_tag, int f) {
                constexpr bool L = decltype(l_tag)::value, B = decltype(b_tag)::value;   // L: there is a tile f + 2; B: f + 1
                const int s = f & 1;
                sched_fence();
#pragma unroll
                for (int x = 0; x < MI * 6; ++x) {
                    const int j = x / MI, i = x % MI;
                    mma(i, j, frag(fw[j]), frag(fa[i]));
                    if (x < kReads && x % 2 == 0) fw[2 + x / 4][x / 2 % 2] = rd_b(s, 2 + x / 4, x / 2 % 2);
                    if constexpr (L) {
                        if (x == kRelease) {
                            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // every fragment of tile f is in registers
                            wg_barrier();
                        }
                        if (x > kRelease && (x - kRelease) % kEvery == 0) issue(f + 2, (x - kRelease) / kEvery - 1);
                    }
                    sched_fence();
                }
                if constexpr (B) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L ? kFront : 0) : "memory");   // all but tile f + 2's
                    wg_barrier();
                }
            };
            // groups 6 and 7, interleaved per A fragment, which is dead after them and refilled from tile f + 1
            auto back_w = [&](auto l_tag, auto prefetch_tag, int f) {
                constexpr bool L = decltype(l_tag)::value, prefetch = decltype(prefetch_tag)::value;
                const int s1 = (f + 1) & 1;
                sched_fence();
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    mma(i, 6, frag(fw[6]), frag(fa[i]));
                    if (prefetch && i > 0) {
                        fa[i - 1][0] = rd_a(s1, i - 1, 0);
                        fa[i - 1][1] = rd_a(s1, i - 1, 1);
                    }
                    sched_fence();
                    mma(i, 7, frag(fw[7]), frag(fa[i]));
                    if (prefetch && i < 4) fw[i >> 1][i & 1] = rd_b(s1, i >> 1, i & 1);
                    if constexpr (L) {
#pragma unroll
                        for (int l = kFront + i * (NL - kFront) / MI; l < kFront + (i + 1) * (NL - kFront) / MI; ++l) issue(f + 2, l);
                    }
                    sched_fence();
                }
                if constexpr (prefetch) {
                    fa[MI - 1][0] = rd_a(s1, MI - 1, 0);
                    fa[MI - 1][1] = rd_a(s1, MI - 1, 1);
                }
                sched_fence();
            };
            // prologue: tiles 0 and 1
#pragma unroll
            for (int l = 0; l < NL; ++l) issue(0, l);
            if (KT == 2) poison_tail();
#pragma unroll
            for (int l = 0; l < NL; ++l) issue(1, l);
            // (behind the first requests: the scales were written by the kernel before, a trip of their own to memory)
            alpha = descale_factor(scale_a, scale_b, P.ex.scale_inv);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");   // tile 0 has landed, tile 1 may still be in flight
            wg_barrier();
            NTFP8_STAMP(st_first);
            NTFP8_CYCLES(cy_first);
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                fa[i][0] = rd_a(0, i, 0);
                fa[i][1] = rd_a(0, i, 1);
            }
#pragma unroll
            for (int h = 0; h < 4; ++h) fw[h >> 1][h & 1] = rd_b(0, h >> 1, h & 1);

            // (poison_tail() runs between the loads of tile KT - 2 and those of tile KT - 1 = f + 2)
            if (KT == 3) poison_tail();
            if (KT > 2) front_w(Yes{}, Yes{}, 0);
            else front_w(No{}, Yes{}, 0);
            int f = 1;
            for (; f + 3 < KT; ++f) {
                back_w(Yes{}, Yes{}, f - 1);
                front_w(Yes{}, Yes{}, f);
            }
            if (f + 2 < KT) {   // f = KT - 3 >= 1
                back_w(Yes{}, Yes{}, f - 1);
                poison_tail();
                front_w(Yes{}, Yes{}, f);
                ++f;
            }
            if (f + 1 < KT) {   // f = KT - 2 >= 1: back(f - 1) sends the rest of the last tile
                back_w(Yes{}, Yes{}, f - 1);
                front_w(No{}, Yes{}, f);
                ++f;
            }
            back_w(No{}, Yes{}, f - 1);   // f = KT - 1
            front_w(No{}, No{}, f);
            back_w(No{}, No{}, f);
        } else {
        // ---- half tiles ------------------------------------------------------------------------------
        //   front(kt): entered with fa[] = the tile's A fragments and fb[0], fb[1] = its first two B fragments; reads B
        //              fragments 2..7 three groups ahead of their use; ends with the barrier that publishes tile kt + 1 and
        //              releases the stage of tile kt.
        //   back(kt):  refills fa[] / fb[0], fb[1] from tile kt + 1.
        // The stage released by the barrier of tile kt is refilled with tile kt + NS between that barrier and the next, the
        // loads spread over back(kt) and front(kt + 1): twelve of them within 16 MFMAs, and fragment 7 read behind the last group
        // but one, cost 3 % (us, 4096 x 2048 x 4096 in 256 half tiles 29.4 / 28.4; backward of 4096 tokens, 1024 -> 4096,
        // 36.9 / 35.8).
        v4i fb[4][2];
        constexpr int kBackLoads = NL / 3;
        constexpr int kFrontLoads = NL - kBackLoads;
        static_assert(kBackLoads > 0 && kFrontLoads > 0, "every load of a tile is requested once, in back() or in front()");
        // loads: queue the rest of tile kt + NS - 1; WAIT (>= 0): barrier, after all but the newest WAIT
        // loads of this wave have landed (-1: no barrier)
        auto front = [&](auto loads_tag, auto wait_tag, int kt) {
            constexpr bool loads = decltype(loads_tag)::value;
            constexpr int WAIT = decltype(wait_tag)::value;
            const int s = kt % NS;
            sched_fence();
#pragma unroll
            for (int j = 0; j < 6; ++j) {
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    mma(i, j, frag(fb[j & 3]), frag(fa[i]));
                    // B fragment j + 3 (behind group 0 fragments 2 and 3), so that none is on its way at the barrier
                    if (i < 2 && j < 5) fb[(j + (j ? 3 : 2)) & 3][i] = rd_b(s, j + (j ? 3 : 2), i);
                    else if (j == 0) fb[3][i - 2] = rd_b(s, 3, i - 2);
                    if (loads && j > 0 && i >= 2) {   // slot x of n
                        constexpr int n = 5 * (MI - 2);
                        const int x = (j - 1) * (MI - 2) + i - 2;
#pragma unroll
                        for (int l = kBackLoads + x * kFrontLoads / n; l < kBackLoads + (x + 1) * kFrontLoads / n; ++l) issue(kt + NS - 1, l);
                    }
                    sched_fence();
                }
            }
            if constexpr (WAIT >= 0) {
                // Every fragment of tile kt is in registers (or in flight): after the barrier its stage may be
                // overwritten, and tile kt + 1 is complete in the next stage.
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT) : "memory");
                wg_barrier();
            }
        };
        auto back = [&](auto loads_tag, auto prefetch_tag, int kt) {
            constexpr bool loads = decltype(loads_tag)::value, prefetch = decltype(prefetch_tag)::value;
            const int s1 = (kt + 1) % NS;
            sched_fence();
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                // fa[i] is dead after its two MFMAs; it is refilled with the fragment of the next tile one step later
                mma(i, kBigNJ - 2, frag(fb[(kBigNJ - 2) & 3]), frag(fa[i]));
                if (prefetch && i > 0) {
                    fa[i - 1][0] = rd_a(s1, i - 1, 0);
                    fa[i - 1][1] = rd_a(s1, i - 1, 1);
                }
                sched_fence();
                mma(i, kBigNJ - 1, frag(fb[(kBigNJ - 1) & 3]), frag(fa[i]));
                if constexpr (loads) {   // loads [i kBackLoads / MI, (i + 1) kBackLoads / MI) ride on this step
#pragma unroll
                    for (int l = i * kBackLoads / MI; l < (i + 1) * kBackLoads / MI; ++l) issue(kt + NS, l);
                }
                if (prefetch && i < 4) fb[i >> 1][i & 1] = rd_b(s1, i >> 1, i & 1);
                sched_fence();
            }
            if constexpr (prefetch) {
                fa[MI - 1][0] = rd_a(s1, MI - 1, 0);
                fa[MI - 1][1] = rd_a(s1, MI - 1, 1);
            }
            sched_fence();
        };
        // Three stages: the loads of tile t are queued while tile t - 3's stage is the one just released, i.e.
        // two K-tiles before tile t is published.  A half-tile K-tile is only 32 MFMAs (about 0.55 us): with
        // two stages the loads had half a K-tile to arrive, less than an L2 hit takes.
        using Wait = std::integral_constant<int, NL>;   // the NL loads of the newest tile may still be in flight
        using WaitAll = std::integral_constant<int, 0>;
        using NoBarrier = std::integral_constant<int, -1>;
        // prologue: tiles 0, 1 and (if there is one) 2
#pragma unroll
        for (int l = 0; l < NL; ++l) issue(0, l);
        if (KT == 2) poison_tail();
#pragma unroll
        for (int l = 0; l < NL; ++l) issue(1, l);
        if (KT > 2) {
            if (KT == 3) poison_tail();
#pragma unroll
            for (int l = 0; l < NL; ++l) issue(2, l);
        }
        alpha = descale_factor(scale_a, scale_b, P.ex.scale_inv);   // (as for whole tiles)
        if (KT > 2) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NL) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");
        }
        wg_barrier();
        NTFP8_STAMP(st_first);
        NTFP8_CYCLES(cy_first);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            fa[i][0] = rd_a(0, i, 0);
            fa[i][1] = rd_a(0, i, 1);
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) fb[h >> 1][h & 1] = rd_b(0, h >> 1, h & 1);

        // front(0) queues nothing (tile 3 goes into the stage that front(0) itself still reads)
        if (KT > 2) front(No{}, Wait{}, 0);
        else front(No{}, WaitAll{}, 0);
        int f = 1;
        for (; f + 2 < KT; ++f) {   // tile f + 2 is loaded during back(f - 1); front(f)
            if (f + 3 == KT) poison_tail();
            back(Yes{}, Yes{}, f - 1);
            front(Yes{}, Wait{}, f);
        }
        if (f + 1 < KT) {   // f = KT - 2 >= 1: nothing left to load
            back(No{}, Yes{}, f - 1);
            front(No{}, WaitAll{}, f);
            ++f;
        }
        back(No{}, Yes{}, f - 1);   // f = KT - 1
        front(No{}, NoBarrier{}, f);
        back(No{}, No{}, f);
        }
    };
    if constexpr (kBT) {
        if (G.at) kloop(std::true_type{});   // uniform for the workgroup
        else kloop(std::false_type{});
    } else {
        kloop(std::false_type{});
    }

    NTFP8_STAMP(st_loop);
    NTFP8_CYCLES(cy_loop);
    {
        void* const Dv = P.D;
        // output type, accumulation and bias are properties of the problem, not of the kernel (fp8 outputs apart)
        auto epilogue = [&](auto bias_tag, const float (*bv)[4]) {
            constexpr bool kBias = decltype(bias_tag)::value;
            if constexpr (kFp8Out) {
                const float scale_d = *P.fp8.scale;
                const bool slow = scale_is_degenerate(scale_d);
                const uint32_t amax =
                    P.d_dtype == NTFP8_OUT_E4M3
                        ? store_wave_tile16_fp8<kE4M3, MI, kBigNJ, kBias>(acc, static_cast<uint8_t*>(Dv), P.fp8.Dt, alpha, scale_d, slow, M,
                                                                     N, m0 + wm, n0 + wn, lane, bv)
                        : store_wave_tile16_fp8<kE5M2, MI, kBigNJ, kBias>(acc, static_cast<uint8_t*>(Dv), P.fp8.Dt, alpha, scale_d, slow, M,
                                                                     N, m0 + wm, n0 + wn, lane, bv);
                publish_amax(amax, P.fp8.ws);
                finish_fp8(L, P.fp8.ws, bid);
            } else if (P.d_dtype == NTFP8_BF16) {
                store_wave_tile16<NTFP8_BF16, false, MI, kBigNJ, kBias>(acc, Dv, alpha, M, N, m0 + wm, n0 + wn, lane, bv);
            } else if (P.d_dtype == NTFP8_F16) {
                store_wave_tile16<NTFP8_F16, false, MI, kBigNJ, kBias>(acc, Dv, alpha, M, N, m0 + wm, n0 + wn, lane, bv);
            } else if (P.accumulate) {
                store_wave_tile16<NTFP8_F32, true, MI, kBigNJ, kBias>(acc, Dv, alpha, M, N, m0 + wm, n0 + wn, lane, bv);
            } else {
                store_wave_tile16<NTFP8_F32, false, MI, kBigNJ, kBias>(acc, Dv, alpha, M, N, m0 + wm, n0 + wn, lane, bv);
            }
        };
        // (no bias together with a transposed B operand: the backward GEMMs that read one have none, and their
        // instantiation has no registers to spare for the second set of epilogues)
        bool with_bias = false;
        if constexpr (!kBT) with_bias = P.ex.bias != nullptr;   // uniform
        if (with_bias) {
            float bv[kBigNJ][4];
            load_bias16<kBigNJ>(bv, P.ex.bias, P.ex.bias_dtype, N, n0 + wn, lane);
            epilogue(std::true_type{}, bv);
        } else {
            epilogue(std::false_type{}, nullptr);
        }
    }
#ifdef NTFP8_STAMPS
    {
        const unsigned long long st_issued = wall_clock64();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const unsigned long long st_drained = wall_clock64();
        if (threadIdx.x == 0) {
            unsigned long long* o = g_stamps + (size_t)(blockIdx.x % kStampSlots) * 8;
            o[0] = st_entry, o[1] = st_first, o[2] = st_loop, o[3] = st_issued, o[4] = st_drained;
            // HW_ID (cu 11:8, sh 12, se 15:13) | XCC_ID << 32 | MI << 40
            o[5] = (unsigned long long)__builtin_amdgcn_s_getreg((31 << 11) | 4) |
                   ((unsigned long long)(__builtin_amdgcn_s_getreg((31 << 11) | 20) & 0xf) << 32) | ((unsigned long long)MI << 40);
            o[6] = cy_first, o[7] = cy_loop;
        }
    }
#endif
}

}  // namespace ntfp8
