// FP8 GEMM in 128 x 128, 128 x 64 and 64 x 64 tiles (gfx950): the shapes whose 256-wide tiles would leave CUs idle.
// Included by gemm_mid.hip.
//
// Four waves of a TM x TN tile: 2 x 2 waves of 64 x 64 (128 x 128), or four of TM / 4 x 64 below each other (TN = 64), as
// MI x 4 accumulator blocks of V_MFMA_F32_16X16X128_F8F6F4, k ascending: the same instruction in the same order as the
// 256-wide kernel, hence the same results bit for bit.
//
// Pipeline: four LDS stages of a K-tile (32, 24 or 16 KB) filled straight from memory (buffer_load ... lds), one barrier
// per K-tile.  Between barriers kt and kt + 1 a wave reads all fragments of tile kt + 1 into a second set of registers
// while its MFMAs work on the set of tile kt, and requests tile kt + 4 into the stage that barrier kt has released:
// every load has three K-tiles of time to arrive and every LDS read one.  Tiles past the end are requested like
// any other, with offsets past the descriptor (no traffic, zeros), so that the number of loads in flight is the same
// in every trip.
//
// Bound by LDS: reads and deposits of a K-tile at 128 bytes a cycle are 768 (128 x 128), 576 (128 x 64) and 448 cycles, the MFMAs
// 512, 256 and 128.  A K-tile takes 390, 290 and 185 ns (350 for two workgroups of 64 x 64 on a CU), so that 128 x 64 tiles are
// the fastest way where they are one round of workgroups: 2048 x 1024 x 4096 in 64 x 64 / 128 x 128 / 128 x 64 tiles 15.2 / 15.6 /
// 12.9 us.  (A wave's own rows of A straight into registers, 16 rows of 64 bytes a load: 21.2 and 19.5 us in 64 x 64 and 128 x 64.)
//
// Operand layouts are run-time properties of a problem, as in the 256-wide kernel: K-contiguous, B given as [K, N], or A
// given as [K, M] next to such a B; a transposed operand is staged as it lies in memory, 128 rows of k with TM or TN bytes each,
// and gathered with DS_READ_B64_TR_B8 (gemm_big.h describes the instruction).
#pragma once

namespace ntfp8 {

template <int FA, int FB, int TM, int TN, bool kFp8Out>
__global__ __launch_bounds__(kBigThreads, TM == 64 ? 2 : 1) void gemm_mid_kernel(const BigLaunch L) {
    constexpr int WN = TN / 64, WM = kBigWaves / WN;   // waves along N, along M
    constexpr int MI = TM / 16 / WM, NJ = 4, NS = 4;
    constexpr int kLoadsA = TM / 32, kLoadsB = TN / 32;   // wave-level 1 KB loads of an operand's K-tile per wave
    constexpr int kLoads = kLoadsA + kLoadsB;
    __shared__ __attribute__((aligned(1024))) uint8_t sA[NS][TM * kBK];
    __shared__ __attribute__((aligned(1024))) uint8_t sB[NS][TN * kBK];

    // within a round of workgroups an XCD works on a contiguous run of the tile list (workgroups are dealt round robin)
    int pid;
    {
        const int round0 = quotient((int)blockIdx.x, L.round_size, L.round_magic) * L.round_size, local = blockIdx.x - round0;
        const int in_round = min(L.round_size, (int)gridDim.x - round0);
        pid = round0 + run_of_xcd(local, in_round);
    }
    // (uniform) the tail of a launch of 256-wide tiles: parts of the tiles from full_blocks on
    const bool tail = L.tail_tiles != 0;
    constexpr int kAcross = 256 / TN, kParts = 256 / TM * kAcross;
    const int part = tail ? pid % kParts : 0;
    if (tail) pid = L.full_blocks + pid / kParts;
    const Picked G = pick_problem(L, pid);
    const BigProblem& P = L.p[G.which];
    const int M = G.M, N = G.N, K = G.K;
    const float scale_a = *G.scale_a, scale_b = *G.scale_b;
    pid -= G.tile_begin;
    int pid_m, pid_n;
    tile_in_group(pid, G.tiles_m, G.tiles_n, G.magic, pid_m, pid_n);
    const int m0 = pid_m * (tail ? 256 : TM) + part / kAcross * TM, n0 = pid_n * (tail ? 256 : TN) + part % kAcross * TN;
    if (m0 >= M || n0 >= N) return;   // a part of an edge tile with nothing in it (no bookkeeping inside such launches)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN * (16 * MI), wn = wave % WN * 64;
    const int KT = (K + kBK - 1) / kBK;
    float alpha = 0.0f;

    v4f acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

    auto kloop = [&](auto at_tag, auto bt_tag) {
        constexpr bool kAT = decltype(at_tag)::value, kBT = decltype(bt_tag)::value;
        // A K-contiguous operand is addressed from its tile's first row (any tensor size); rows past the end fall
        // behind the descriptor and read as zeros.  A transposed one is addressed from its first element (< 2 GiB): rows
        // k >= K fall behind the descriptor, columns past the end wrap into the next row and reach no stored output.
        const __amdgpu_buffer_rsrc_t ra = kAT ? make_rsrc(G.A, (uint32_t)((int64_t)M * K))
                                              : make_rsrc(G.A + (int64_t)m0 * K, (uint32_t)(min(M - m0, TM) * (int64_t)K));
        const __amdgpu_buffer_rsrc_t rb = kBT ? make_rsrc(G.B, (uint32_t)((int64_t)N * K))
                                              : make_rsrc(G.B + (int64_t)n0 * K, (uint32_t)(min(N - n0, TN) * (int64_t)K));
        constexpr uint32_t kNowhere = 0xfffffff0u;
        // offset of this lane's 16 bytes of load i of K-tile 0; position p of row r receives chunk p ^ swizzle(r)
        const int ld_kc = ((lane & 7) ^ (lane >> 3) ^ (wave & 1)) << 4;   // K-contiguous: 8 rows per load, swz16
        typedef std::integral_constant<int, TM> WideA;
        typedef std::integral_constant<int, TN> WideB;
        auto offset = [&](auto width_tag, bool transposed, int i, int first, int extent) -> uint32_t {
            constexpr int T = decltype(width_tag)::value;
            const int w = wave + kBigWaves * i;
            if (!transposed) return (uint32_t)(w * 8 + (lane >> 3)) * (uint32_t)K + ld_kc;
            if constexpr (T == 128) {
                const int k = w * 8 + (lane >> 3);
                return (uint32_t)k * (uint32_t)extent + (uint32_t)(first + (((lane & 7) ^ (((k >> 1) & 3) | (((k >> 5) & 1) << 2))) << 4));
            } else {
                const int k = w * 16 + (lane >> 2);
                return (uint32_t)k * (uint32_t)extent + (uint32_t)(first + (((lane & 3) ^ (((k >> 2) & 1) | (((k >> 5) & 1) << 1))) << 4));
            }
        };
        uint32_t a_off[kLoadsA], b_off[kLoadsB];
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) a_off[i] = offset(WideA{}, kAT, i, m0, M);
#pragma unroll
        for (int i = 0; i < kLoadsB; ++i) b_off[i] = offset(WideB{}, kBT, i, n0, N);
        const int a_step = kAT ? kBK * M : kBK, b_step = kBT ? kBK * N : kBK;
        const bool tail_dead = (KT - 1) * kBK + ld_kc >= K;
        // request of K-tile kt in pieces: piece l (A's loads first) after prepare(kt)
        int rq_s = 0, rq_a = 0, rq_b = 0;
        auto prepare = [&](int kt) {
            // (uniform) chunks at k >= K must not read into the next row: the last tile's, then whole tiles
            if (kt >= KT - 1) {
#pragma unroll
                for (int i = 0; i < kLoadsA; ++i)
                    if (kt >= KT || (!kAT && tail_dead)) a_off[i] = kNowhere;
#pragma unroll
                for (int i = 0; i < kLoadsB; ++i)
                    if (kt >= KT || (!kBT && tail_dead)) b_off[i] = kNowhere;
            }
            rq_s = kt % NS;
            rq_a = kt < KT ? kt * a_step : 0, rq_b = kt < KT ? kt * b_step : 0;
        };
        auto request = [&](int l) {
            if (l < kLoadsA) lds_load16(ra, (lds_ptr)(uintptr_t)&sA[rq_s][(wave + kBigWaves * l) * 1024], a_off[l], rq_a);
            else lds_load16(rb, (lds_ptr)(uintptr_t)&sB[rq_s][(wave + kBigWaves * (l - kLoadsA)) * 1024], b_off[l - kLoadsA], rq_b);
        };

        // fragments: lane -> row lane % 16 of a 16-row block, k 32 (lane / 16) .. + 31
        const int frow = lane & 15, fk = (lane >> 4) * 2;
        const int rd0 = lds_off16(frow, fk), rd1 = lds_off16(frow, fk + 1);   // + 2048 bytes per block of 16 rows
        const int tr_row = (lane & 15) >> 1;
        // (out here for both widths: computed inside half(), the compiler no longer tells the transposing reads from the loads in
        // flight and waits for all of those)
        const int base128 = ((lane >> 4) * 32 + tr_row) * 128 + (lane & 1) * 8, base64 = ((lane >> 4) * 32 + tr_row) * 64 + (lane & 1) * 8;
        const int x128 = ((tr_row >> 1) & 3) | (((lane >> 4) & 1) << 2), x64 = ((tr_row >> 2) & 1) | (((lane >> 4) & 1) << 1);
        typedef int v2i __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) v2i* tr_ptr;
        // half h of the fragment of rows / columns first + 16 blk .. + 15
        auto half = [&](auto t_tag, auto width_tag, uint8_t* stage, int first, int blk, int h) -> v4i {
            if constexpr (decltype(t_tag)::value) {
                constexpr int T = decltype(width_tag)::value;
                constexpr bool kWide = T == 128;
                uint8_t* p = stage + (kWide ? base128 : base64) + (((first / 16 + blk) ^ (kWide ? x128 : x64)) << 4) + h * (16 * T);
                const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)p);
                const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((tr_ptr)(p + 8 * T));
                return (v4i){lo.x, lo.y, hi.x, hi.y};
            } else {
                return *reinterpret_cast<const v4i*>(stage + (h ? rd1 : rd0) + first * kBK + blk * 2048);
            }
        };
        struct Frags {
            v4i a[MI][2], b[NJ][2];
        };
        constexpr int kHalves = 2 * (MI + NJ), kMfmas = MI * NJ;
        auto read = [&](int s, Frags& f, int x) {   // x-th half of the fragments in stage s: b0, a0, a1, .., b1, b2, ..
            const int q = x >> 1, h = x & 1;
            if (q == 0) f.b[0][h] = half(bt_tag, WideB{}, sB[s], wn, 0, h);
            else if (q <= MI) f.a[q - 1][h] = half(at_tag, WideA{}, sA[s], wm, q - 1, h);
            else f.b[q - MI][h] = half(bt_tag, WideB{}, sB[s], wn, q - MI, h);
        };
        auto frag = [](const v4i (&x)[2]) -> v8i { return (v8i){x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w}; };
        // The MFMAs of one K-tile on fragments `f`.  A wave issues in order, so the LDS reads of the next tile (into `g`)
        // and the requests of the tile after the ones in flight stand between them, one or two behind each MFMA; a
        // fence behind each such group keeps the compiler from gathering the reads in front.
        auto multiply = [&](auto more_tag, const Frags& f, Frags& g, int next) {
            constexpr bool kMore = decltype(more_tag)::value;
            const int s = next % NS;
            sched_fence();
#pragma unroll
            for (int x = 0; x < kMfmas; ++x) {
                const int j = x / MI, i = x % MI;
                acc[i][j] = mfma_16x16x128<FA, FB>(frag(f.b[j]), frag(f.a[i]), acc[i][j]);
                if constexpr (kMore) {
#pragma unroll
                    for (int y = x * kHalves / kMfmas; y < (x + 1) * kHalves / kMfmas; ++y) read(s, g, y);
#pragma unroll
                    for (int l = x * kLoads / kMfmas; l < (x + 1) * kLoads / kMfmas; ++l) request(l);
                    sched_fence();
                }
            }
        };
        // barrier kt: this wave's fragments of tile kt are in registers and its part of tile kt + 1 has landed
        auto arrive = [&]() {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kLoads) : "memory");
            wg_barrier();
        };

        using Yes = std::true_type;
        using No = std::false_type;
        Frags f0, f1;
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            prepare(t);
#pragma unroll
            for (int l = 0; l < kLoads; ++l) request(l);
        }
        // (behind the first requests: the scales were written by the kernel before, a trip of their own to memory)
        alpha = descale_factor(scale_a, scale_b, P.ex.scale_inv);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * kLoads) : "memory");
        wg_barrier();
#pragma unroll
        for (int x = 0; x < kHalves; ++x) read(0, f0, x);
        int kt = 0;
        for (; kt + 2 <= KT - 1; kt += 2) {
            prepare(kt + NS);
            arrive();
            multiply(Yes{}, f0, f1, kt + 1);
            prepare(kt + 1 + NS);
            arrive();
            multiply(Yes{}, f1, f0, kt + 2);
        }
        if (kt + 1 <= KT - 1) {   // one more tile to read: the last
            prepare(kt + NS);
            arrive();
            multiply(Yes{}, f0, f1, kt + 1);
            multiply(No{}, f1, f0, 0);
        } else {
            multiply(No{}, f0, f1, 0);
        }
        // (loads still in flight write zeros into stages nobody reads again; they are waited for before the wave ends)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    if (G.at) kloop(std::true_type{}, std::true_type{});   // uniform for the workgroup
    else if (G.bt) kloop(std::false_type{}, std::true_type{});
    else kloop(std::false_type{}, std::false_type{});

    auto epilogue = [&](auto bias_tag, const float (*bv)[4]) {
        constexpr bool kBias = decltype(bias_tag)::value;
        const int mb = m0 + wm, nb = n0 + wn;
        if constexpr (kFp8Out) {
            const float scale_d = *P.fp8.scale;
            const bool slow = scale_is_degenerate(scale_d);
            uint8_t* D = static_cast<uint8_t*>(P.D);
            const uint32_t amax = P.d_dtype == NTFP8_OUT_E4M3
                                      ? store_wave_tile16_fp8<kE4M3, MI, NJ, kBias>(acc, D, P.fp8.Dt, alpha, scale_d, slow, M, N, mb, nb, lane, bv)
                                      : store_wave_tile16_fp8<kE5M2, MI, NJ, kBias>(acc, D, P.fp8.Dt, alpha, scale_d, slow, M, N, mb, nb, lane, bv);
            publish_amax(amax, P.fp8.ws);
            finish_fp8(L, P.fp8.ws, blockIdx.x);
        } else if (P.d_dtype == NTFP8_BF16) {
            store_wave_tile16<NTFP8_BF16, false, MI, NJ, kBias>(acc, P.D, alpha, M, N, mb, nb, lane, bv);
        } else if (P.d_dtype == NTFP8_F16) {
            store_wave_tile16<NTFP8_F16, false, MI, NJ, kBias>(acc, P.D, alpha, M, N, mb, nb, lane, bv);
        } else if (P.accumulate) {
            store_wave_tile16<NTFP8_F32, true, MI, NJ, kBias>(acc, P.D, alpha, M, N, mb, nb, lane, bv);
        } else {
            store_wave_tile16<NTFP8_F32, false, MI, NJ, kBias>(acc, P.D, alpha, M, N, mb, nb, lane, bv);
        }
    };
    if (P.ex.bias) {   // uniform
        float bv[NJ][4];
        load_bias16<NJ>(bv, P.ex.bias, P.ex.bias_dtype, N, n0 + wn, lane);
        epilogue(std::true_type{}, bv);
    } else {
        epilogue(std::false_type{}, nullptr);
    }
}

}  // namespace ntfp8
