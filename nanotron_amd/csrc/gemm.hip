// FP8 GEMM for gfx950:  D[M,N] (+)= (A[M,K] . B[N,K]^T) * (1/scale_a)(1/scale_b)
//
// Both operands are contiguous along K (the only form the reference issues); the big kernel also takes B as
// its transpose, a [K, N] tensor.  fp32 accumulation on the matrix cores (e4m3 / e5m2 selectable per
// operand), operand tiles staged in XOR-swizzled LDS, descale + one rounding in the epilogue to fp32
// (optionally added to what is there), bf16, fp16 or fp8 bytes.
//
// Kernels:
//   gemm_nt_big_kernel    (gemm_big.h) 256 x 256 x 128 tiles, 4 waves of 128 x 128 with 16x16x128 MFMAs,
//                         loads straight into LDS, two stages.  The partial last round of tiles over the CUs is
//                         computed in parts: 128-row half tiles, or tiles of the next kernel.
//   gemm_mid_kernel       (gemm_mid.h) 128 x 128, 128 x 64 and 64 x 64 tiles of the same instruction, loads straight into four LDS
//                         stages: shapes that have too few 256-wide tiles, and operands beyond the 2 GiB reach of a
//                         buffer descriptor's 32-bit offsets.
//   gemm_few_kernel       (gemm_few.h) up to 32 rows against a full-size weight: 16 or 32 columns per workgroup, K
//                         split over its waves.
//   gemm_any_kernel       (gemm_any.h) any K and alignment: 64- or 128-wide tiles, fp8 widened to bf16 on its way to
//                         the matrix cores.
//   gemm_tiny_kernel      the smallest of those, one output per thread.
//   gemm_nt_kernel        128 x 128 x 128 tiles, loads through registers: fp8 outputs whose rows or columns do not come in
//                         whole words (the other kernels' fp8 epilogue stores nothing smaller), and large results of
//                         fewer than two K-tiles.
#include "gemm_common.h"
#include "gemm_big.h"
#include "gemm_choice.h"

namespace ntfp8 {

// ---------------------------------------------------------------------------------------------
constexpr int kMinTransposed = 128;   // rows and columns of a result whose B is given as its transpose: more than this
enum GemmPath { kPathNone = -1, kPathAny = 0, kPathPlain = 1, kPathTiles = 2 };

int launch_mid(const BigLaunch& L, int fa, int fb, int tile_m, int tile_n, bool fp8_out, int tiles, hipStream_t st);
int launch_few(const BigProblem& p, int fa, int fb, hipStream_t st);
int launch_any(const BigLaunch& L, int fa, int fb, int tile, bool fp8_out, int tiles, hipStream_t st);
int launch_plain(const GemmDesc& g, hipStream_t st);
int launch_tiny(const BigProblem& p, int fa, int fb, hipStream_t st);
int run_amax_finalize(Workspace* ws, const ScalarIO& io, hipStream_t st);

// A launch of one problem of fewer than two K-tiles (the 256-wide tiles cannot take it) and more 64-wide tiles than the
// chip works on at once: nothing hides the prologue and epilogue of the one or two workgroups per CU of the smaller tiles,
// and 16- and 32-bit rows that end inside a 64-byte piece of memory make their streaming stores partial writes (for fp8
// only the transposed copy has any).  us, tiles of gemm_mid.h / gemm_nt_kernel, K 144 to 240:
//   bf16, whole pieces:   513 to 1024 tiles of 64 5.7 / 6.1, 1025 to 1536 9.0 / 7.8, 3136 x 3920 25.1 / 12.1
//   bf16, others:         up to 256 tiles 4.0 / 4.8, 257 to 512 5.7 / 5.3, 513 to 1024 8.0 / 6.1, more 18.5 / 10.1
//   fp8:                  257 to 512 tiles 9.3 / 11.3, 513 to 1024 10.7 / 12.2, 1025 to 1536 16.0 / 13.4
//   fp8 with its copy, N % 64 != 0:  257 to 512 11.7 / 12.5, 513 to 768 14.2 / 13.2, more 38.7 / 22.1
static bool short_k(const GemmDesc& g, int cus) {
    if (g.K >= 2 * kBK || g.tb) return false;
    const int64_t tiles = (((int64_t)g.M + 63) / 64) * (((int64_t)g.N + 63) / 64);
    const bool whole = (int64_t)g.N * (g.d_dtype == NTFP8_F32 ? 4 : is_fp8_out(g.d_dtype) ? 1 : 2) % 64 == 0;
    const int per_cu = whole ? 4 : !is_fp8_out(g.d_dtype) ? 1 : g.Dt ? 2 : 4;
    return tiles > per_cu * cus;
}

// which kernels serve a problem
static int path_of(const GemmDesc& g) {
    const bool aligned16 = (g.K % 16 == 0) &&
                           ((reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.B)) & 15) == 0 &&
                           (reinterpret_cast<uintptr_t>(g.D) & 15) == 0;
    if (!aligned16) return g.tb ? kPathNone : kPathAny;
    // the tiles' fp8 epilogue stores whole words through 32-bit buffer offsets
    const bool fp8_ok = !is_fp8_out(g.d_dtype) ||
                        (g.N % 16 == 0 && g.M % 4 == 0 && (int64_t)g.M * g.N < (1LL << 32) - 16 &&
                         (reinterpret_cast<uintptr_t>(g.Dt) & 15) == 0);
    // an operand given as its transpose, [K, N] or [K, M], is loaded in 16-byte pieces of its rows; a transposed A is
    // read only next to a transposed B (the wgrad form)
    if (g.ta && (!g.tb || g.M % 16 != 0)) return kPathNone;
    if (g.tb) return (g.N % 16 == 0 && fits32(g) && g.M > kMinTransposed && g.N > kMinTransposed && g.K >= 2 * kBK && fp8_ok) ? kPathTiles : kPathNone;
    if (!fp8_ok) return kPathPlain;
    return (int64_t)g.K * 128 < (1LL << 31) ? kPathTiles : kPathAny;   // (a tile's rows within reach of 32-bit offsets)
}

// The tile list of a launch, problem by problem, longest K first: the long tiles start together and the shorter ones fill
// the rounds behind them.  Returns the number of tiles.
static int64_t list_tiles(const GemmDesc* const* g, int n, Edge edge, BigLaunch* L) {
    int order[kBigMaxProblems];
    by_depth(g, n, order);
    *L = {};
    L->count = n;
    int64_t tiles = 0;
    for (int i = 0; i < n; ++i) {
        const GemmDesc& d = *g[order[i]];
        BigProblem& p = L->p[i];
        p.A = static_cast<const uint8_t*>(d.A);
        p.B = static_cast<const uint8_t*>(d.B);
        p.D = d.D;
        p.scale_a = d.sa;
        p.scale_b = d.sb;
        p.M = d.M;
        p.N = d.N;
        p.K = d.K;
        p.tiles_m = (d.M - 1) / edge.m + 1;
        p.tiles_n = (d.N - 1) / edge.n + 1;
        p.magic = magic_of((uint32_t)kGroupM * (uint32_t)p.tiles_n);
        p.tile_begin = (int)tiles;
        p.d_dtype = d.d_dtype;
        p.accumulate = d.accumulate;
        p.fp8 = Fp8Out{d.sd, static_cast<uint8_t*>(d.Dt), static_cast<Workspace*>(d.ws)};
        p.ex = GemmExtras{d.bias, d.bias_dtype, d.scale_inv};
        p.at = d.ta;
        p.bt = d.tb;
        tiles += (int64_t)p.tiles_m * p.tiles_n;
    }
    return tiles;
}

// A few rows against a weight whose columns the 64-wide tiles spread over few CUs (gemm_few.h).  The lines, us in 64-wide
// tiles / there, weights not in a cache:
//   16 rows, N x K:  4096 x 1024 4.5 / 4.6     4096 x 1536 5.2 / 4.9     5120 x 1536 5.2 / 5.7     8192 x 1536 6.5 / 6.8
//                    4096 x 2048 7.5 / 5.0     6144 x 3072 9.7 / 7.5     8192 x 4096 13.6 / 10.0   10240 x 4096 12.5 / 15.0
//   32 rows:         4096 x 2048 6.0 / 6.6     2048 x 3072 7.0 / 6.9     4096 x 4096 11.5 / 9.1    5120 x 4096 11.2 / 15.3
//                    4096 x 14336 31.9 / 21.7  5120 x 14336 31.5 / 39.5
static bool few_rows(const GemmDesc& g, int cus) {
    if (g.M > 32 || g.tb || is_fp8_out(g.d_dtype)) return false;
    if (g.M <= 16) return (g.K >= 2048 && g.N <= 32 * cus) || (g.K >= 1024 && g.N <= 16 * cus);
    return g.K >= 3072 && g.N <= 16 * cus;
}

// Bookkeeping of an fp8 output by the workgroup that finishes last, where the launch is one round of workgroups; behind more
// of them by a kernel of its own, since there every workgroup holds up the next one's start until its stores are out and
// its ticket is drawn.  us of GPU time, launches in a row, last workgroup / kernel: 1056 x 4064 x 144 19.4 / 15.6,
// 3552 x 3776 x 144 29.0 / 25.5 (1088 and 3540 64-wide tiles), 256 to 512 256-wide tiles 61.6 / 60.6; up to one round
// 7.1 / 7.2 and 3 us less of host time.
static void finish_inside(const GemmDesc* const* g, int n, int64_t tiles, BigLaunch* L) {
    if (n != 1 || !g[0]->fin || tiles > L->round_size) return;
    L->fin = *g[0]->fin;
    L->fin_blocks = (int)tiles;
}
static int finish_behind(const GemmDesc& g, int rc, hipStream_t st) {
    return rc == NTFP8_OK && g.fin ? run_amax_finalize(static_cast<Workspace*>(g.ws), *g.fin, st) : rc;
}

// One launch over up to kBigMaxProblems problems of the same operand formats, in the tile size that takes least (256-wide
// tiles: one more launch for a tail in parts).
template <int FA, int FB>
static int launch_tiles(const GemmDesc* const* g, int n, int cus, hipStream_t st) {
    const TileChoice choice = choose_tiles(g, n, cus);
    const Edge edge = choice.edge;
    const int parts = choice.parts;
    BigLaunch L;
    const int64_t tiles = list_tiles(g, n, edge, &L);
    if (tiles > 0x7fffffff) return NTFP8_ERR_SIZE;
    const bool fp8_out = is_fp8_out(g[0]->d_dtype);
    L.round_size = cus * (edge.m == 64 ? 2 : 1);
    L.round_magic = magic_of((uint32_t)L.round_size);
    finish_inside(g, n, tiles, &L);
    if (edge.m != 256) {
        const int rc = launch_mid(L, FA, FB, edge.m, edge.n, fp8_out, (int)tiles, st);
        return L.fin_blocks ? rc : finish_behind(*g[0], rc, st);
    }
    L.tail_tiles = parts > 1 ? (int)(tiles % cus) : 0;
    L.full_blocks = (int)tiles - L.tail_tiles;
    if (L.fin_blocks) L.fin_blocks = L.full_blocks + 2 * L.tail_tiles;
    (void)hipGetLastError();   // an error left behind by an unrelated earlier call is not this launch's
    auto go = [&](auto fp8_tag, auto bt_tag) {
        constexpr bool kFp8Out = decltype(fp8_tag)::value, kBT = decltype(bt_tag)::value;
        if (L.full_blocks > 0)
            hipLaunchKernelGGL((gemm_nt_big_kernel<FA, FB, 8, kFp8Out, kBT>), dim3(L.full_blocks), dim3(kBigThreads), 0, st, L);
        if (parts == 2)
            hipLaunchKernelGGL((gemm_nt_big_kernel<FA, FB, 4, kFp8Out, kBT>), dim3(2 * L.tail_tiles), dim3(kBigThreads), 0, st, L);
    };
#ifdef NTFP8_PROFILE_NARROW
    go(std::false_type{}, std::false_type{});
#else
    if (g[0]->tb) {
        if (fp8_out) go(std::true_type{}, std::true_type{});
        else go(std::false_type{}, std::true_type{});
    } else {
        if (fp8_out) go(std::true_type{}, std::false_type{});
        else go(std::false_type{}, std::false_type{});
    }
#endif
    int rc = hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
    if (parts > 2 && rc == NTFP8_OK) rc = launch_mid(L, FA, FB, 128, parts == 4 ? 128 : 64, fp8_out, parts * L.tail_tiles, st);
    return L.fin_blocks ? rc : finish_behind(*g[0], rc, st);
}

// Problems no 16-byte chunk of which lies in one piece: 128-wide tiles once there is one for every CU, 64-wide below
// (us, 64 / 128 wide: 1536 x 1536 x 1021, 144 tiles of 128, 18.4 / 20.4; 2048 x 2048 x 1021, 256 tiles, 23.4 / 21.6;
// 4096 x 4096 x 4095 262 / 179)
static int launch_any_tiles(const GemmDesc* const* g, int n, int cus, hipStream_t st) {
    BigLaunch L;
    int edge = 128;
    int64_t tiles = list_tiles(g, n, Edge{edge, edge}, &L);
    if (tiles < cus) edge = 64, tiles = list_tiles(g, n, Edge{edge, edge}, &L);
    if (tiles > 0x7fffffff) return NTFP8_ERR_SIZE;
    L.round_size = 2 * cus;   // (LDS: two workgroups of 128-wide tiles on a CU, more of the others)
    finish_inside(g, n, tiles, &L);
    const int rc = launch_any(L, g[0]->fmt_a, g[0]->fmt_b, edge, is_fp8_out(g[0]->d_dtype), (int)tiles, st);
    return L.fin_blocks ? rc : finish_behind(*g[0], rc, st);
}

// One problem of any K so small that a thread per output is done before a tile has been through LDS.  us, tiles / thread per
// output: K 16 to 31, up to 2^16 outputs 5.5 / 4.3, to 2^17 5.8 / 5.1, beyond 6.0 / 6.5; K 32 to 63 5.6 / 6.0 on average, equal
// at 40; fp8 outputs with their bookkeeping K 16 to 31 8.8 / 7.1.
static bool tiny(const GemmDesc& g) {
    const int64_t out = (int64_t)g.M * g.N;
    return g.K < 40 && out <= 1 << 17 && out * g.K <= 40 << 16;
}

static int dispatch(const GemmDesc* const* g, int n, int path, hipStream_t st) {
    const int fa = g[0]->fmt_a, fb = g[0]->fmt_b, cus = cu_count();   // (asked once: the question goes to the runtime)
    if (path == kPathNone) return NTFP8_ERR_UNSUPPORTED;
#ifdef NTFP8_PROFILE_NARROW
    // experiment builds of the profiling library carry one instantiation only: e4m3 x e4m3, K-contiguous operands,
    // 16-bit or fp32 output (what the loop experiments launch); everything else is refused
    if (fa != kE4M3 || fb != kE4M3 || path != kPathTiles || g[0]->tb || is_fp8_out(g[0]->d_dtype)) return NTFP8_ERR_UNSUPPORTED;
    return launch_tiles<kE4M3, kE4M3>(g, n, cus, st);
#else
    if (path == kPathAny && n == 1 && tiny(*g[0])) {
        BigLaunch L;
        list_tiles(g, 1, Edge{64, 64}, &L);
        return finish_behind(*g[0], launch_tiny(L.p[0], fa, fb, st), st);
    }
    if (path == kPathAny) return launch_any_tiles(g, n, cus, st);
    if (path == kPathPlain || (n == 1 && short_k(*g[0], cus))) return finish_behind(*g[0], launch_plain(*g[0], st), st);
    if (n == 1 && few_rows(*g[0], cus)) {
        BigLaunch L;
        list_tiles(g, 1, Edge{64, 64}, &L);
        return launch_few(L.p[0], fa, fb, st);
    }
    if (fa == kE4M3) return fb == kE4M3 ? launch_tiles<kE4M3, kE4M3>(g, n, cus, st) : launch_tiles<kE4M3, kE5M2>(g, n, cus, st);
    return fb == kE4M3 ? launch_tiles<kE5M2, kE4M3>(g, n, cus, st) : launch_tiles<kE5M2, kE5M2>(g, n, cus, st);
#endif
}

int run_gemm(const GemmDesc& g, hipStream_t st) {
    const GemmDesc* one[1] = {&g};
    return dispatch(one, 1, path_of(g), st);
}

// Independent problems (no output of one is an operand of another).  Problems that go to the same tile kernel and share their operand formats go out together, up to kBigMaxProblems per launch; the rest one by one.
int run_gemm_batch(const GemmDesc* g, int n, hipStream_t st) {
    bool done[64] = {false};
    if (n > 64) return NTFP8_ERR_SIZE;
    // a problem no kernel serves fails the whole call before anything is launched
    for (int i = 0; i < n; ++i)
        if (path_of(g[i]) == kPathNone) return NTFP8_ERR_UNSUPPORTED;
    for (int i = 0; i < n; ++i) {
        if (done[i]) continue;
        const GemmDesc* group[kBigMaxProblems];
        int cnt = 0;
        const int path = path_of(g[i]);
        group[cnt++] = &g[i];
        done[i] = true;
        if (path != kPathPlain) {
            for (int j = i + 1; j < n && cnt < kBigMaxProblems; ++j)
                if (!done[j] && g[j].fmt_a == g[i].fmt_a && g[j].fmt_b == g[i].fmt_b && path_of(g[j]) == path &&
                    is_fp8_out(g[j].d_dtype) == is_fp8_out(g[i].d_dtype) && g[j].tb == g[i].tb) {
                    group[cnt++] = &g[j];
                    done[j] = true;
                }
        }
        const int rc = dispatch(group, cnt, path, st);
        if (rc != NTFP8_OK) return rc;
    }
    return NTFP8_OK;
}

}  // namespace ntfp8

// The tile size of a launch of these problems on a GPU of `cus` CUs, and in how many parts the tiles of a partial last round of
// 256-wide ones are computed; for tests, which have to know what they reach.  Nothing is launched and no pointer of a
// problem is followed.  NTFP8_ERR_UNSUPPORTED where they do not share a launch of the tile kernels.
extern "C" __attribute__((visibility("default"))) int ntfp8_debug_gemm_tiles(const ntfp8_gemm_desc* p, int n, int cus, int* tile_m, int* tile_n, int* parts) {
    using namespace ntfp8;
    if (!p || !tile_m || !tile_n || !parts) return NTFP8_ERR_NULL;
    if (n < 1 || n > kBigMaxProblems || cus < 1) return NTFP8_ERR_SIZE;
    GemmDesc g[kBigMaxProblems] = {};
    const GemmDesc* all[kBigMaxProblems];
    for (int i = 0; i < n; ++i) {
        if (p[i].M < 1 || p[i].N < 1 || p[i].K < 1 || p[i].M > 0x7fffffff || p[i].N > 0x7fffffff || p[i].K > 0x7fffffff) return NTFP8_ERR_SIZE;
        g[i].A = p[i].A, g[i].B = p[i].B, g[i].D = p[i].D, g[i].Dt = p[i].D_t;
        g[i].M = (int)p[i].M, g[i].N = (int)p[i].N, g[i].K = (int)p[i].K;
        g[i].d_dtype = p[i].d_dtype, g[i].accumulate = p[i].accumulate;
        g[i].tb = p[i].b_transposed, g[i].ta = p[i].a_transposed;
        all[i] = &g[i];
        if (path_of(g[i]) != kPathTiles || g[i].tb != g[0].tb || is_fp8_out(g[i].d_dtype) != is_fp8_out(g[0].d_dtype)) return NTFP8_ERR_UNSUPPORTED;
    }
    if (n == 1 && (short_k(g[0], cus) || few_rows(g[0], cus))) return NTFP8_ERR_UNSUPPORTED;
    const TileChoice c = choose_tiles(all, n, cus);
    *tile_m = c.edge.m, *tile_n = c.edge.n, *parts = c.parts;
    return NTFP8_OK;
}

#ifdef NTFP8_STAMPS
// Profiling build only: copies the per-workgroup time stamps of the last gemm_nt_big_kernel launches to host memory
// (8 x uint64 per workgroup index, see gemm_big.h).  Synchronises the device.
extern "C" __attribute__((visibility("default"))) int ntfp8_debug_stamps(void* dst, size_t bytes) {
    if (!dst || bytes > sizeof(unsigned long long) * ntfp8::kStampSlots * 8) return dst ? NTFP8_ERR_SIZE : NTFP8_ERR_NULL;
    return hipMemcpyFromSymbol(dst, HIP_SYMBOL(ntfp8::g_stamps), bytes) == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}
extern "C" __attribute__((visibility("default"))) int ntfp8_debug_set_tile_order(int plain) {
    const int v = plain ? 1 : 0;
    return hipMemcpyToSymbol(HIP_SYMBOL(ntfp8::g_plain_tile_order), &v, sizeof(v)) == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH;
}
#endif
