// amax reduction, delayed-scaling history roll + scale update, saturating casts to OCP FP8,
// dequantisation and byte transpose for gfx950.  All kernels are HBM-bandwidth bound on large tensors: one pass
// over the input with 128-bit loads and stores, a wavefront reduction for the amax, one word stored per
// block and the bookkeeping by the highest-numbered block, which waits for the words, in the same launch.
#include "common.h"
#include "reduce.h"

namespace ntfp8 {

constexpr int kThreads = 256;       // dequant / transpose / scalar kernels
constexpr int kFlatThreads = 1024;  // streaming quantise kernel: one block per CU, 16 waves
constexpr int kTileThreads = 256;   // tile (transposing) quantise kernel
constexpr int kVec = 16;  // elements per thread per step: 16 fp8 bytes = one 128-bit store

typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));


// ---------------------------------------------------------------------------------------------
// Loads of E = 4 or 16 elements.  `mx` receives max|x| of them as a comparable unsigned pattern in
// the *source* format (fp32 bits for float, 16-bit patterns for half / bf16).
// kStream: the load is marked streaming and leaves no line behind in the memory-side cache: for passes that read their
// tensor once, or last.  In a training step they run behind a GEMM whose output fills that cache, and an ordinary read waits
// for the lines it displaces.  The amax pass of current scaling, which a cast follows, uses ordinary loads: the cast finds part
// of the tensor in the cache (bf16 4096 x 4096, amax and cast: ordinary / ordinary 15.4 us, ordinary / streaming 13.7,
// streaming / streaming 18.2).  Streaming loads have to take whole lines, since a line is not there for a second load.
template <bool kStream, int kAlign, typename V>
__device__ __forceinline__ V load_vec(const void* p) {   // p: kAlign-byte aligned
    typedef V VA __attribute__((aligned(kAlign)));
    if constexpr (kStream) return __builtin_nontemporal_load(static_cast<const VA*>(p));
    else return *static_cast<const VA*>(p);
}
template <typename T>
struct Src;

template <>
struct Src<float> {
    static constexpr int kDtype = NTFP8_F32;
    __device__ static __forceinline__ void unpack(u4 w, float (&v)[4], uint32_t& mx) {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = __uint_as_float(w[i]);
            m = max(m, w[i] & 0x7fffffffu);
        }
        mx = m;
    }
    template <int E, bool kStream>
    __device__ static __forceinline__ void load(const float* p, float (&v)[E], uint32_t& mx) {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < E / 4; ++i) {
            const f4 t = load_vec<kStream, 4, f4>(p + 4 * i);
            v[4 * i + 0] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        }
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t a = __float_as_uint(v[i]) & 0x7fffffffu;
            m = a > m ? a : m;
        }
        mx = m;
    }
    __device__ static __forceinline__ float load1(const float* p, uint32_t& m) {
        const float x = *p;
        m = __float_as_uint(x) & 0x7fffffffu;
        return x;
    }
    __device__ static __forceinline__ bool has_nan(uint32_t m) { return m > kInfBits; }
    __device__ static __forceinline__ uint32_t to_f32_bits(uint32_t m) { return m; }
};

template <bool kBf16>
struct Src16 {
    __device__ static __forceinline__ float cvt(uint32_t h) {
        if constexpr (kBf16) return bf16_bits_to_float(h);
        else return half_bits_to_float(h);
    }
    template <int E, bool kStream>
    __device__ static __forceinline__ void load(const uint16_t* p, float (&v)[E], uint32_t& mx) {
        uint32_t w[E / 2];
        if constexpr (E == 4) {
            typedef uint32_t u2 __attribute__((ext_vector_type(2)));
            const u2 a = load_vec<kStream, 2, u2>(p);
            w[0] = a.x, w[1] = a.y;
        } else {
#pragma unroll
            for (int i = 0; i < E / 8; ++i) {
                const u4 a = load_vec<kStream, 2, u4>(p + 8 * i);
                w[4 * i] = a.x, w[4 * i + 1] = a.y, w[4 * i + 2] = a.z, w[4 * i + 3] = a.w;
            }
        }
        widen<E>(w, v, mx);
    }
    __device__ static __forceinline__ void unpack(u4 w, float (&v)[8], uint32_t& mx) {
        const uint32_t a[4] = {w.x, w.y, w.z, w.w};
        widen<8>(a, v, mx);
    }
    template <int E>
    __device__ static __forceinline__ void widen(const uint32_t (&w)[E / 2], float (&v)[E], uint32_t& mx) {
        typedef unsigned short us2 __attribute__((ext_vector_type(2)));
        us2 m = {0, 0};
#pragma unroll
        for (int i = 0; i < E / 2; ++i) {
            if constexpr (kBf16) {
                v[2 * i] = __uint_as_float(w[i] << 16);
                v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
            } else {
                v[2 * i] = half_bits_to_float(w[i] & 0xffffu);
                v[2 * i + 1] = half_bits_to_float(w[i] >> 16);
            }
            const uint32_t ab = w[i] & 0x7fff7fffu;
            us2 t;
            __builtin_memcpy(&t, &ab, 4);
            m = __builtin_elementwise_max(m, t);
        }
        mx = m.x > m.y ? m.x : m.y;
    }
    __device__ static __forceinline__ float load1(const uint16_t* p, uint32_t& m) {
        const uint32_t h = *p;
        m = h & 0x7fffu;
        return cvt(h);
    }
    __device__ static __forceinline__ bool has_nan(uint32_t m) { return m > (kBf16 ? 0x7f80u : 0x7c00u); }
    __device__ static __forceinline__ uint32_t to_f32_bits(uint32_t m) { return __float_as_uint(cvt(m)); }
};

struct bf16_tag {};
struct f16_tag {};
template <>
struct Src<bf16_tag> : Src16<true> {
    static constexpr int kDtype = NTFP8_BF16;
    typedef uint16_t elem;
};
template <>
struct Src<f16_tag> : Src16<false> {
    static constexpr int kDtype = NTFP8_F16;
    typedef uint16_t elem;
};
template <typename T>
struct ElemOf {
    typedef uint16_t type;
};
template <>
struct ElemOf<float> {
    typedef float type;
};

// E scaled values -> E fp8 bytes.  `slow` = this group may contain a NaN (NaN input or a
// degenerate scale): patch the NaN bytes to sign|0x7F.
template <int F, int E>
__device__ __forceinline__ void encode(const float (&v)[E], float scale, bool slow, uint32_t (&w)[E / 4]) {
    float y[E];
#pragma unroll
    for (int i = 0; i < E; ++i) y[i] = v[i] * scale;
#pragma unroll
    for (int i = 0; i < E / 4; ++i)
        w[i] = cvt4<F>(sat<F>(y[4 * i]), sat<F>(y[4 * i + 1]), sat<F>(y[4 * i + 2]), sat<F>(y[4 * i + 3]));
    if (slow) {
#pragma unroll
        for (int i = 0; i < E; ++i) w[i >> 2] = patch_nan(w[i >> 2], i & 3, y[i]);
    }
}
template <int F>
__device__ __forceinline__ u4 encode16(const float (&v)[16], float scale, bool slow) {
    uint32_t w[4];
    encode<F, 16>(v, scale, slow, w);
    return (u4){w[0], w[1], w[2], w[3]};
}

template <int F>
__device__ __forceinline__ uint8_t encode1(float x, float scale) {
    const float y = x * scale;
    uint32_t w = cvt4<F>(sat<F>(y), 0.0f, 0.0f, 0.0f);
    w = patch_nan(w, 0, y);
    return (uint8_t)(w & 0xffu);
}

// ---------------------------------------------------------------------------------------------
// The bookkeeping of reduce.h for maxima that another kernel (the fp8-output GEMM epilogue) left in the slots.
__global__ __launch_bounds__(64) void amax_finalize_kernel(Workspace* ws, ScalarIO io) {
    const EpiloguePrefetch pre = prefetch_epilogue(io, kModeDelayed);
    finalize_wave(ws, io, kModeDelayed, pre);
}

__device__ __forceinline__ bool degenerate_scale(float s) {
    const uint32_t b = __float_as_uint(s) & 0x7fffffffu;
    return b == 0u || b >= kInfBits;
}

// Cast-only launches: the scale the bytes were made with, beside an amax of zero (none was taken).
__device__ __forceinline__ void record_cast_scale(const ScalarIO& io, float scale, uint32_t bid) {
    if (io.scale_out && bid == 0 && threadIdx.x == 0) {
        *io.scale_out = scale;
        *io.amax_out = 0.0f;
    }
}

// ---------------------------------------------------------------------------------------------
// Flat (no transpose) kernel: amax only, cast only, or both (delayed scaling).
//
// Bound by HBM.  A lane's load is 16 bytes and the wave's 64 loads lie side by side: 1 KB of whole lines per instruction
// (16 elements per lane in a row, as two or four loads 32 or 64 bytes apart, touch every line two or four times, which a
// streaming load pays for; the bytes then leave 8 or 4 a lane).  A workgroup takes spans of 16384 elements, two in flight.
// us, 16 elements per lane / side by side, 4096 x 4096 and 4096 x 14336: bf16 delayed step 12.5 and 34.0 / 12.0 and 32.6, cast
// 10.4 and 31.4 / 9.8 and 29.9 (5.9 TB/s), current scaling 15.4 and 47.6 / 13.7 and 44.2; fp32 delayed step 24.9 and 76.6 /
// 17.3 and 51.7, cast 16.2 and 54.3 / 15.4 and 49.9.  (Probes with two to eight workgroups of 256 or 512 threads per CU: 5 to
// 20 % slower.  A span requested again as soon as it is done, instead of two at a time: the same, and 0.2 us more for small
// tensors.)
template <typename S>
constexpr int kChunk = 16 / (int)sizeof(typename ElemOf<S>::type);   // elements of a 16-byte load
template <typename S>
constexpr int kSpan = kFlatThreads * (kVec / kChunk<S>);             // loads of a span

template <int E>
__device__ __forceinline__ void store_chunk(uint8_t* __restrict__ p, const uint32_t (&w)[E / 4]) {   // p: E-byte aligned
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    if constexpr (E == 8) __builtin_nontemporal_store((u2){w[0], w[1]}, reinterpret_cast<u2*>(p));
    else __builtin_nontemporal_store(w[0], reinterpret_cast<uint32_t*>(p));
}

// Streams a tensor of n elements, n_vec whole 16-byte chunks of it as vectors: `body(v, m, index)` for every chunk,
// `one(x, m, index)` for elements past them (all of them where a pointer is misaligned).
// kOne: one chunk for every thread is all there is (a kernel of its own: small tensors are bound by latency, which code read
// from memory is part of).
template <typename S, bool kOne, typename Body, typename One>
__device__ __forceinline__ void for_each_chunk(const typename ElemOf<S>::type* __restrict__ x, int64_t n_vec, int64_t n, uint32_t bid,
                                               uint32_t nblocks, Body body, One one) {
    typedef Src<S> L;
    constexpr int E = kChunk<S>, U = kVec / E;
    const int64_t full = n_vec / kSpan<S>;
    int64_t g = bid;
    auto spans = [&](auto count_tag) {
        constexpr int G = decltype(count_tag)::value;
        float v[G * U][E];
        uint32_t m[G * U];
        auto index = [&](int k) -> int64_t {
            return ((g + (int64_t)(k / U) * nblocks) * kSpan<S> + k % U * kFlatThreads + (int)threadIdx.x) * E;
        };
#pragma unroll
        for (int k = 0; k < G * U; ++k) L::template load<E, true>(x + index(k), v[k], m[k]);
#pragma unroll
        for (int k = 0; k < G * U; ++k) body(v[k], m[k], index(k));
        g += (int64_t)G * nblocks;
    };
    auto chunk = [&](int64_t c) {
        float v[E];
        uint32_t m;
        L::template load<E, true>(x + c * E, v, m);
        body(v, m, c * E);
    };
    if constexpr (kOne) {
        const int64_t c = (int64_t)bid * kFlatThreads + threadIdx.x;
        if (c < n_vec) chunk(c);
    } else {
        while (g + nblocks < full) spans(std::integral_constant<int, 2>{});
        if (g < full) spans(std::integral_constant<int, 1>{});
        if (g == full)   // what is left of the last span: one workgroup's
            for (int64_t c = full * kSpan<S> + threadIdx.x; c < n_vec; c += kFlatThreads) chunk(c);
    }
    for (int64_t j = n_vec * E + (int64_t)bid * kFlatThreads + threadIdx.x; j < n; j += (int64_t)nblocks * kFlatThreads) {
        uint32_t m;
        const float v = L::load1(x + j, m);
        one(v, m, j);
    }
}

// max|x| alone: 16 elements per lane in a row and ordinary loads (the first touches every line, the others find it in the
// cache; and the pass that follows finds lines in the memory-side cache).  fp32 11008 x 4096, 16 elements in a row / side by
// side: 32.2 / 33.1 us.
template <typename S, bool kOne>
__device__ __forceinline__ uint32_t flat_max(const typename ElemOf<S>::type* __restrict__ x, int64_t n_vec, int64_t n, uint32_t bid,
                                             uint32_t nblocks) {
    typedef Src<S> L;
    uint32_t m_run = 0;
    if constexpr (kOne) {
        constexpr int E = kChunk<S>;
        const int64_t c = (int64_t)bid * kFlatThreads + threadIdx.x;
        float v[E];
        uint32_t m = 0;
        if (c < n_vec) L::template load<E, false>(x + c * E, v, m);
        const int64_t j = n_vec * E + c;   // fewer than E elements past the chunks
        if (j < n) (void)L::load1(x + j, m_run);
        return m > m_run ? m : m_run;
    }
    n_vec /= kVec / kChunk<S>;
    const int64_t stride = (int64_t)nblocks * kFlatThreads;
    int64_t i = (int64_t)bid * kFlatThreads + threadIdx.x;
    for (; i + stride < n_vec; i += 2 * stride) {
        float v0[16], v1[16];
        uint32_t m0, m1;
        L::template load<16, false>(x + i * kVec, v0, m0);
        L::template load<16, false>(x + (i + stride) * kVec, v1, m1);
        m_run = m0 > m_run ? m0 : m_run;
        m_run = m1 > m_run ? m1 : m_run;
    }
    if (i < n_vec) {
        float v0[16];
        uint32_t m0;
        L::template load<16, false>(x + i * kVec, v0, m0);
        m_run = m0 > m_run ? m0 : m_run;
    }
    for (int64_t j = n_vec * kVec + (int64_t)bid * kFlatThreads + threadIdx.x; j < n; j += stride) {
        uint32_t m;
        (void)L::load1(x + j, m);
        m_run = m > m_run ? m : m_run;
    }
    return m_run;
}

template <typename S, int F, int MODE, bool kOne = false>
__device__ __forceinline__ void quant_flat_body(const typename ElemOf<S>::type* __restrict__ x, int64_t n_vec, int64_t n,
                                                uint8_t* __restrict__ out, const float* __restrict__ scale_ptr,
                                                Workspace* ws, const ScalarIO& io, uint32_t bid, uint32_t nblocks) {
    typedef Src<S> L;
    constexpr bool kCast = MODE != kModeAmaxOnly;
    constexpr bool kAmax = MODE != kModeCastOnly;
    constexpr int E = kChunk<S>;
    float scale = 1.0f;
    bool degen = false;
    if constexpr (kCast) {
        scale = *scale_ptr;
        degen = degenerate_scale(scale);
    }
    if constexpr (!kAmax) record_cast_scale(io, scale, bid);
    EpiloguePrefetch pre = {0.0f, 1.0f};
    if constexpr (kAmax) pre = prefetch_epilogue(io, MODE);
    uint32_t m_run = 0;  // in source-format bits
    if constexpr (!kCast) {
        m_run = flat_max<S, kOne>(x, n_vec, n, bid, nblocks);
    } else {
        for_each_chunk<S, kOne>(
            x, n_vec, n, bid, nblocks,
            [&](const float(&v)[E], uint32_t m, int64_t at) {
                if constexpr (kAmax) m_run = m > m_run ? m : m_run;
                uint32_t w[E / 4];
                encode<F, E>(v, scale, degen || L::has_nan(m), w);
                store_chunk<E>(out + at, w);
            },
            [&](float v, uint32_t m, int64_t j) {
                if constexpr (kAmax) m_run = m > m_run ? m : m_run;
                out[j] = encode1<F>(v, scale);
            });
    }
    if constexpr (kAmax) publish_and_finalize<kFlatThreads>(L::to_f32_bits(m_run), ws, io, MODE, pre, bid, nblocks);
}

template <typename S, int F, int MODE, bool kOne>
__global__ __launch_bounds__(kFlatThreads) void quant_flat_kernel(const typename ElemOf<S>::type* __restrict__ x,
                                                              int64_t n_vec, int64_t n, uint8_t* __restrict__ out,
                                                              const float* __restrict__ scale_ptr, Workspace* ws,
                                                              ScalarIO io) {
    quant_flat_body<S, F, MODE, kOne>(x, n_vec, n, out, scale_ptr, ws, io, blockIdx.x, gridDim.x);
}

// One source tensor, both formats, one pass: the fused delayed-scaling step of an e4m3 role and an e5m2 role that
// quantise the same tensor (4 bytes per bf16 element instead of 2 x 3).  The amax is shared; each role has its own
// scale, history and output.
template <typename S>
__global__ __launch_bounds__(kFlatThreads) void quant_flat_dual_kernel(const typename ElemOf<S>::type* __restrict__ x,
                                                                   int64_t n_vec, int64_t n, uint8_t* __restrict__ out0,
                                                                   uint8_t* __restrict__ out1, Workspace* ws, ScalarIO io0,
                                                                   ScalarIO io1) {
    typedef Src<S> L;
    const float s0 = *io0.scale_state, s1 = *io1.scale_state;
    const bool d0 = degenerate_scale(s0), d1 = degenerate_scale(s1);
    const EpiloguePrefetch pre0 = prefetch_epilogue(io0, kModeDelayed);
    const EpiloguePrefetch pre1 = prefetch_epilogue(io1, kModeDelayed);
    uint32_t m_run = 0;
    constexpr int E = kChunk<S>;
    for_each_chunk<S, false>(
        x, n_vec, n, blockIdx.x, gridDim.x,
        [&](const float(&v)[E], uint32_t m, int64_t at) {
            m_run = m > m_run ? m : m_run;
            uint32_t w[E / 4];
            encode<kE4M3, E>(v, s0, d0 || L::has_nan(m), w);
            store_chunk<E>(out0 + at, w);
            encode<kE5M2, E>(v, s1, d1 || L::has_nan(m), w);
            store_chunk<E>(out1 + at, w);
        },
        [&](float v, uint32_t m, int64_t j) {
            m_run = m > m_run ? m : m_run;
            out0[j] = encode1<kE4M3>(v, s0);
            out1[j] = encode1<kE5M2>(v, s1);
        });
    publish_and_finalize<kFlatThreads>(L::to_f32_bits(m_run), ws, io0, kModeDelayed, pre0, blockIdx.x, gridDim.x, &io1, &pre1);
}

// Several tensors, one launch (the fused delayed-scaling step of each): the workgroups of tensor t follow those of
// tensor t - 1, so the tail of one tensor (its last loads, its reduction, its bookkeeping) runs under the streaming
// of the next instead of in front of a kernel boundary.  Every tensor has its own workspace.
constexpr int kMaxMulti = 16;
struct MultiQuant {
    struct Tensor {
        const void* x;
        uint8_t* out;
        int64_t n_vec, n;
        Workspace* ws;
        ScalarIO io;
        int first_block, blocks;
    } t[kMaxMulti];
    int count;
};

template <typename S, int F>
__global__ __launch_bounds__(kFlatThreads) void quant_flat_multi_kernel(const MultiQuant Q) {
    int which = 0;
#pragma unroll
    for (int i = 1; i < kMaxMulti; ++i)
        if (i < Q.count && (int)blockIdx.x >= Q.t[i].first_block) which = i;
    const MultiQuant::Tensor& T = Q.t[which];
    quant_flat_body<S, F, kModeDelayed>(static_cast<const typename ElemOf<S>::type*>(T.x), T.n_vec, T.n, T.out,
                                        T.io.scale_state, T.ws, T.io, blockIdx.x - T.first_block, T.blocks);
}

// ---------------------------------------------------------------------------------------------
// Byte tiles turned around in LDS: the cast that also writes the transposed bytes, and the transpose of fp8 bytes.
//
// A workgroup of 256 threads takes a tile of kT x kT bytes; a thread holds 4 rows x E columns of it (E = 16: kT = 128,
// E = 4: kT = 64).  Four v_perm pairs turn each 4 x 4 block of bytes around, so LDS receives whole words, [column][row]:
// a quarter of the stores that single bytes would need.  The 16-byte row chunks of a column are XORed with the
// column's group (E = 16) or the columns are one word apart from a multiple of the banks (E = 4), which spreads both the
// stores and the reads over the banks.  Global accesses are 16 bytes wide whatever the alignment of a row (gfx950
// serves misaligned ones).  At the edges of the matrix loads are clamped to its last row and column (the copies reach
// neither a stored byte nor change a maximum) and the last bytes of a row are stored 8, 4, 2, 1 at a time.
//
// Bound by HBM on large tensors, by the latency of one tile on small ones.  128-wide tiles from one tile per CU on,
// 64-wide ones below: see the measurements at tile_edge().  Against 64-wide tiles of single bytes (transpose), byte
// stores into LDS (cast) and one element per thread (any shape that is no multiple of 128), us before / now: transpose
// 4096 x 4096 19.7 / 6.0 (5.5 TB/s), 2048 x 2048 6.5 / 3.0; fp32 cast with copy 4096 x 4096 26.6 / 16.9, 11008 x 4096
// 68 / 54 (5.0 TB/s), 4095 x 4097 143 / 27; bf16 delayed step with copy 1021 x 1024 13.5 / 7.1, 1021 x 2304 19.7 / 9.1.
template <int E>
struct Tile {
    static constexpr int kT = E == 16 ? 128 : 64;
    static constexpr int kPitch = E == 16 ? 32 : 17;   // words between columns in LDS
    static constexpr int kChunks = kT / 16;            // 16-byte row chunks per column
};
typedef u4 u4_any __attribute__((aligned(1)));

// the first n (1 .. 15) bytes of q
__device__ __forceinline__ void store_head(uint8_t* __restrict__ p, u4 q, int n) {
    typedef uint64_t u64_any __attribute__((aligned(1)));
    typedef uint32_t u32_any __attribute__((aligned(1)));
    typedef uint16_t u16_any __attribute__((aligned(1)));
    uint64_t lo = q.x | ((uint64_t)q.y << 32);
    if (n & 8) {
        *reinterpret_cast<u64_any*>(p) = lo;
        lo = q.z | ((uint64_t)q.w << 32);
        p += 8;
    }
    if (n & 4) {
        *reinterpret_cast<u32_any*>(p) = (uint32_t)lo;
        lo >>= 32;
        p += 4;
    }
    if (n & 2) {
        *reinterpret_cast<u16_any*>(p) = (uint16_t)lo;
        lo >>= 16;
        p += 2;
    }
    if (n & 1) *p = (uint8_t)lo;
}

// w[r][q] = bytes 4 q .. 4 q + 3 of row r of the thread's block -> LDS
template <int E>
__device__ __forceinline__ void deposit_block(uint32_t* __restrict__ tile, const uint32_t (&w)[4][E / 4], int cgrp, int rgrp) {
    const int pos = E == 16 ? ((((rgrp >> 2) ^ cgrp) & 7) << 2) | (rgrp & 3) : rgrp;
#pragma unroll
    for (int q = 0; q < E / 4; ++q) {
        const uint32_t a = __builtin_amdgcn_perm(w[1][q], w[0][q], 0x05010400u), b = __builtin_amdgcn_perm(w[3][q], w[2][q], 0x05010400u);
        const uint32_t c = __builtin_amdgcn_perm(w[1][q], w[0][q], 0x07030602u), d = __builtin_amdgcn_perm(w[3][q], w[2][q], 0x07030602u);
        uint32_t* t = tile + (cgrp * E + 4 * q) * Tile<E>::kPitch + pos;
        t[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        t[Tile<E>::kPitch] = __builtin_amdgcn_perm(b, a, 0x07060302u);
        t[2 * Tile<E>::kPitch] = __builtin_amdgcn_perm(d, c, 0x05040100u);
        t[3 * Tile<E>::kPitch] = __builtin_amdgcn_perm(d, c, 0x07060302u);
    }
}

// the tile's columns as rows of out_t [cols, rows]
template <int E>
__device__ __forceinline__ void emit_columns(const uint32_t* __restrict__ tile, uint8_t* __restrict__ out_t, int64_t rows,
                                             int64_t cols, int64_t row0, int64_t col0) {
    typedef Tile<E> T;
#pragma unroll
    for (int it = 0; it < T::kT * T::kChunks / kTileThreads; ++it) {
        const int idx = threadIdx.x + kTileThreads * it;
        const int c = idx / T::kChunks, ch = idx % T::kChunks;
        u4 q;
        if constexpr (E == 16) {
            q = *reinterpret_cast<const u4*>(tile + c * T::kPitch + (((ch ^ (c >> 4)) & 7) << 2));
        } else {
            const uint32_t* t = tile + c * T::kPitch + 4 * ch;
            q = (u4){t[0], t[1], t[2], t[3]};
        }
        const int64_t r = row0 + ch * 16;
        if (col0 + c >= cols || r >= rows) continue;
        uint8_t* p = out_t + (col0 + c) * rows + r;
        if (r + 16 <= rows) {
            __builtin_nontemporal_store(q, reinterpret_cast<u4_any*>(p));
        } else {
            store_head(p, q, (int)(rows - r));
        }
    }
}

// one row of the thread's block: `inside` of its bytes lie inside the matrix
template <int E>
__device__ __forceinline__ void store_row_bytes(uint8_t* __restrict__ p, const uint32_t (&w)[E / 4], int64_t inside) {
    typedef uint32_t u32_any __attribute__((aligned(1)));
    if constexpr (E == 16) {
        const u4 q = {w[0], w[1], w[2], w[3]};
        if (inside >= 16) __builtin_nontemporal_store(q, reinterpret_cast<u4_any*>(p));
        else store_head(p, q, (int)inside);
    } else {
        if (inside >= 4) *reinterpret_cast<u32_any*>(p) = w[0];
        else store_head(p, (u4){w[0], 0u, 0u, 0u}, (int)inside);
    }
}

// Eight lanes hold 128 columns of a row, lane l as Q loads of 16 / Q columns each, 128 / Q columns apart (so that one load of
// the eight lanes is a whole line).  gather_span exchanges the loads' bytes among Q neighbouring lanes; lane l then holds the
// 16 consecutive columns of group span_group(l).
template <int Q>
__device__ __forceinline__ int span_group(int l) {
    return (l % Q) * (8 / Q) + l / Q;
}
template <int kPerm>
__device__ __forceinline__ void exchange(uint32_t& a, uint32_t& b, bool upper) {   // a lower lane's b <-> its upper partner's a
    const uint32_t r = (uint32_t)__builtin_amdgcn_mov_dpp((int)(upper ? a : b), kPerm, 0xf, 0xf, true);
    a = upper ? r : a;
    b = upper ? b : r;
}
template <int Q>
__device__ __forceinline__ void gather_span(uint32_t (&w)[4], int l) {
    if constexpr (Q == 2) {   // w[0..1]: the first load's words
        exchange<0xB1>(w[0], w[2], l & 1);   // quad_perm [1, 0, 3, 2]
        exchange<0xB1>(w[1], w[3], l & 1);
    } else {
        exchange<0xB1>(w[0], w[1], l & 1);
        exchange<0xB1>(w[2], w[3], l & 1);
        exchange<0x4E>(w[0], w[2], l & 2);   // quad_perm [2, 3, 0, 1]
        exchange<0x4E>(w[1], w[3], l & 2);
    }
}

template <typename S, int F, bool kAmax, int E, bool kStream>
__global__ __launch_bounds__(kTileThreads) void quant_transpose_kernel(const typename ElemOf<S>::type* __restrict__ x,
                                                                   int64_t rows, int64_t cols,
                                                                   uint8_t* __restrict__ out,
                                                                   uint8_t* __restrict__ out_t,
                                                                   const float* __restrict__ scale_ptr,
                                                                   Workspace* ws, ScalarIO io) {
    typedef Src<S> L;
    typedef Tile<E> T;
    // whole lines per load of eight lanes (not for fp32 rows that start anywhere: 36.7 against 34.8 us, 4095 x 4097)
    constexpr bool kLines = E == 16 && (kStream || sizeof(*x) == 2);
    __shared__ __attribute__((aligned(16))) uint32_t tile[T::kT * T::kPitch];
    const float scale = *scale_ptr;
    const bool degen = degenerate_scale(scale);
    const int64_t tiles_c = (cols + T::kT - 1) / T::kT;
    const int64_t tiles = ((rows + T::kT - 1) / T::kT) * tiles_c;
    const int lane_grp = threadIdx.x % (T::kT / E), rgrp = threadIdx.x / (T::kT / E);
    EpiloguePrefetch pre = {0.0f, 1.0f};
    if constexpr (kAmax) pre = prefetch_epilogue(io, kModeDelayed);
    else record_cast_scale(io, scale, blockIdx.x);
    uint32_t m_run = 0;
    // persistent over tiles: the number of blocks (and so of reduction atomics) stays small
    for (int64_t tile_id = blockIdx.x; tile_id < tiles; tile_id += gridDim.x) {
        const int64_t row0 = (tile_id / tiles_c) * T::kT, col0 = (tile_id % tiles_c) * T::kT;
        uint32_t w[4][E / 4];
        int cgrp = lane_grp;   // the thread's columns: E from E cgrp on
        bool whole = false;
        if constexpr (kLines) whole = col0 + T::kT <= cols;   // uniform
        if (whole) {
            if constexpr (kLines) {
                constexpr int C = kChunk<S>, Q = E / C;   // Q loads of C elements a row, kT / Q columns apart
                cgrp = span_group<Q>(lane_grp);
                u4 raw[4][Q];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = row0 + rgrp * 4 + r;
                    const typename ElemOf<S>::type* p = x + (row < rows ? row : rows - 1) * cols + col0 + lane_grp * C;
#pragma unroll
                    for (int q = 0; q < Q; ++q) raw[r][q] = load_vec<kStream, sizeof(*x), u4>(p + q * (T::kT / Q));
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = row0 + rgrp * 4 + r;
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        float v[C];
                        uint32_t e[C / 4], m;
                        L::unpack(raw[r][q], v, m);
                        encode<F, C>(v, scale, degen || L::has_nan(m), e);
#pragma unroll
                        for (int i = 0; i < C / 4; ++i) w[r][q * (C / 4) + i] = e[i];
                        if constexpr (kAmax) m_run = m > m_run ? m : m_run;
                    }
                    gather_span<Q>(w[r], lane_grp);
                    if (out && row < rows) store_row_bytes<E>(out + row * cols + col0 + cgrp * E, w[r], E);
                }
            }
        } else {
            const int64_t c = col0 + cgrp * E;
            float v[4][E];
            uint32_t m[4];
            if (c + E <= cols) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = row0 + rgrp * 4 + r;
                    L::template load<E, kStream>(x + (row < rows ? row : rows - 1) * cols + c, v[r], m[r]);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = row0 + rgrp * 4 + r;
                    const typename ElemOf<S>::type* p = x + (row < rows ? row : rows - 1) * cols;
                    m[r] = 0;
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        uint32_t me;
                        v[r][e] = L::load1(p + (c + e < cols ? c + e : cols - 1), me);
                        m[r] = me > m[r] ? me : m[r];
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = row0 + rgrp * 4 + r;
                if constexpr (kAmax) m_run = m[r] > m_run ? m[r] : m_run;
                encode<F, E>(v[r], scale, degen || L::has_nan(m[r]), w[r]);
                if (out && row < rows && c < cols) store_row_bytes<E>(out + row * cols + c, w[r], cols - c);
            }
        }
        deposit_block<E>(tile, w, cgrp, rgrp);
        __syncthreads();
        emit_columns<E>(tile, out_t, rows, cols, row0, col0);
        __syncthreads();  // the tile buffer is reused by the next trip
    }
    if constexpr (kAmax) publish_and_finalize<kTileThreads>(L::to_f32_bits(m_run), ws, io, kModeDelayed, pre);
}

// The same for small tensors, one element per thread: bound by the latency of one pass, which a tile's trip through LDS
// and its code (read from memory by every CU) lengthen.  us, tiles / here: cast of 333 x 515 fp32 4.9 / 3.9, 223 x 162
// 4.8 / 3.2, delayed step of 2^15 elements bf16 5.8 / 4.7.
template <typename S, int F, bool kAmax>
__global__ __launch_bounds__(kThreads) void quant_transpose_small_kernel(const typename ElemOf<S>::type* __restrict__ x, int rows, int cols,
                                                                     uint8_t* __restrict__ out, uint8_t* __restrict__ out_t,
                                                                     const float* __restrict__ scale_ptr, Workspace* ws, ScalarIO io) {
    typedef Src<S> L;
    const float scale = *scale_ptr;
    EpiloguePrefetch pre = {0.0f, 1.0f};
    if constexpr (kAmax) pre = prefetch_epilogue(io, kModeDelayed);
    else record_cast_scale(io, scale, blockIdx.x);
    const uint32_t n = (uint32_t)rows * cols;
    uint32_t m = 0;
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j < n) {
        const uint8_t b = encode1<F>(L::load1(x + j, m), scale);
        if (out) out[j] = b;
        out_t[j % (uint32_t)cols * rows + j / (uint32_t)cols] = b;
    }
    if constexpr (kAmax) publish_and_finalize<kThreads>(L::to_f32_bits(m), ws, io, kModeDelayed, pre);
}

// [rows, cols] bytes -> [cols, rows]
template <int E>
__global__ __launch_bounds__(kTileThreads) void transpose_kernel(const uint8_t* __restrict__ in, int64_t rows, int64_t cols,
                                                                 uint8_t* __restrict__ out) {
    typedef Tile<E> T;
    __shared__ __attribute__((aligned(16))) uint32_t tile[T::kT * T::kPitch];
    const int64_t tiles_c = (cols + T::kT - 1) / T::kT;
    const int64_t tiles = ((rows + T::kT - 1) / T::kT) * tiles_c;
    const int cgrp = threadIdx.x % (T::kT / E), rgrp = threadIdx.x / (T::kT / E);
    for (int64_t tile_id = blockIdx.x; tile_id < tiles; tile_id += gridDim.x) {
        const int64_t row0 = (tile_id / tiles_c) * T::kT, col0 = (tile_id % tiles_c) * T::kT;
        const int64_t c = col0 + cgrp * E;
        uint32_t w[4][E / 4];
        typedef uint32_t win __attribute__((ext_vector_type(E / 4)));
        typedef win win_any __attribute__((aligned(1)));
        if (c + E <= cols) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = row0 + rgrp * 4 + r;
                const win v = *reinterpret_cast<const win_any*>(in + (row < rows ? row : rows - 1) * cols + c);
#pragma unroll
                for (int q = 0; q < E / 4; ++q) w[r][q] = v[q];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = row0 + rgrp * 4 + r;
                const uint8_t* p = in + (row < rows ? row : rows - 1) * cols;
#pragma unroll
                for (int q = 0; q < E / 4; ++q) w[r][q] = 0;
#pragma unroll
                for (int e = 0; e < E; ++e) w[r][e >> 2] |= (uint32_t)p[c + e < cols ? c + e : cols - 1] << (8 * (e & 3));
            }
        }
        deposit_block<E>(tile, w, cgrp, rgrp);
        __syncthreads();
        emit_columns<E>(tile, out, rows, cols, row0, col0);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------------------
// Current scaling of a small tensor in one launch: one workgroup holds all of it in registers, takes the amax, decides
// on the scale (with everything the amax-only launch books: history, first use) and casts.  The two launches this
// replaces cost their latency twice (fp32 128 x 128 with its transposed copy 4.9 + 3.7 us, and another 3 us of host
// time); one workgroup is slower than the chip from about kOnceMax elements on.  With a transposed copy the bytes pass
// through LDS, one word of padding per row, and leave as words of four rows.
constexpr int kOnceGroups = 4;
constexpr int64_t kOnceMax = (int64_t)kOnceGroups * kFlatThreads * kVec;   // 65536 elements
template <typename S, int F, bool kT>
__global__ __launch_bounds__(kFlatThreads) void quant_once_kernel(const typename ElemOf<S>::type* __restrict__ x, int rows, int cols,
                                                              uint8_t* __restrict__ out, uint8_t* __restrict__ out_t, ScalarIO io) {
    typedef Src<S> L;
    __shared__ uint32_t s_part[kFlatThreads / 64];
    __shared__ float s_scale;
    __shared__ __attribute__((aligned(16))) uint32_t tile[kT ? kOnceMax / 4 + kOnceMax / 16 : 1];
    const int n = rows * cols, n_vec = n / kVec, t = threadIdx.x;
    const EpiloguePrefetch pre = prefetch_epilogue(io, kModeAmaxOnly);
    float v[kOnceGroups][kVec];
    uint32_t m[kOnceGroups] = {0, 0, 0, 0}, mt = 0;
    float tail = 0.0f;
#pragma unroll
    for (int i = 0; i < kOnceGroups; ++i)
        if (t + i * kFlatThreads < n_vec) L::template load<kVec, false>(x + (t + i * kFlatThreads) * kVec, v[i], m[i]);
    const int j = n_vec * kVec + t;
    if (j < n) tail = L::load1(x + j, mt);
    uint32_t mr = mt;
#pragma unroll
    for (int i = 0; i < kOnceGroups; ++i) mr = m[i] > mr ? m[i] : mr;
    const uint32_t wm = wave_max_u32(mr);
    if ((t & 63) == 0) s_part[t >> 6] = wm;
    __syncthreads();
    if (t < 64) {
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < kFlatThreads / 64; ++i) bits = s_part[i] > bits ? s_part[i] : bits;
        bits = L::to_f32_bits(bits);
        if (bits > kInfBits) bits = kNanBits;
        const float used = bookkeep(bits, io, kModeAmaxOnly, pre);
        if (t == 0) s_scale = used;
    }
    __syncthreads();
    const float scale = s_scale;
    const bool degen = degenerate_scale(scale);
    const int pitch = cols / 4 + 1;   // words
#pragma unroll
    for (int i = 0; i < kOnceGroups; ++i) {
        const int g = t + i * kFlatThreads;
        if (g >= n_vec) break;
        const u4 q = encode16<F>(v[i], scale, degen || L::has_nan(m[i]));
        *reinterpret_cast<u4*>(out + g * kVec) = q;
        if constexpr (kT) {   // (cols is a multiple of 16: a group lies in one row)
            const int r = g * kVec / cols, c = g * kVec % cols;
            uint32_t* p = tile + r * pitch + c / 4;
            p[0] = q.x, p[1] = q.y, p[2] = q.z, p[3] = q.w;
        }
    }
    if (j < n) out[j] = encode1<F>(tail, scale);
    if constexpr (kT) {
        __syncthreads();
        const int quads = rows / 4;   // rows is a multiple of 4
        for (int b = t; b < quads * (cols / 4); b += kFlatThreads) {
            const int r = b % quads, c = b / quads;
            const uint32_t* p = tile + 4 * r * pitch + c;
            const uint32_t w0 = p[0], w1 = p[pitch], w2 = p[2 * pitch], w3 = p[3 * pitch];
            const uint32_t lo01 = __builtin_amdgcn_perm(w1, w0, 0x05010400u), lo23 = __builtin_amdgcn_perm(w3, w2, 0x05010400u);
            const uint32_t hi01 = __builtin_amdgcn_perm(w1, w0, 0x07030602u), hi23 = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
            uint32_t* o = reinterpret_cast<uint32_t*>(out_t) + c * 4 * quads + r;
            o[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
            o[quads] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
            o[2 * quads] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
            o[3 * quads] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Column sums in fp32 (the bias gradient: the output gradient summed over the tokens), rounded once to the output type.
// HBM-bound on large tensors, latency-bound on small ones.  A workgroup sums a run of rows of 64 columns, 16 threads of
// 4 columns side by side and 16 rows of them; the runs of one column block are put together by the workgroup that
// arrives last, in order, so the result does not depend on timing.  Partial sums and tickets go through device-scope
// accesses, as the reductions above.
template <int OUT>
__device__ __forceinline__ void store_dequant1(void* __restrict__ out, int64_t j, float v);
constexpr int kSumCols = 64, kSumTickets = NTFP8_WORKSPACE_BYTES / 4;
template <typename S, bool kVec4>
__global__ __launch_bounds__(kThreads) void column_sum_kernel(const typename ElemOf<S>::type* __restrict__ x, int64_t rows, int64_t cols,
                                                          int64_t run, void* __restrict__ out, int out_dtype,
                                                          float* __restrict__ partial, uint32_t* __restrict__ tickets) {
    typedef Src<S> L;
    __shared__ float part[16][kSumCols];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int64_t c = (int64_t)blockIdx.x * kSumCols + tx * 4;
    const int64_t r0 = blockIdx.y * run, r1 = min(r0 + run, rows);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    auto row = [&](int64_t r, float (&v)[4]) {
        uint32_t m;
        if constexpr (kVec4) {
            if (c < cols) L::template load<4, false>(x + r * cols + c, v, m);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = L::load1(x + r * cols + (c + e < cols ? c + e : cols - 1), m);
        }
    };
    int64_t r = r0 + ty;
    for (; r + 48 < r1; r += 64) {
        float v[4][4] = {};
#pragma unroll
        for (int u = 0; u < 4; ++u) row(r + 16 * u, v[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += v[u][e];
    }
    for (; r < r1; r += 16) {
        float v[4] = {};
        row(r, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += v[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) part[ty][tx * 4 + e] = s[e];
    __syncthreads();
    if (threadIdx.x >= 64) return;
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) total += part[i][threadIdx.x];
    const int64_t col = (int64_t)blockIdx.x * kSumCols + threadIdx.x;
    if (gridDim.y > 1) {
        if (col < cols) __hip_atomic_store(partial + blockIdx.y * cols + col, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's sums are in place before its ticket is drawn
        uint32_t ticket = 0;
        if (threadIdx.x == 0) ticket = __hip_atomic_fetch_add(tickets + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(ticket) != gridDim.y - 1) return;
        if (threadIdx.x == 0) __hip_atomic_store(tickets + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        total = 0.0f;
        const int64_t at = col < cols ? col : cols - 1;
        for (uint32_t y0 = 0; y0 < gridDim.y; y0 += 16) {   // 16 requested before the first is needed
            float p[16];
#pragma unroll
            for (uint32_t y = 0; y < 16; ++y)
                p[y] = __hip_atomic_load(partial + min(y0 + y, gridDim.y - 1) * cols + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (uint32_t y = 0; y < 16; ++y)
                if (y0 + y < gridDim.y) total += p[y];
        }
    }
    if (col >= cols) return;
    if (out_dtype == NTFP8_F32) store_dequant1<NTFP8_F32>(out, col, total);
    else if (out_dtype == NTFP8_F16) store_dequant1<NTFP8_F16>(out, col, total);
    else store_dequant1<NTFP8_BF16>(out, col, total);
}

// ---------------------------------------------------------------------------------------------
// Dequantise: out = out_dtype(decode(byte) * (1 / scale)).
template <int F>
__device__ __forceinline__ float decode1(uint32_t b) {
    if constexpr (F == kE4M3) return __builtin_amdgcn_cvt_f32_fp8((int)b, 0);
    else return __builtin_amdgcn_cvt_f32_bf8((int)b, 0);
}

// fp32 value -> one output element of type OUT, as dequantised.  The fp32 product is kept a value of its own: folded into
// a mixed-precision fma (x*y + 0) the conversion would turn -0 into +0.
template <int OUT>
__device__ __forceinline__ void store_dequant1(void* __restrict__ out, int64_t j, float v) {
    asm volatile("" : "+v"(v));
    if constexpr (OUT == NTFP8_F32) ((float*)out)[j] = v;
    else if constexpr (OUT == NTFP8_F16) ((__half*)out)[j] = __float2half_rn(v);
    else {
        // bf16 round-to-nearest-even with NaN kept quiet
        uint32_t u = __float_as_uint(v);
        uint16_t r;
        if ((u & 0x7fffffffu) > kInfBits) r = (uint16_t)((u >> 16) | 0x40u);
        else r = (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
        ((uint16_t*)out)[j] = r;
    }
}
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){a, b}, v2bf));
}
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    asm volatile("" : "+v"(a), "+v"(b));   // (no mixed-precision fma, as above)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){a, b}, v2h));
}
// the two low or the two high fp8 codes of a word -> fp32
template <int F, bool kHigh>
__device__ __forceinline__ void decode2(uint32_t w, float& a, float& b) {
    if constexpr (F == kE4M3) {
        const auto p = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, kHigh);
        a = p[0], b = p[1];
    } else {
        const auto p = __builtin_amdgcn_cvt_pk_f32_bf8((int)w, kHigh);
        a = p[0], b = p[1];
    }
}

// HBM-bound.  A lane writes 16 bytes per group (8 16-bit or 4 fp32 elements, read as 8 or 4 bytes), so that a wave's
// loads and stores each cover one contiguous piece, and has kUnroll groups in flight.  Loads go through the caches (the
// bytes were usually written by the kernel before), stores are streaming.  bf16, 4096 x 4096 (50.3 MB): 15.5 us with one
// byte per lane and trip, 8.1 us (6.2 TB/s) now; streaming loads as well 9.4 us, ordinary stores 9.0 us, one group per
// trip 9.3 us.  kUnroll: groups a thread has in flight; one where that still is no more than eight workgroups per CU (us, one
// / four: 16-bit of 2^18 to 2^20 elements 3.04 / 3.11, 2^21 to 2^22 3.7 / 3.8, 2^23 to 2^24 6.5 / 6.0; fp32 of 2^19 to 2^21
// 3.55 / 3.60, 2^22 to 2^23 6.8 / 6.0).
// `is_inverse`: scale_ptr holds 1 / scale already (the form tex.cast_from_fp8 is handed, src/nanotron/fp8/tensor.py:74)
template <int F, int OUT, int kUnroll>
__global__ __launch_bounds__(kThreads) void dequant_kernel(const uint8_t* __restrict__ in, int64_t n_vec, int64_t n,
                                                           const float* __restrict__ scale_ptr, void* __restrict__ out,
                                                           int is_inverse) {
    constexpr int kE = OUT == NTFP8_F32 ? 4 : 8;   // elements per group
    typedef uint32_t win __attribute__((ext_vector_type(kE / 4)));
    typedef win win_any __attribute__((aligned(1)));   // the input may start anywhere
    const float inv = is_inverse ? *scale_ptr : 1.0f / *scale_ptr;
    const int64_t stride = (int64_t)gridDim.x * (kThreads * kUnroll);
    for (int64_t i = (int64_t)blockIdx.x * (kThreads * kUnroll) + threadIdx.x; i < n_vec; i += stride) {
        win w[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
            if (i + u * kThreads < n_vec) w[u] = *reinterpret_cast<const win_any*>(in + (i + u * kThreads) * kE);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (i + u * kThreads >= n_vec) break;
            float v[kE];
#pragma unroll
            for (int h = 0; h < kE / 4; ++h) {
                decode2<F, false>(w[u][h], v[4 * h], v[4 * h + 1]);
                decode2<F, true>(w[u][h], v[4 * h + 2], v[4 * h + 3]);
            }
#pragma unroll
            for (int e = 0; e < kE; ++e) v[e] *= inv;
            u4 o;
            if constexpr (OUT == NTFP8_F32) o = (u4){__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
            else if constexpr (OUT == NTFP8_F16) o = (u4){pack_f16(v[0], v[1]), pack_f16(v[2], v[3]), pack_f16(v[4], v[5]), pack_f16(v[6], v[7])};
            else o = (u4){pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
            __builtin_nontemporal_store(o, reinterpret_cast<u4*>(out) + i + u * kThreads);
        }
    }
    // elements past the last group (all of them when the output is not 16-byte aligned)
    for (int64_t j = n_vec * kE + (int64_t)blockIdx.x * kThreads + threadIdx.x; j < n; j += (int64_t)gridDim.x * kThreads)
        store_dequant1<OUT>(out, j, decode1<F>(in[j]) * inv);
}

// ---------------------------------------------------------------------------------------------
// Bandwidth yardsticks: the access pattern of the flat quantise kernel (one 1024-thread workgroup per CU, two spans of
// 16 bf16 elements per lane in flight, 16-byte streaming loads side by side) with the arithmetic and the reduction taken
// out.  kProbeRead: 32 bytes read per lane and span, nothing written.  kProbeHalf: 32 bytes read, 16 written (the traffic of
// a bf16 -> fp8 cast).  kProbeCopy: 32 read, 32 written.
enum ProbeMode { kProbeRead = NTFP8_PROBE_READ, kProbeHalf = NTFP8_PROBE_HALF, kProbeCopy = NTFP8_PROBE_COPY };
template <int MODE>
__global__ __launch_bounds__(kFlatThreads) void stream_probe_kernel(const u4* __restrict__ src, int64_t n_vec, u4* __restrict__ dst) {
    const int64_t stride = (int64_t)gridDim.x * kFlatThreads;
    int64_t i = (int64_t)blockIdx.x * kFlatThreads + threadIdx.x;
    u4 seen = {0u, 0u, 0u, 0u};
    auto one = [&](int64_t k) {
        const int64_t span = k / kFlatThreads;
        const bool whole = (span + 1) * kFlatThreads <= n_vec;
        const int64_t ka = whole ? 2 * span * kFlatThreads + threadIdx.x : 2 * k, kb = whole ? ka + kFlatThreads : ka + 1;
        const u4 a = __builtin_nontemporal_load(src + ka), b = __builtin_nontemporal_load(src + kb);
        if constexpr (MODE == kProbeRead) seen = seen | (a ^ b);
        else if constexpr (MODE == kProbeHalf) __builtin_nontemporal_store(a ^ b, dst + k);
        else {
            __builtin_nontemporal_store(a, dst + ka);
            __builtin_nontemporal_store(b, dst + kb);
        }
    };
    for (; i + stride < n_vec; i += 2 * stride) {
        one(i);
        one(i + stride);
    }
    if (i < n_vec) one(i);
    if constexpr (MODE == kProbeRead) {
        // keeps the loads alive; a word of dst is written only if every bit of some lane's xor came out set
        if ((seen.x & seen.y & seen.z & seen.w) == 0xffffffffu) reinterpret_cast<uint32_t*>(dst)[0] = 1u;
    }
}

__global__ void update_scale_kernel(const float* amax, const float* old_scale, int fmt, int margin, float* out,
                                    int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = update_scale(amax[i], old_scale[i], fmt, margin);
}

// ---------------------------------------------------------------------------------------------
// Host-side launchers.
// blocks for `work_items` thread-steps with `threads` per block, at most `per_cu_blocks` per CU
static int grid_for(int64_t work_items, int threads = kThreads, int per_cu_blocks = 8) {
    int64_t want = (work_items + threads - 1) / threads;
    int64_t cap = (int64_t)cu_count() * per_cu_blocks;   // (one per CU for whatever takes a maximum: fewer than kCells)
    if (want < 1) want = 1;
    return (int)(want < cap ? want : cap);
}

// The launch macro reports through the thread's last-error slot.  hipGetLastError() reads and clears it; an error
// left there by an unrelated earlier call of this thread is dropped by clear_stale_error() before a launch, so that
// check_launch() speaks for this library's launch only.
static void clear_stale_error() { (void)hipGetLastError(); }
static int check_launch() { return hipGetLastError() == hipSuccess ? NTFP8_OK : NTFP8_ERR_LAUNCH; }

// Workgroups of the flat kernels: two spans each until there is one workgroup per CU; for a tensor by itself one span each as
// long as there are CUs for that.
template <typename S>
static int flat_grid(int64_t n_vec, int64_t n, bool alone = false) {
    if (n_vec == 0) return grid_for(n, kFlatThreads, 1);
    const int64_t spans = (n_vec + kSpan<S> - 1) / kSpan<S>, cus = cu_count();
    return (int)(alone && spans <= cus ? spans : std::min((spans + 1) / 2, cus));
}

// A chunk for every thread where that is no more than a workgroup per CU.  us, spans / chunks: bf16 16 x 4096 cast 2.9 / 2.4, delayed
// step 5.2 / 4.0; 1024 x 2048 3.6 / 2.9 and 6.2 / 5.2; fp32 512 x 1024 3.6 / 2.4 and 6.7 / 4.7, current scaling 8.9 / 7.0.  Beyond,
// one span a workgroup instead of two: bf16 2048 x 2048 delayed step 6.7 / 6.0, fp32 7.8 / 7.1.
template <typename S, int F, bool kOne>
static int launch_flat_grid(int grid, int mode, const typename ElemOf<S>::type* x, int64_t n_vec, int64_t n, uint8_t* out, const float* scale_ptr,
                            Workspace* ws, const ScalarIO& io, hipStream_t st) {
#define NT_FLAT(M) hipLaunchKernelGGL((quant_flat_kernel<S, F, M, kOne>), dim3(grid), dim3(kFlatThreads), 0, st, x, n_vec, n, out, scale_ptr, ws, io)
    if (mode == kModeAmaxOnly) NT_FLAT(kModeAmaxOnly);
    else if (mode == kModeCastOnly) NT_FLAT(kModeCastOnly);
    else NT_FLAT(kModeDelayed);
#undef NT_FLAT
    return check_launch();
}
template <typename S, int F>
static int launch_flat(int mode, const void* x, int64_t n, bool vec_ok, uint8_t* out, const float* scale_ptr,
                       Workspace* ws, const ScalarIO& io, hipStream_t st) {
    const int64_t n_vec = vec_ok ? n / kChunk<S> : 0;
    const typename ElemOf<S>::type* xp = static_cast<const typename ElemOf<S>::type*>(x);
    if (n_vec > 0 && n_vec <= (int64_t)cu_count() * kFlatThreads)
        return launch_flat_grid<S, F, true>(grid_for(n_vec, kFlatThreads, 1), mode, xp, n_vec, n, out, scale_ptr, ws, io, st);
    return launch_flat_grid<S, F, false>(flat_grid<S>(n_vec, n, true), mode, xp, n_vec, n, out, scale_ptr, ws, io, st);
}

// Columns per thread (16: 128-wide tiles, 4: 64-wide) of the kernels that turn tiles around, and their tile count: 128-wide
// from `from` of them on, in eighths of the CUs.  us, 128 / 64 wide:
//   delayed step with copy (5 eighths: from there on 64-wide tiles are more workgroups than have a word each, reduce.h),
//     bf16, 128 to 159 tiles 7.8 / 8.7, 160 to 191 8.2 / 9.6, 224 to 255 8.4 / 10.8; fp32 9.5 / 9.3, 9.9 / 10.4, 10.9 / 13.3
//   cast with copy (7 eighths), bf16, 160 to 191 tiles 5.8 / 5.5, 192 to 223 5.8 / 5.9, 224 to 255 6.2 / 6.3; fp32 6.3 / 5.9,
//     6.3 / 6.4, 6.6 / 6.9; rows of any alignment 7.3 / 6.6, 7.3 / 7.2, 7.6 / 7.8
//   transpose (8) of 4096 x 4096 bytes 6.0 / 9.2
static int tile_edge(int64_t rows, int64_t cols, int cus, int from, int64_t* tiles) {
    const int64_t t128 = ((rows + 127) / 128) * ((cols + 127) / 128);
    if (8 * t128 >= (int64_t)from * cus) {
        *tiles = t128;
        return 16;
    }
    *tiles = ((rows + 63) / 64) * ((cols + 63) / 64);
    return 4;
}

template <typename S, int F, bool kAmax>
static int launch_transpose(const void* x, int64_t rows, int64_t cols, uint8_t* out, uint8_t* out_t, const float* scale_ptr,
                            Workspace* ws, const ScalarIO& io, hipStream_t st) {
    typedef typename ElemOf<S>::type E;
    const E* xp = static_cast<const E*>(x);
    // One element per thread up to where tiles are faster.  us, tiles / small kernel, 16-bit: cast of 2^17 to 2^17.5 elements
    // 4.1 / 3.6, to 2^18 4.1 / 3.9, to 2^18.5 4.2 / 4.4; delayed step up to 2^17 6.1 / 5.4, beyond (more workgroups than
    // have a word each, reduce.h) 6.1 / 7.0.
    if (rows * cols <= (kAmax ? (int64_t)kCells * kThreads : 3 << 16)) {
        const int grid = (int)((rows * cols + kThreads - 1) / kThreads);
        hipLaunchKernelGGL((quant_transpose_small_kernel<S, F, kAmax>), dim3(grid), dim3(kThreads), 0, st, xp, (int)rows, (int)cols, out, out_t,
                           scale_ptr, ws, io);
        return check_launch();
    }
    int64_t tiles;
    const int cus = cu_count();
    const int e = tile_edge(rows, cols, cus, kAmax ? 5 : 7, &tiles);
    // (kAmax: no more workgroups than have a word each; with three per CU and tickets bf16 of 1024 tiles took 25.4 us
    // instead of 24.2, fp32 of 512 24.6 instead of 23.6)
    const int64_t cap = kAmax ? std::min<int64_t>(2 * cus, kCells) : 8 * cus;
    const int grid = (int)(tiles < cap ? tiles : cap);
    // Streaming loads where rows start on lines.  us, one row of 16 elements per thread and load / whole lines, streaming: cast
    // with copy bf16 4096 x 4096 15.9 / 14.7, fp32 22.2 / 19.9, 11008 x 4096 54.0 / 50.3; delayed step bf16 18.5 / 16.6, fp32
    // 11008 x 4096 57.8 / 53.5.  Rows that start anywhere: bf16 4095 x 4097 whole lines, streaming 30.7, ordinary 29.2.
    constexpr bool kSmall = kAmax && sizeof(E) == 2;
    const bool lines = cols * (int64_t)sizeof(E) % 128 == 0 && (reinterpret_cast<uintptr_t>(x) & 127) == 0;
    if (e == 16 && lines)
        hipLaunchKernelGGL((quant_transpose_kernel<S, F, kAmax, 16, true>), dim3(grid), dim3(kTileThreads), 0, st, xp, rows, cols, out,
                           out_t, scale_ptr, ws, io);
    else if (e == 16)
        hipLaunchKernelGGL((quant_transpose_kernel<S, F, kAmax, 16, false>), dim3(grid), dim3(kTileThreads), 0, st, xp, rows, cols, out,
                           out_t, scale_ptr, ws, io);
    else
        hipLaunchKernelGGL((quant_transpose_kernel<S, F, kAmax, 4, kSmall>), dim3(grid), dim3(kTileThreads), 0, st, xp, rows, cols, out,
                           out_t, scale_ptr, ws, io);
    return check_launch();
}

template <typename S>
static int dispatch_fmt_flat(int fmt, int mode, const void* x, int64_t n, bool vec_ok, uint8_t* out,
                             const float* scale_ptr, Workspace* ws, const ScalarIO& io, hipStream_t st) {
    return fmt == kE4M3 ? launch_flat<S, kE4M3>(mode, x, n, vec_ok, out, scale_ptr, ws, io, st)
                        : launch_flat<S, kE5M2>(mode, x, n, vec_ok, out, scale_ptr, ws, io, st);
}

template <typename S>
static int dispatch_fmt_tr(int fmt, bool with_amax, const void* x, int64_t rows, int64_t cols, uint8_t* out, uint8_t* out_t,
                           const float* scale_ptr, Workspace* ws, const ScalarIO& io, hipStream_t st) {
    if (fmt == kE4M3)
        return with_amax ? launch_transpose<S, kE4M3, true>(x, rows, cols, out, out_t, scale_ptr, ws, io, st)
                         : launch_transpose<S, kE4M3, false>(x, rows, cols, out, out_t, scale_ptr, ws, io, st);
    return with_amax ? launch_transpose<S, kE5M2, true>(x, rows, cols, out, out_t, scale_ptr, ws, io, st)
                     : launch_transpose<S, kE5M2, false>(x, rows, cols, out, out_t, scale_ptr, ws, io, st);
}

static bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

int run_quant(int mode, const void* x, int x_dtype, int64_t rows, int64_t cols, int fmt, uint8_t* out, uint8_t* out_t,
              const float* scale_ptr, Workspace* ws, const ScalarIO& io, hipStream_t st);

template <typename S>
static void launch_once(int fmt, const void* x, int rows, int cols, uint8_t* out, uint8_t* out_t, const ScalarIO& io, hipStream_t st) {
    const typename ElemOf<S>::type* xp = static_cast<const typename ElemOf<S>::type*>(x);
#define NT_ONCE(F, T) hipLaunchKernelGGL((quant_once_kernel<S, F, T>), dim3(1), dim3(kFlatThreads), 0, st, xp, rows, cols, out, out_t, io)
    if (fmt == kE4M3) {
        if (out_t) NT_ONCE(kE4M3, true);
        else NT_ONCE(kE4M3, false);
    } else {
        if (out_t) NT_ONCE(kE5M2, true);
        else NT_ONCE(kE5M2, false);
    }
#undef NT_ONCE
}

// Current scaling (or a role's first use): amax, scale, cast.  One launch of one workgroup for small tensors, two launches
// otherwise.
int run_quant_current(const void* x, int x_dtype, int64_t rows, int64_t cols, int fmt, uint8_t* out, uint8_t* out_t, Workspace* ws,
                      const ScalarIO& io, hipStream_t st) {
    const int64_t n = rows * cols;
    if (n <= kOnceMax && out && aligned(x, 16) && aligned(out, 16) &&
        (!out_t || (cols % kVec == 0 && rows % 4 == 0 && aligned(out_t, 4)))) {
        clear_stale_error();
        switch (x_dtype) {
            case NTFP8_F32: launch_once<float>(fmt, x, (int)rows, (int)cols, out, out_t, io, st); break;
            case NTFP8_F16: launch_once<f16_tag>(fmt, x, (int)rows, (int)cols, out, out_t, io, st); break;
            default: launch_once<bf16_tag>(fmt, x, (int)rows, (int)cols, out, out_t, io, st); break;
        }
        return check_launch();
    }
    const int rc = run_quant(kModeAmaxOnly, x, x_dtype, n, 1, fmt, nullptr, nullptr, nullptr, ws, io, st);
    if (rc != NTFP8_OK) return rc;
    const ScalarIO none = {nullptr, nullptr, nullptr, nullptr, nullptr, 0, fmt, 0};
    return run_quant(kModeCastOnly, x, x_dtype, rows, cols, fmt, out, out_t, io.scale_out, nullptr, none, st);
}

// row runs of a column sum: about two workgroups per CU, no run shorter than 64 rows
int column_sum_runs(int64_t rows, int64_t cols) {
    const int64_t blocks = (cols + kSumCols - 1) / kSumCols;
    if (blocks > kSumTickets) return 1;
    int64_t runs = 2 * (int64_t)cu_count() / blocks;
    if (runs > (rows + 63) / 64) runs = (rows + 63) / 64;
    return (int)(runs < 1 ? 1 : runs > 64 ? 64 : runs);
}

int run_column_sum(const void* x, int x_dtype, int64_t rows, int64_t cols, void* out, int out_dtype, float* partial, void* ws, hipStream_t st) {
    clear_stale_error();
    const int runs = column_sum_runs(rows, cols);
    const int64_t blocks = (cols + kSumCols - 1) / kSumCols;
    if (blocks > 0x7fffffff) return NTFP8_ERR_SIZE;
    const int64_t run = ((rows + runs - 1) / runs + 15) / 16 * 16;
    const dim3 grid((unsigned)blocks, (unsigned)((rows + run - 1) / run));
    uint32_t* tk = static_cast<uint32_t*>(ws);
#define NT_SUM(S) \
    if (cols % 4 == 0) hipLaunchKernelGGL((column_sum_kernel<S, true>), grid, dim3(kThreads), 0, st, static_cast<const ElemOf<S>::type*>(x), rows, cols, run, out, out_dtype, partial, tk); \
    else hipLaunchKernelGGL((column_sum_kernel<S, false>), grid, dim3(kThreads), 0, st, static_cast<const ElemOf<S>::type*>(x), rows, cols, run, out, out_dtype, partial, tk)
    if (x_dtype == NTFP8_F32) { NT_SUM(float); }
    else if (x_dtype == NTFP8_F16) { NT_SUM(f16_tag); }
    else { NT_SUM(bf16_tag); }
#undef NT_SUM
    return check_launch();
}

// mode: kModeAmaxOnly / kModeCastOnly / kModeDelayed.  out_t may be NULL.
int run_quant(int mode, const void* x, int x_dtype, int64_t rows, int64_t cols, int fmt, uint8_t* out, uint8_t* out_t,
              const float* scale_ptr, Workspace* ws, const ScalarIO& io, hipStream_t st) {
    clear_stale_error();
    const int64_t n = rows * cols;
    if (mode != kModeAmaxOnly && out_t != nullptr) {
        const bool with_amax = mode == kModeDelayed;
        switch (x_dtype) {
            case NTFP8_F32: return dispatch_fmt_tr<float>(fmt, with_amax, x, rows, cols, out, out_t, scale_ptr, ws, io, st);
            case NTFP8_F16: return dispatch_fmt_tr<f16_tag>(fmt, with_amax, x, rows, cols, out, out_t, scale_ptr, ws, io, st);
            default: return dispatch_fmt_tr<bf16_tag>(fmt, with_amax, x, rows, cols, out, out_t, scale_ptr, ws, io, st);
        }
    }
    const bool vec_ok = aligned(x, 16) && (mode == kModeAmaxOnly || aligned(out, 16));
    switch (x_dtype) {
        case NTFP8_F32: return dispatch_fmt_flat<float>(fmt, mode, x, n, vec_ok, out, scale_ptr, ws, io, st);
        case NTFP8_F16: return dispatch_fmt_flat<f16_tag>(fmt, mode, x, n, vec_ok, out, scale_ptr, ws, io, st);
        default: return dispatch_fmt_flat<bf16_tag>(fmt, mode, x, n, vec_ok, out, scale_ptr, ws, io, st);
    }
}

template <typename S, int F>
static int launch_flat_multi(const QuantDesc* const* q, int count, hipStream_t st) {
    clear_stale_error();
    MultiQuant Q = {};
    Q.count = count;
    int blocks = 0;
    for (int i = 0; i < count; ++i) {
        const QuantDesc& d = *q[i];
        const int64_t n = d.rows * d.cols;
        const bool vec_ok = aligned(d.x, 16) && aligned(d.out, 16);
        MultiQuant::Tensor& T = Q.t[i];
        T.x = d.x;
        T.out = static_cast<uint8_t*>(d.out);
        T.n = n;
        T.n_vec = vec_ok ? n / kChunk<S> : 0;
        T.ws = static_cast<Workspace*>(d.ws);
        T.io = d.io;
        T.first_block = blocks;
        T.blocks = flat_grid<S>(T.n_vec, n);
        blocks += T.blocks;
    }
    hipLaunchKernelGGL((quant_flat_multi_kernel<S, F>), dim3(blocks), dim3(kFlatThreads), 0, st, Q);
    return check_launch();
}

template <typename S>
static int dispatch_flat_multi(int fmt, const QuantDesc* const* q, int count, hipStream_t st) {
    return fmt == kE4M3 ? launch_flat_multi<S, kE4M3>(q, count, st) : launch_flat_multi<S, kE5M2>(q, count, st);
}

// The fused delayed-scaling step of several tensors.  Tensors without a transposed copy that share source type and
// format go out together, up to kMaxMulti per launch; the others one by one.
int run_quant_delayed_batch(const QuantDesc* q, int count, hipStream_t st) {
    bool done[NTFP8_MAX_BATCH] = {false};
    for (int i = 0; i < count; ++i) {
        if (done[i]) continue;
        done[i] = true;
        if (q[i].out_t != nullptr || q[i].out == nullptr) {
            const int rc = run_quant(kModeDelayed, q[i].x, q[i].x_dtype, q[i].rows, q[i].cols, q[i].fmt,
                                     static_cast<uint8_t*>(q[i].out), static_cast<uint8_t*>(q[i].out_t), q[i].io.scale_state,
                                     static_cast<Workspace*>(q[i].ws), q[i].io, st);
            if (rc != NTFP8_OK) return rc;
            continue;
        }
        const QuantDesc* group[kMaxMulti];
        int cnt = 0;
        group[cnt++] = &q[i];
        for (int j = i + 1; j < count && cnt < kMaxMulti; ++j)
            if (!done[j] && q[j].out_t == nullptr && q[j].out != nullptr && q[j].x_dtype == q[i].x_dtype && q[j].fmt == q[i].fmt) {
                group[cnt++] = &q[j];
                done[j] = true;
            }
        int rc;
        switch (q[i].x_dtype) {
            case NTFP8_F32: rc = dispatch_flat_multi<float>(q[i].fmt, group, cnt, st); break;
            case NTFP8_F16: rc = dispatch_flat_multi<f16_tag>(q[i].fmt, group, cnt, st); break;
            default: rc = dispatch_flat_multi<bf16_tag>(q[i].fmt, group, cnt, st); break;
        }
        if (rc != NTFP8_OK) return rc;
    }
    return NTFP8_OK;
}

// Both formats from one pass over x (flat layout only).
int run_quant_dual(const void* x, int x_dtype, int64_t n, uint8_t* out_e4m3, uint8_t* out_e5m2, Workspace* ws,
                   const ScalarIO& io_e4m3, const ScalarIO& io_e5m2, hipStream_t st) {
    clear_stale_error();
    const bool vec_ok = aligned(x, 16) && aligned(out_e4m3, 16) && aligned(out_e5m2, 16);
#define NT_DUAL(S) \
    do { \
        const int64_t n_vec = vec_ok ? n / kChunk<S> : 0; \
        hipLaunchKernelGGL((quant_flat_dual_kernel<S>), dim3(flat_grid<S>(n_vec, n)), dim3(kFlatThreads), 0, st, \
                           static_cast<const ElemOf<S>::type*>(x), n_vec, n, out_e4m3, out_e5m2, ws, io_e4m3, io_e5m2); \
    } while (0)
    if (x_dtype == NTFP8_F32) NT_DUAL(float);
    else if (x_dtype == NTFP8_F16) NT_DUAL(f16_tag);
    else NT_DUAL(bf16_tag);
#undef NT_DUAL
    return check_launch();
}

// ---------------------------------------------------------------------------------------------
// Reduction workspaces that live in the library's own device image, for callers that cannot allocate device
// memory (HIP graph capture, serving loops): one Workspace per tensor of a batched call.  Every GPU the library
// runs on holds its own copy of the array, at its own address, until the process ends; the name below is only a
// host-side handle of it, the address comes from hipGetSymbolAddress with that device current.
static __device__ __align__(256) unsigned char scratch[NTFP8_STATIC_MAX_TENSORS * NTFP8_WORKSPACE_BYTES];

// Device address of `scratch` on the current device, resolved at the first call for that device.  Nothing is launched:
// a device image starts with the array zeroed and every kernel leaves its workspace zero, so there is nothing to
// clear, and a clearing kernel on the first caller's stream would race with a first user on another stream.
int static_scratch(void** out, hipStream_t) {
    static std::atomic<void*> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return NTFP8_ERR_LAUNCH;
    void* p = cached[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        // (threads that race here resolve the same address)
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return NTFP8_ERR_LAUNCH;
        cached[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return NTFP8_OK;
}

// run_quant_delayed_batch with the workspaces taken from the static array (count <= NTFP8_STATIC_MAX_TENSORS)
int run_quant_delayed_batch_static(QuantDesc* q, int count, hipStream_t st) {
    void* base = nullptr;
    const int rc = static_scratch(&base, st);
    if (rc != NTFP8_OK) return rc;
    for (int i = 0; i < count; ++i) q[i].ws = static_cast<unsigned char*>(base) + (size_t)i * NTFP8_WORKSPACE_BYTES;
    return run_quant_delayed_batch(q, count, st);
}

int run_dequant(const void* in, int fmt, const float* scale, int is_inverse, int64_t n, void* out, int out_dtype,
                hipStream_t st) {
    clear_stale_error();
    const int64_t n_vec = aligned(out, 16) ? n / (out_dtype == NTFP8_F32 ? 4 : 8) : 0;
    const bool one = n_vec <= (int64_t)cu_count() * 8 * kThreads;
    const int grid = grid_for(n_vec > 0 ? (one ? n_vec : (n_vec + 3) / 4) : n, kThreads, 32);
    const uint8_t* p = static_cast<const uint8_t*>(in);
#define NT_DQ(F, O) \
    do { \
        if (one) hipLaunchKernelGGL((dequant_kernel<F, O, 1>), dim3(grid), dim3(kThreads), 0, st, p, n_vec, n, scale, out, is_inverse); \
        else hipLaunchKernelGGL((dequant_kernel<F, O, 4>), dim3(grid), dim3(kThreads), 0, st, p, n_vec, n, scale, out, is_inverse); \
    } while (0)
    if (fmt == kE4M3) {
        if (out_dtype == NTFP8_F32) NT_DQ(kE4M3, NTFP8_F32);
        else if (out_dtype == NTFP8_F16) NT_DQ(kE4M3, NTFP8_F16);
        else NT_DQ(kE4M3, NTFP8_BF16);
    } else {
        if (out_dtype == NTFP8_F32) NT_DQ(kE5M2, NTFP8_F32);
        else if (out_dtype == NTFP8_F16) NT_DQ(kE5M2, NTFP8_F16);
        else NT_DQ(kE5M2, NTFP8_BF16);
    }
#undef NT_DQ
    return check_launch();
}

int run_transpose(const void* in, int64_t rows, int64_t cols, void* out, hipStream_t st) {
    clear_stale_error();
    int64_t tiles;
    const int cus = cu_count();
    const int e = tile_edge(rows, cols, cus, 8, &tiles);
    const int64_t cap = (int64_t)cus * 8;
    const int grid = (int)(tiles < cap ? tiles : cap);
    const uint8_t* p = static_cast<const uint8_t*>(in);
    uint8_t* o = static_cast<uint8_t*>(out);
    if (e == 16) hipLaunchKernelGGL((transpose_kernel<16>), dim3(grid), dim3(kTileThreads), 0, st, p, rows, cols, o);
    else hipLaunchKernelGGL((transpose_kernel<4>), dim3(grid), dim3(kTileThreads), 0, st, p, rows, cols, o);
    return check_launch();
}

int run_stream_probe(int mode, const void* src, int64_t bytes, void* dst, hipStream_t st) {
    clear_stale_error();
    const int64_t n_vec = bytes / 32;
    const int grid = grid_for((n_vec + 1) / 2, kFlatThreads, 1);
    const u4* s = static_cast<const u4*>(src);
    u4* d = static_cast<u4*>(dst);
    if (mode == kProbeRead) hipLaunchKernelGGL((stream_probe_kernel<kProbeRead>), dim3(grid), dim3(kFlatThreads), 0, st, s, n_vec, d);
    else if (mode == kProbeHalf) hipLaunchKernelGGL((stream_probe_kernel<kProbeHalf>), dim3(grid), dim3(kFlatThreads), 0, st, s, n_vec, d);
    else hipLaunchKernelGGL((stream_probe_kernel<kProbeCopy>), dim3(grid), dim3(kFlatThreads), 0, st, s, n_vec, d);
    return check_launch();
}

int run_amax_finalize(Workspace* ws, const ScalarIO& io, hipStream_t st) {
    clear_stale_error();
    hipLaunchKernelGGL(amax_finalize_kernel, dim3(1), dim3(64), 0, st, ws, io);
    return check_launch();
}

int run_update_scale(const float* amax, const float* old_scale, int fmt, int margin, float* out, int64_t n,
                     hipStream_t st) {
    clear_stale_error();
    const int64_t blocks = (n + 255) / 256;
    if (blocks > 0x7fffffff) return NTFP8_ERR_SIZE;
    hipLaunchKernelGGL(update_scale_kernel, dim3((int)blocks), dim3(256), 0, st, amax, old_scale, fmt, margin, out, n);
    return check_launch();
}

}  // namespace ntfp8
