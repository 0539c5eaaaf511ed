// What follows the partial maxima of a launch: publication, arrival count, and the bookkeeping of a tensor role by the
// workgroup that arrives last.  Shared by the quantise kernels and the fp8-output GEMM epilogues.
#pragma once
#include "common.h"

namespace ntfp8 {

// ---------------------------------------------------------------------------------------------
// Block reduction of the partial max, publication, and the bookkeeping epilogue of one block.
//
// Inter-block traffic uses relaxed device-scope atomics only (they execute at the level where all XCDs agree).  In a
// quantise launch a block's maximum is one word that says by itself that it has arrived (publish_and_finalize); in a GEMM
// the wave's own memory counter orders two: the maxima of a workgroup's waves are in the slots before it draws a ticket.
// A release fence here would write back the whole L2 once per block, which costs more than the streaming pass itself.
// What the bookkeeping block's epilogue will read, requested by the first wave of every block while the
// tensor is still streaming: the history entry that moves into this lane's slot and the scale in
// force.  It takes one round trip out of the dependent chain at the end of the kernel.
struct EpiloguePrefetch {
    float hist_prev;  // hist[lane - 1] (lanes 1 .. hist_len-1; histories of up to 64 entries)
    float scale;      // *scale_state; amax-only mode: *old_scale (1.0 if there is none)
};
__device__ __forceinline__ EpiloguePrefetch prefetch_epilogue(const ScalarIO& io, int mode) {
    EpiloguePrefetch p = {0.0f, 1.0f};
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        if (io.hist && io.hist_len <= 64 && lane >= 1 && lane < io.hist_len) p.hist_prev = io.hist[lane - 1];
        if (mode != kModeAmaxOnly) p.scale = *io.scale_state;
        else if (io.old_scale) p.scale = *io.old_scale;
    }
    return p;
}

// Bookkeeping of one launch, run by one wave (lanes 0..63 of a workgroup) once every workgroup's maximum is in
// the slots: amax, history roll, next scale; leaves the workspace zeroed.  Every global access is one round
// trip for the whole wave instead of one per history entry.
//
// collect_amax: the maximum over the slots as a bit pattern (NaN patterns normalised to the quiet NaN).
__device__ inline uint32_t collect_amax(Workspace* ws) {
    const int lane = threadIdx.x;
    uint32_t bits = 0;
    if (lane < kMaxSlots) bits = __hip_atomic_load(&ws->slot[lane].bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bits = wave_max_u32(bits);
    if (bits > kInfBits) bits = kNanBits;
    return bits;
}

// bookkeep: what one tensor role learns from the amax `bits` of this launch.  Returns the scale in force.
__device__ inline float bookkeep(uint32_t bits, const ScalarIO& io, int mode, const EpiloguePrefetch& pre) {
    const int lane = threadIdx.x;
    const float a = __uint_as_float(bits);
    float used;
    if (mode == kModeAmaxOnly) {
        // (the flag and the held scale are read here, before lane 0 writes either below)
        if (io.init_flag && *io.init_flag != 0.0f) used = *io.scale_state;
        else used = update_scale(a, pre.scale, io.fmt, io.margin);
    } else {
        used = pre.scale;
    }
    uint32_t hm = bits;
    if (io.hist && io.hist_len <= 64) {
        const bool ok = lane < io.hist_len;
        const float h = lane == 0 ? a : pre.hist_prev;
        if (ok) io.hist[lane] = h;
        const uint32_t hb = wave_max_u32(ok ? (__float_as_uint(h) & 0x7fffffffu) : 0u);
        hm = hb > hm ? hb : hm;
        if (hm > kInfBits) hm = kNanBits;
    } else if (io.hist) {
        // hist[i] <- hist[i-1], hist[0] <- a; 64 entries per trip, highest chunk first so that an entry is
        // read before the chunk below overwrites it
        for (int base = ((io.hist_len - 1) / 64) * 64; base >= 0; base -= 64) {
            const int i = base + lane;
            const bool ok = i < io.hist_len;
            float h = 0.0f;
            if (ok) h = (i == 0) ? a : io.hist[i - 1];
            if (ok) io.hist[i] = h;
            const uint32_t hb = wave_max_u32(ok ? (__float_as_uint(h) & 0x7fffffffu) : 0u);
            hm = hb > hm ? hb : hm;
        }
        if (hm > kInfBits) hm = kNanBits;
    }
    if (lane == 0) {
        uint32_t out_bits = bits;
        if (io.amax_in) {   // running maximum kept by the caller (NaN patterns compare above everything)
            uint32_t prev = __float_as_uint(*io.amax_in) & 0x7fffffffu;
            if (prev > kInfBits) prev = kNanBits;
            out_bits = prev > out_bits ? prev : out_bits;
        }
        if (io.amax_out) *io.amax_out = __uint_as_float(out_bits);
        if (io.scale_out) *io.scale_out = used;
        if (io.scale_inv_out) *io.scale_inv_out = 1.0f / used;
        if (io.hist) *io.scale_state = update_scale(__uint_as_float(hm), used, io.fmt, io.margin);
        if (io.init_flag && bits != 0u && bits < kInfBits) *io.init_flag = 1.0f;
    }
    return used;
}

__device__ inline void clear_workspace(Workspace* ws) {
    const int lane = threadIdx.x;
    if (lane == 0) __hip_atomic_store(&ws->ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane < kMaxSlots) {
        __hip_atomic_store(&ws->slot[lane].bits, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ws->slot[lane].ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

__device__ inline void finalize_wave(Workspace* ws, const ScalarIO& io, int mode, const EpiloguePrefetch& pre) {
    bookkeep(collect_amax(ws), io, mode, pre);
    clear_workspace(ws);
}

// Two-level arrival count: a block publishes into the slot of its group and draws a ticket there; the last block of a
// group draws a ticket of the launch.  All blocks finish at about the same time, and their atomics on one address would
// queue one behind the other.  True for the block that arrives last; called by one thread.
__device__ __forceinline__ bool draw_ticket(Workspace* ws, uint32_t bid, uint32_t nblocks) {
    const uint32_t grp = bid % kMaxSlots;
    const uint32_t in_group = (nblocks - grp + kMaxSlots - 1) / kMaxSlots;
    const uint32_t t = __hip_atomic_fetch_add(&ws->slot[grp].ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t != in_group - 1) return false;
    const uint32_t groups = nblocks < (uint32_t)kMaxSlots ? nblocks : (uint32_t)kMaxSlots;
    return __hip_atomic_fetch_add(&ws->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == groups - 1;
}

// Quantise launches (at most kCells workgroups reduce one tensor): the workspace as one word per workgroup.  A workgroup
// stores its maximum, marked as present, and is done; the one with the highest number (dispatched last) reads the words
// until all are there.  That is one store and one read behind the last maximum, where slots and tickets need four
// dependent round trips to the memory side (maximum, ticket of the group, ticket of the launch, slots).  Bound by that
// latency on small tensors: delayed step of bf16 2048 x 2048 8.8 -> 7.3 us, 4096 x 4096 12.0 -> 10.8 us alone and 14.9 ->
// 13.4 us inside a training step.  Nobody waits for the reading wave, so every word arrives; the trip limit (many seconds)
// only keeps a workspace that two overlapping launches share against the rules from holding the GPU.
constexpr uint32_t kCells = NTFP8_WORKSPACE_BYTES / 4, kPresent = 0x80000000u;
__device__ inline uint32_t collect_cells(uint32_t own, Workspace* ws, uint32_t others) {
    uint32_t* cell = reinterpret_cast<uint32_t*>(ws);
    uint32_t best = own, trips = 1u << 25;
    for (uint32_t base = threadIdx.x; base - threadIdx.x < others; base += 256) {
        uint32_t v[4];
        for (;;) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                v[j] = kPresent;
                if (base + 64 * j < others) v[j] = __hip_atomic_load(cell + base + 64 * j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (__all((v[0] & v[1] & v[2] & v[3] & kPresent) != 0u) || --trips == 0u) break;
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t m = v[j] & ~kPresent;
            best = m > best ? m : best;
            if (base + 64 * j < others) __hip_atomic_store(cell + base + 64 * j, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (trips == 0u) trips = 1u;
    }
    best = wave_max_u32(best);
    return best > kInfBits ? kNanBits : best;
}

// `bid` of `nblocks` (at most kCells): this workgroup's place among the workgroups that reduce the same tensor (the whole
// grid, except in a launch that carries several tensors).
// `io2` / `pre2`: a second tensor role fed by the same amax (one source tensor quantised to both formats).
template <int THREADS>
__device__ inline void publish_and_finalize(uint32_t m_f32bits, Workspace* ws, const ScalarIO& io, int mode,
                                            const EpiloguePrefetch& pre, uint32_t bid = blockIdx.x,
                                            uint32_t nblocks = gridDim.x, const ScalarIO* io2 = nullptr,
                                            const EpiloguePrefetch* pre2 = nullptr) {
    __shared__ uint32_t s_part[THREADS / 64];
    const uint32_t wm = wave_max_u32(m_f32bits);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = wm;
    __syncthreads();
    if (threadIdx.x >= 64) return;   // the rest is the first wave's
    uint32_t bm = 0;
#pragma unroll
    for (int i = 0; i < THREADS / 64; ++i) bm = s_part[i] > bm ? s_part[i] : bm;
    if (bid != nblocks - 1) {
        if (threadIdx.x == 0)
            __hip_atomic_store(reinterpret_cast<uint32_t*>(ws) + bid, bm | kPresent, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    const uint32_t bits = collect_cells(bm, ws, nblocks - 1);
    bookkeep(bits, io, mode, pre);
    if (io2) bookkeep(bits, *io2, mode, *pre2);
}

}  // namespace ntfp8
