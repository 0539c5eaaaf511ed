// Tile size of a launch of the MFMA tile kernels (gemm_big.h, gemm_mid.h).  Host code, included by gemm.hip.
#pragma once
#include <algorithm>

namespace ntfp8 {

// operands within reach of 32-bit buffer offsets: what the 256-wide tiles and transposed operands need
inline bool fits32(const GemmDesc& g) {
    return (int64_t)(g.M + 256) * g.K < (1LL << 31) && (int64_t)(g.N + kBigN) * g.K < (1LL << 31);
}
// the 256-wide tiles' pipeline starts with two K-tiles
inline bool big_ok(const GemmDesc& g) { return fits32(g) && g.K >= 2 * kBK; }

// What a launch of one problem takes in tiles of 256 x 256, 128 x 128, 128 x 64 or 64 x 64, in nanoseconds: rounds of workgroups
// times what a workgroup takes for its K-tiles and for everything else.  The constants are fits to launches with bf16 output
// (plain / B transposed / both transposed), warm operands; what matters is where the lines cross.
//   us, 256 / 128 / 64 wide:  1024 x 1024 x 1024  10.1 / 7.5 / 4.8     2048 x 1024 x 4096  26.5 / 16.3 / 15.3
//   2048 x 2048 x 2048  16.7 / 11.8 / 16.9      both transposed  19.6 / 12.6 / 24.3
//   2048 x 4096 x 4096  32.5 / 40.4 / 55.8      4096 x 4096 x 4096  51.9 / 73.5 / 101
//   128 x 128 / 128 x 64 / 64 x 64:  2048 x 1024 x 1024 7.6 / 5.9 / 6.6, x 4096 15.6 / 12.9 / 15.2; B transposed 8.0 / 6.6 / 8.0 and
//   16.9 / 16.3 / 20.2; both transposed x 2048 12.1 / 10.4 / 13.6; 1021 x 2304 x 1024 (288 tiles of 128 x 64) 7.8 / 10.4 / 9.0
//   at equal estimates:   3696 x 1088 x 944 (bf16) 10.6 / - / 11.8     1072 x 3600 x 320 (fp8 output) 12.5 / - / 17.6
struct Edge {
    int m, n;
};
struct TileTime {   // a tile: per_k ns for a K-tile and `rest`
    int64_t per_k, rest;
    int64_t slots;   // workgroups at once
};
// `alone`: 64-wide tiles, of which no more than one goes to a CU
inline TileTime tile_time(Edge e, int form, bool alone, int64_t cus) {
    static constexpr int kAlone[3] = {185, 260, 280}, kPair[3] = {350, 530, 620};
    if (e.m == 256) return {1400, 7000, cus};
    if (e.n == 128) return {390, 5200, cus};
    if (e.m == 128) return {form ? 400 : 290, 3600, cus};
    return {alone ? kAlone[form] : kPair[form], alone ? 3000 : 3500, 2 * cus};
}
// The partial last round of 256-wide tiles is computed in parts if there is a CU for each: in how many (1: whole), unless all of
// the list in one launch ends earlier (shallow tiles beside a few deep ones).  Halves are the 256-wide kernel's own; behind full
// rounds quarters (128 x 128) and eighths (128 x 64) are quicker yet.  Backward launches with 1 to 64 tiles in the last round, us,
// halves / these: 2912 tokens, 2544 -> 3520, 77.0 / 67.1; 3152, 2464 -> 3712, 72.3 / 59.3; 1888, 3232 -> 3872, 67.8 / 63.3.
inline int tail_parts(int64_t tiles, int64_t cus) {
    const int64_t rem = tiles % cus;
    if (rem == 0 || 2 * rem > cus) return 1;
    return tiles < cus || 4 * rem > cus ? 2 : 8 * rem > cus ? 4 : 8;
}
inline TileTime tail_time(int parts, int form, int64_t cus) {
    if (parts == 2) return {700, 7000, cus};
    return tile_time(parts == 4 ? Edge{128, 128} : Edge{128, 64}, form, false, cus);
}
// (a tile's edges are powers of two)
inline int64_t tiles_of(const GemmDesc& g, Edge e) {
    return (((int64_t)g.M + e.m - 1) >> __builtin_ctz(e.m)) * (((int64_t)g.N + e.n - 1) >> __builtin_ctz(e.n));
}
inline int form_of(const GemmDesc& g) { return g.ta ? 2 : g.tb ? 1 : 0; }
inline int64_t k_tiles(const GemmDesc& g) { return (g.K + kBK - 1) / kBK; }

// A second round of 128 x 64 tiles, both operands K-contiguous: nothing of its start or of the first round's stores is hidden, the more so the
// narrower the output's rows are in a tile.  The other way there are halves of 256-wide tiles (up to 128 of them).  us, those / two rounds
// (387 to 507 tiles of 128 x 64):
//   K               256          512          1024         1536         2048         3072         4096         6144
//   16-bit       6.1 /  7.5   7.4 /  8.4   9.7 / 10.1  12.1 / 13.0  14.3 / 14.2  19.0 / 20.0  23.2 / 22.3  32.5 / 32.3
//   fp32         8.1 /  8.4   9.5 /  9.5  11.8 / 11.2  14.3 / 14.1  16.4 / 15.1  21.1 / 21.0  25.5 / 23.1  34.4 / 33.2
//   fp8          8.1 / 10.1   9.5 / 11.3  11.8 / 12.9  14.3 / 15.6  16.5 / 16.7  21.3 / 22.5  25.6 / 25.2  34.7 / 34.9
//   and copy    11.1 / 14.4  12.8 / 15.6  15.2 / 17.4  17.3 / 19.5  19.9 / 20.8  24.4 / 26.5  28.5 / 28.6  37.7 / 38.2
inline int64_t narrow_again(const GemmDesc& g) {
    return is_fp8_out(g.d_dtype) ? (g.Dt ? 3700 : 2700) : g.d_dtype == NTFP8_F32 ? 400 : 1500;
}

// *parts: of the tiles of a partial last round of 256-wide ones
inline int64_t cost_of_one(const GemmDesc& g, Edge edge, int64_t cus, int* parts) {
    const int64_t tiles = tiles_of(g, edge), k = k_tiles(g);
    const int form = form_of(g);
    TileTime whole = tile_time(edge, form, false, cus);
    // One problem on part of the CUs: the chip is clocked higher (129 to 255 tiles 950 to 1200 ns a K-tile), and the 256-wide tiles
    // are the fastest wherever 128-wide ones need more than two rounds (129 to 255 tiles, K 512 to 8192, every form, 16-bit, fp32
    // and accumulated: 1.08 to 1.95 times).  Two rounds of those are faster from a K of about 700 on, which is where the ordinary
    // price has the line: 504 of them against 132 tiles, us, 128 / 256 wide: K = 1024 bf16 14.2 / 15.9, fp32 16.5 / 19.7, both
    // transposed 18.4 / 20.2; K = 512 11.5 / 11.9, 13.6 / 15.7, 15.0 / 16.0; K = 4096 bf16 32.0 / 39.0.
    if (edge.m == 256 && tiles < cus && tiles_of(g, Edge{128, 128}) > 2 * cus) whole.per_k = 1150;
    const int64_t slots = whole.slots, rem = tiles % slots;
    auto cost = [&](int split) -> int64_t {
        const TileTime end = split > 1 ? tail_time(split, form, cus) : edge.m == 64 && rem <= cus ? tile_time(edge, form, true, cus) : whole;
        const int64_t more = edge.m == 128 && edge.n == 64 && form == 0 ? (tiles - 1) / slots * narrow_again(g) : 0;
        return tiles / slots * (whole.per_k * k + whole.rest) + (rem == 0 ? 0 : end.per_k * k + end.rest) + more;
    };
    const int64_t as_is = cost(*parts = 1);
    const int split = edge.m == 256 ? tail_parts(tiles, cus) : 1;
    if (split == 1) return as_is;
    const int64_t cut = cost(split);
    if (cut < as_is) *parts = split;
    return std::min(cut, as_is);
}

// Several problems in one launch, longest K first: when the last of the chip's eight XCDs is done.  Each works off its own share of the
// list, every round's run of tiles (run_of_xcd), in order, the next tile on the CU that is free first; the deep tiles at the head of
// the list all fall to the first XCDs, whose share of the next round waits behind them (a dgrad of 54 128-wide tiles of 25 K-tiles
// beside a wgrad of 225 tiles of 6, 768 tokens, 1056 -> 3184: 28 us, where a list that all CUs share would end after 15).
// Tile times are those of a tile among unlike ones, with their outputs: fits to 12800 drawn launches of two to four problems.
// There the choice costs 0.3 % more than the best tile size on average; by the average depth of the tiles 4.7 %, by the mean of
// that and of one list for the whole chip 1.4 %, where one launch in thirty took 1.05 to 1.6 times what it takes by the average depth.
struct ListTime {
    int64_t per_k, rest, out32, out_acc;   // ns: a K-tile, the rest, and on top of it fp32 outputs, added to what is there
};
inline ListTime list_time(Edge e, int form) {
    if (e.m == 256) return {1100, 9700, 2200, 10000};
    if (e.n == 128) return {430, 5000, 550, 2500};
    if (e.m == 128) return {form ? 400 : 290, 3600, 270, 1250};
    return {tile_time(e, form, true, 1).per_k, 1700, 140, 620};   // (alone on its CU)
}
inline ListTime list_half_time() { return {700, 7000, 1100, 5000}; }
inline int64_t takes(const ListTime& t, const GemmDesc& g) {
    return t.per_k * k_tiles(g) + t.rest + (g.accumulate ? t.out_acc : g.d_dtype == NTFP8_F32 ? t.out32 : 0);
}

// A list in one tile size: its problems, longest K first, the tiles up to the end of each and what one of them takes
struct TileList {
    int n, form;
    Edge edge;
    int64_t cus, end[kBigMaxProblems], time[kBigMaxProblems];
};
// Its first `left` tiles; any time from `limit` on where they take that long
inline int64_t list_end(const TileList& L, int64_t left, int64_t limit) {
    const bool pairs = L.edge.m == 64;   // two workgroups on a CU
    const int64_t cus_x = std::max<int64_t>(L.cus / kXcds, 1), slots = (pairs ? 2 : 1) * L.cus;
    const int64_t alone = tile_time(L.edge, L.form, true, L.cus).per_k, shared = pairs ? tile_time(L.edge, L.form, false, L.cus).per_k : alone;
    int64_t before[kBigMaxProblems] = {0}, worst = 0;
    for (int x = 0; x < kXcds; ++x) {
        // this XCD's tiles of each problem (in order: its run of a round lies behind that of the round before)
        int64_t t[kBigMaxProblems] = {0};
        for (int64_t r = 0; r < left; r += slots) {
            const int64_t in = std::min(slots, left - r);
            int64_t lo = r + x * (in / kXcds) + std::min<int64_t>(x, in % kXcds);
            const int64_t hi = lo + in / kXcds + (x < in % kXcds);
            for (int i = 0; lo < hi; ++i) {
                const int64_t c = std::min(hi, L.end[i]) - lo;
                if (c > 0) t[i] += c, lo += c;
            }
        }
        if (x > 0 && std::equal(t, t + L.n, before)) continue;
        std::copy(t, t + L.n, before);
        // groups of slots that are busy for equally long: one more for the last tiles of a problem, which do not fill a group
        struct {
            int64_t until, count;
        } at[kBigMaxProblems + 1];
        at[0] = {0, (pairs ? 2 : 1) * cus_x};
        int groups = 1;
        int64_t handed_out = 0, last = 0;   // when the last tile was, and when all of them are done
        for (int i = 0; i < L.n; ++i) {
            while (t[i] > 0) {
                int first = 0;
                for (int j = 1; j < groups; ++j)
                    if (at[j].until < at[first].until) first = j;
                handed_out = at[first].until;
                const int64_t until = handed_out + L.time[i], c = std::min(t[i], at[first].count);
                last = std::max(last, until);
                t[i] -= c;
                at[first].count -= c;
                int to = 0;
                while (to < groups && at[to].until != until) ++to;
                if (to < groups) {
                    at[to].count += c;
                    if (at[first].count == 0) at[first] = at[--groups];
                } else {
                    at[at[first].count == 0 ? first : groups++] = {until, c};
                }
            }
        }
        if (pairs) {   // slower by `shared` / `alone` until the last tile is handed out, and while there are more than CUs
            int64_t busy = 0, now = handed_out, ns = handed_out * shared;
            for (int j = 0; j < groups; ++j) busy += at[j].until > handed_out ? at[j].count : 0;
            while (now < last) {
                int64_t next = last, ends = 0;
                for (int j = 0; j < groups; ++j)
                    if (at[j].until > now) next = std::min(next, at[j].until);
                for (int j = 0; j < groups; ++j) ends += at[j].until == next ? at[j].count : 0;
                ns += (next - now) * (busy > cus_x ? shared : alone);
                now = next;
                busy -= ends;
            }
            last = ns / alone;
        }
        worst = std::max(worst, last);
        if (worst >= limit) break;
    }
    return worst;
}
inline int64_t cost_of_list(const GemmDesc* const* g, int n, const int* order, Edge edge, int64_t cus, int64_t limit, int* parts) {
    TileList L = {n, 0, edge, cus, {}, {}};
    const int64_t slots = (edge.m == 64 ? 2 : 1) * cus;
    int64_t tiles = 0, work = 0, longest = 0;
    for (int i = 0; i < n; ++i) {
        const GemmDesc& d = *g[order[i]];
        const int64_t t = tiles_of(d, edge);
        L.form = std::max(L.form, form_of(d));
        L.time[i] = takes(list_time(edge, form_of(d)), d);
        L.end[i] = tiles += t;
        work += t * L.time[i];
        longest = std::max(longest, L.time[i]);
    }
    *parts = 1;
    const int64_t rem = tiles % slots;
    const int split = edge.m == 256 ? tail_parts(tiles, cus) : 1;
    if (tiles > 64 * slots) return work / slots * (edge.m == 64 ? 2 : 1);   // (so many rounds even out)
    if (split == 1) return std::max(work / slots, longest) >= limit ? limit : list_end(L, tiles, limit);
    const int64_t as_is = list_end(L, tiles, limit);
    // the deepest tile of the last round
    int i = 0;
    while (L.end[i] <= tiles - rem) ++i;
    const GemmDesc& d = *g[order[i]];
    const ListTime part = split == 2 ? list_half_time() : list_time(split == 4 ? Edge{128, 128} : Edge{128, 64}, form_of(d));
    const int64_t cut = takes(part, d) + (tiles > rem ? list_end(L, tiles - rem, limit) : 0);
    if (cut < as_is) *parts = split;
    return std::min(cut, as_is);
}

// the problems of a list: longest K first
inline void by_depth(const GemmDesc* const* g, int n, int* order) {
    for (int i = 0; i < n; ++i) order[i] = i;
    for (int i = 1; i < n; ++i)   // insertion sort, stable, K descending
        for (int j = i; j > 0 && g[order[j]]->K > g[order[j - 1]]->K; --j) std::swap(order[j], order[j - 1]);
}

struct TileChoice {
    Edge edge;
    int parts;   // of the tiles of a partial last round of 256-wide ones
};
inline TileChoice choose_tiles(const GemmDesc* const* g, int n, int cus) {
    bool big = true;
    for (int i = 0; i < n; ++i) big = big && big_ok(*g[i]);
    int order[kBigMaxProblems];
    by_depth(g, n, order);
    int64_t best = INT64_MAX;
    auto cost_in = [&](Edge e, int* parts) { return n == 1 ? cost_of_one(*g[0], e, cus, parts) : cost_of_list(g, n, order, e, cus, best, parts); };
    TileChoice c{{128, 128}, 1};
    best = cost_in(c.edge, &c.parts);
    // (where the lines meet, the wider tiles for one problem, the narrower for several)
    const int first = n == 1 ? 256 : 64;
    for (const Edge e : {Edge{first, first}, Edge{320 - first, 320 - first}, Edge{128, 64}}) {
        if (e.m == 256 && !big) continue;
        int p;
        const int64_t cost = cost_in(e, &p);
        if (cost < best) best = cost, c = {e, p};
    }
    return c;
}

}  // namespace ntfp8
