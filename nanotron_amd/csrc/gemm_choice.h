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

// What a launch of `n` problems takes in tiles of 256 x 256, 128 x 128, 128 x 64 or 64 x 64, in nanoseconds: rounds of workgroups times what a
// workgroup takes for its K-tiles and for everything else.  The constants are fits to launches of one problem with
// bf16 output (plain / B transposed / both transposed), warm operands; what matters is where the lines cross.
//   us, 256 / 128 / 64 wide:  1024 x 1024 x 1024  10.1 / 7.5 / 4.8     2048 x 1024 x 4096  26.5 / 16.3 / 15.3
//   2048 x 2048 x 2048  16.7 / 11.8 / 16.9      both transposed  19.6 / 12.6 / 24.3
//   2048 x 4096 x 4096  32.5 / 40.4 / 55.8      4096 x 4096 x 4096  51.9 / 73.5 / 101
//   128 x 128 / 128 x 64 / 64 x 64:  2048 x 1024 x 1024 7.6 / 5.9 / 6.6, x 4096 15.6 / 12.9 / 15.2; B transposed 8.0 / 6.6 / 8.0 and
//   16.9 / 16.3 / 20.2; both transposed x 2048 12.1 / 10.4 / 13.6; 1021 x 2304 x 1024 (288 tiles of 128 x 64) 7.8 / 10.4 / 9.0
//   at equal estimates:   3696 x 1088 x 944 (bf16) 10.6 / - / 11.8     1072 x 3600 x 320 (fp8 output) 12.5 / - / 17.6,
//                         528 x 2528 x 1008 with its weight gradient 19.5 / - / 14.8
// Several problems: the mean of what their average depth gives and of the end of the list as the CUs work it off, longest tile
// first.  Over 273 drawn forward and backward launches of 256 to 4096 tokens the choice then costs 0.9 % more than the best tile
// size on average; by the average depth alone 2.6 % (a dgrad of a few deep tiles beside a wgrad of many shallow ones looks as
// if the deep ones could be shared out: 1280 tokens, 2560 -> 6912, 82 us in 256-wide tiles, 62 in 128-wide), by the end of the
// list alone 1.8 %.
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
inline int64_t tiles_of(const GemmDesc& g, Edge e) { return (((int64_t)g.M + e.m - 1) / e.m) * (((int64_t)g.N + e.n - 1) / e.n); }
inline int64_t k_tiles(const GemmDesc& g) { return (g.K + kBK - 1) / kBK; }

// When the last of `left` tiles ends, the first of the list (problems by `order`, longest K first): groups of CUs that are busy for
// equally long, the next tiles go to those that are free first.  -1: too many groups.  *next_k: depth of the tile behind them.
inline int64_t list_end(const GemmDesc* const* g, int n, const int* order, Edge edge, const TileTime& time, int64_t left, int64_t* next_k) {
    struct {
        int64_t until, count;
    } at[4 * kBigMaxProblems + 2] = {{0, time.slots}};
    int groups = 1;
    *next_k = 0;
    for (int i = 0; i < n; ++i) {
        const GemmDesc& d = *g[order[i]];
        int64_t t = tiles_of(d, edge);
        if (t > left && *next_k == 0) *next_k = k_tiles(d);
        t = std::min(t, left);
        left -= t;
        const int64_t takes = time.per_k * k_tiles(d) + time.rest;
        while (t > 0) {
            int first = 0;
            for (int j = 1; j < groups; ++j)
                if (at[j].until < at[first].until) first = j;
            const int64_t now = at[first].until, c = std::min(t, at[first].count);
            t -= c;
            at[first].count -= c;
            int to = 0;
            while (to < groups && at[to].until != now + takes) ++to;
            if (to < groups) {
                at[to].count += c;
                if (at[first].count == 0) at[first] = at[--groups];
            } else if (at[first].count == 0) {
                at[first] = {now + takes, c};
            } else if (groups < (int)(sizeof(at) / sizeof(at[0]))) {
                at[groups++] = {now + takes, c};
            } else {
                return -1;
            }
        }
    }
    int64_t busy = 0;
    for (int j = 0; j < groups; ++j) busy = std::max(busy, at[j].until);
    return busy;
}

// `order`: the problems, longest K first.  *parts: of the tiles of a partial last round of 256-wide ones
inline int64_t launch_cost(const GemmDesc* const* g, int n, const int* order, Edge edge, int64_t cus, int* parts) {
    int64_t tiles = 0, kt = 0;   // kt: summed over the tiles
    int form = 0;
    for (int i = 0; i < n; ++i) {
        const int64_t t = tiles_of(*g[i], edge);
        tiles += t;
        kt += t * k_tiles(*g[i]);
        form = g[i]->ta ? 2 : (g[i]->tb && form < 1 ? 1 : form);
    }
    const int64_t k = kt / tiles;   // K-tiles of an average tile
    TileTime whole = tile_time(edge, form, false, cus);
    const TileTime few = tile_time(edge, form, true, cus);
    // One problem on part of the CUs: the chip is clocked higher (129 to 255 tiles 950 to 1200 ns a K-tile), and the 256-wide tiles
    // are the fastest wherever 128-wide ones need more than two rounds (129 to 255 tiles, K 512 to 8192, every form, 16-bit, fp32
    // and accumulated: 1.08 to 1.95 times).  Two rounds of those are faster from a K of about 700 on, which is where the ordinary
    // price has the line: 504 of them against 132 tiles, us, 128 / 256 wide: K = 1024 bf16 14.2 / 15.9, fp32 16.5 / 19.7, both
    // transposed 18.4 / 20.2; K = 512 11.5 / 11.9, 13.6 / 15.7, 15.0 / 16.0; K = 4096 bf16 32.0 / 39.0.
    if (n == 1 && edge.m == 256 && tiles < cus && tiles_of(*g[0], Edge{128, 128}) > 2 * cus) whole.per_k = 1150;
    const int64_t slots = whole.slots, rem = tiles % slots;
    auto cost = [&](int split) -> int64_t {
        const TileTime end = split > 1 ? tail_time(split, form, cus) : edge.m == 64 && rem <= cus ? few : whole;
        const int64_t average = tiles / slots * (whole.per_k * k + whole.rest) + (rem == 0 ? 0 : end.per_k * k + end.rest);
        if (n == 1 || tiles > 64 * slots) return average;
        int64_t next_k;
        const int64_t busy = list_end(g, n, order, edge, edge.m == 64 && tiles <= cus ? few : whole, split > 1 ? tiles - rem : tiles, &next_k);
        if (busy < 0) return average;
        return (average + busy + (split > 1 ? end.per_k * next_k + end.rest : 0)) / 2;
    };
    const int64_t as_is = cost(*parts = 1);
    const int split = edge.m == 256 ? tail_parts(tiles, cus) : 1;
    if (split == 1) return as_is;
    const int64_t cut = cost(split);
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
    TileChoice c{{128, 128}, 1};
    int64_t best = launch_cost(g, n, order, c.edge, cus, &c.parts);
    // (where the lines meet, the wider tiles for one problem, the narrower for several)
    const int first = n == 1 ? 256 : 64;
    for (const Edge e : {Edge{first, first}, Edge{320 - first, 320 - first}, Edge{128, 64}}) {
        if (e.m == 256 && !big) continue;
        int p;
        const int64_t cost = launch_cost(g, n, order, e, cus, &p);
        if (cost < best) best = cost, c = {e, p};
    }
    return c;
}

}  // namespace ntfp8
