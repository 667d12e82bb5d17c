// w6a16_plan.h -- which W6A16 kernel a call runs, in what shape, and the workspace that goes with it.  Host arithmetic on the
// call's sizes alone, so that it can be carried through on the CPU at sizes no test could run.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "w6a16.h"
#include "w6a16_grid.h"

namespace w6 {

constexpr int kTileN = 128;          // columns per strip of the packed layout
constexpr int kTiles = kTileN / 16;  // 16-column tiles per strip
constexpr int kPackBytes = 6144;     // of a chunk of a strip of the packed layout
constexpr int kCounterAlign = 256;   // bytes: workspace alignment
// The arrival counters occupy a fixed region at the start of the workspace, the partials follow it.  Calls with
// different tile counts can share one workspace: the partials of one call never overlap the counters of another,
// and every call leaves the counters it used at zero.
constexpr size_t kCounterRegion = size_t(1) << 20;

// Large-M kernel: M above this, packed weights (no workspace, no split-K).
constexpr int kBigMinM = 256;
// (its loads go through raw buffers: A's batch slice and the packed weight's below 2 GB)
inline bool big_rows(const w6a16_args* a) {
    if (a->M <= kBigMinM || a->format != W6A16_FORMAT_PACKED || a->K < 64) return false;
    const int64_t a_bytes = ((int64_t)(a->M - 1) * a->a_row_stride + a->K) * 2;
    const int64_t w_bytes = ((int64_t)a->N + kTileN - 1) / kTileN * (a->K / 64) * kPackBytes;
    return a_bytes < 0x7FFFFFFF && w_bytes < 0x7FFFFFFF;
}

// What include/w6a16.h promises of the workspace for a shape and split: a fixed region of arrival counters, partial tiles of
// split_k ranges (of 16, 32 or 64 rows by 128 columns) and, above 32 rows, one float per row and chain of two chunks (one
// where a group holds one).  Callers size their workspaces by it and calls with less are refused, so it stays as it is,
// though the kernels use less: the tile kernel the counters and up to four partial tiles where it splits K over workgroups,
// the wide kernel the chains' row sums.
constexpr int kSmallM = 32, kSmallSplit = 8;  // up to these no partial tiles (planes: where the tiles are as many as CUs)
struct Layout {
    bool big, none;  // the large-M kernel; a split of 2..8 of few rows (both without a workspace)
    int m_groups, n_strips, nchains;
    size_t tiles, partial_bytes, total_bytes;
};

inline Layout layout(const w6a16_args* a, int64_t cus) {
    Layout l{};
    l.big = big_rows(a);
    l.n_strips = (int)(((int64_t)a->N + kTileN - 1) / kTileN);
    if (l.big) return l;
    const bool small = a->M <= kSmallM;
    const int rows = small ? 16 : a->M <= 64 ? 32 : 64;  // to a tile
    l.nchains = a->K / (a->group_k % 128 == 0 ? 128 : 64);
    l.m_groups = (int)(((int64_t)a->M + rows - 1) / rows);
    l.none = small && a->split_k >= 2 && a->split_k <= kSmallSplit &&
             (a->format == W6A16_FORMAT_PACKED || (int64_t)a->B * l.m_groups * l.n_strips >= cus);
    if (l.none || (small && a->split_k <= 1)) return l;
    l.tiles = (size_t)a->B * l.m_groups * l.n_strips;
    l.partial_bytes = a->split_k > 1 ? l.tiles * a->split_k * (size_t)rows * kTileN * 4 : 0;
    l.total_bytes = kCounterRegion + l.partial_bytes + (small ? 0 : (size_t)a->B * l.nchains * l.m_groups * rows * 4);
    return l;
}

// The split_k of a shape, which bounds over how many workgroups K may be split: the smallest power of two that gives every CU
// a unit (128 columns by 32 or 64 rows in half or a quarter of a CU's wavefronts; up to 32 rows 512 columns by 16), every range
// keeping a chunk or chain, then doubled while ranges keep 16 and the units one to a CU; up to 32 rows 8 where the strips are
// as many as the CUs.
inline int plan_split(int32_t B, int32_t M, int32_t N, int32_t K, int64_t cus) {
    const bool small = M <= kSmallM;
    const int rows = small ? 16 : M <= 64 ? 32 : 64;
    const int64_t strips = ((int64_t)N + kTileN - 1) / kTileN, tiles = B * (((int64_t)M + rows - 1) / rows) * strips;
    const int64_t units = small ? tiles / strips * ((strips + 3) / 4) : tiles;
    const int chunks = small || K % 128 ? K / 64 : K / 128;
    if (!small) cus = M <= 128 ? cus : 2 * cus;
    int sk = 1;
    while (units * sk < cus && sk * 2 <= 64 && chunks / (sk * 2) >= 1) sk *= 2;
    while (chunks / (sk * 2) >= 16 && units * sk * 2 <= cus && sk * 2 <= 64) sk *= 2;
    if (small && sk >= 2 && tiles >= cus)
        while (sk * 2 <= kSmallSplit && chunks / (sk * 2) >= 1) sk *= 2;
    return sk;
}

// For packed weights: 4 instead of 8 where the strips are fewer than the CUs and a range keeps eight chunks.
inline int plan_split_packed(int32_t B, int32_t M, int32_t N, int32_t K, int64_t cus) {
    const int sk = plan_split(B, M, N, K, cus);
    const int64_t tiles = B * (((int64_t)M + 15) / 16) * (((int64_t)N + kTileN - 1) / kTileN);
    return sk == 8 && M <= kSmallM && tiles < cus && K / 64 / 4 >= 8 ? 4 : sk;
}

// The tile kernel's shape for a call: MT 16-row tiles, NT 16-column tiles a wavefront and CW wavefronts side by side to a
// workgroup, K shared by `parts`, in ks workgroups.
struct TilePlan {
    int mt, nt, cw, parts, ks;
    bool far;
};

// mt, cw and parts depend on the sizes and on split_k only, not on the format, so that planes and packed weights give the
// same bits.  A CU takes its workgroups one after the other, so a shape costs its rounds over the CUs times what one
// workgroup costs per chunk: the KB that pass the CU's L1, 2 per row tile and 3.5 per 64 columns.
inline TilePlan tile_plan(const w6a16_args* a, const Layout& l, bool packed, int64_t cus) {
    TilePlan t{};
    const int chunks = a->K / 64, tiles = a->N / 16;
    auto groups = [&](int mt) { return (int64_t)a->B * (((int64_t)a->M + 16 * mt - 1) / (16 * mt)); };
    auto wgs = [&](int mt, int nt) { return groups(mt) * ((tiles + nt - 1) / nt); };
    auto rounds = [&](int64_t n) { return (n + cus - 1) / cus; };
    // Workgroups that may share a tile's K: none without room for their counters and partial tiles (so split_k bounds it;
    // up to 32 rows a split of at most 8 has no workspace).
    auto room = [&](int mt, int cw) {
        int most = a->M <= kSmallM ? (a->split_k > kSmallSplit ? 4 : 1) : a->split_k >= 4 ? 4 : a->split_k >= 2 ? 2 : 1;
        if ((size_t)(groups(mt) * tiles) * 4 > kCounterRegion) most = 1;
        while (most > 1 && (size_t)wgs(mt, 4 * cw) * most * 16 * mt * 64 * cw * 4 > l.partial_bytes) most >>= 1;
        return most;
    };
    // Workgroups of `wide` K parts, where CUs would be left without work.  Up to 128 chunks one workgroup's parts are short
    // already (us, packed / planes: K = N = 4096, M = 1, 16 / 32 parts 6.9 / 8.2 and 8.4 / 9.0), but for two row tiles on a
    // quarter of the CUs, whose planes gain (K = 8192, N = 2048, M = 20, 8 / 16 parts 13.6 / 13.7 and 19.1 / 13.5; K = N = 2560
    // 6.0 / 6.3 and 9.8 / 9.9).  Deeper K pays (K = 16384, N = 4096, M = 20, 8 / 16 / 32 parts 25.3 / 25.2 / 17.5 and 33.0 / 22.1
    // / 21.9); one row tile has 16 parts to begin with and takes twice as many, no more (M = 1, 16 / 32 / 64 parts 16.5 / 14.0
    // / 14.1 and 17.4 / 17.7 / 17.3).
    auto spread = [&](int mt, int cw, int wide) {
        const int64_t w4 = wgs(mt, 4 * cw), most = room(mt, cw);
        int s = 1;
        while (s < most && chunks >= wide * s * 2 && w4 * s * 2 <= cus &&
               (chunks > 128 || (mt == 2 && w4 * 4 <= cus && s < 2)) && !(mt == 1 && s == 2))
            s *= 2;
        return s;
    };
    // Rows to a workgroup: one tile up to 16 rows, two up to 32; above, two to four tiles and, from three on, 64 or 128
    // columns, whatever costs least (us, packed: K = N = 4096, M = 64: mt 2 10.3, mt 4 13.3; N = 16384: 25.6 / 22.2;
    // K = N = 2560, M = 203: mt 2, 3, 4 14.9 / 11.4 / 12.8).
    t.cw = 1;
    if (a->M <= 16) {
        t.mt = 1;
    } else if (chunks <= 2) {
        // what a workgroup writes costs more than what it reads (us, packed, N = 16384: K = 64, M = 64, mt 1, 2, 4 6.0 / 8.3 /
        // 12.8; M = 256 11.9 / 11.2 / 17; K = 128, M = 128 9.9 / 7.9 / 10.3)
        t.mt = wgs(1, 4) <= 4 * cus ? 1 : 2;
    } else {
        t.mt = 2;
        auto cost = [&](int mt, int cw) { return rounds(wgs(mt, 4 * cw)) * (4 * mt + 7 * cw); };
        int64_t best = cost(2, 1);
        if (a->M > 32)
            for (int mt = 3; mt <= 4; ++mt)
                for (int cw = 1; cw <= 2; ++cw)
                    if (cost(mt, cw) < best) best = cost(mt, cw), t.mt = mt, t.cw = cw;
    }
    const int64_t w4 = wgs(t.mt, 4 * t.cw);
    const int most = room(t.mt, t.cw);
    // Wavefronts that share K: eight to a workgroup (with two column wavefronts four), with one row tile 16 where the
    // workgroups do not fill the chip and a part of 16 has more than one chunk, else 4 (us, packed / planes: K = 4096, N =
    // 16384, M = 1: 4 12.4 / 16.2, 8 12.6 / 16.8, 16 13.3 / 17.7; K = N = 1024, M = 16: 4 4.0 / 5.6, 16 5.4 / 6.6; K = N = 2048,
    // M = 1: 8 4.4 / 7.0, 16 5.2 / 6.4), and twice or four times as many where a deep K would otherwise leave CUs without work
    // (K = 16384, N = 4096, M = 1: 16 parts in one workgroup 16.4, 32 in two 14.1).
    int wide = t.mt == 1 ? (w4 < cus && chunks > 16 ? 16 : 4) : 8 / t.cw;
    // Two row tiles and more, several rounds over the CUs: fewer to a workgroup, several of which then share a CU and fewer
    // follow each other.  A round costs its chunks a part and about 4/3 of a chunk for its start and end (K = 1024, N = 65536,
    // us, packed: M = 32, 8, 4, 2, 1 parts 25.5 / 18.8 / 18.7 / 20.5; M = 128, 4, 2, 1 53.9 / 46.3 / 43.8; M = 192 76.7 / 64.4 /
    // 71.1; K = 4096, N = 16384, M = 128 32.2 / 41.9 / 69).
    if (t.mt > 1) {
        const int full = wide;
        auto cost = [&](int n) { return (w4 * n + cus * full - 1) / (cus * full) * (3 * ((chunks + n - 1) / n) + 4); };
        for (int n = full / 2; n >= 1 && w4 > cus; n /= 2)
            if (cost(n) < cost(wide)) wide = n;
    }
    t.parts = std::min(chunks, wide * spread(t.mt, t.cw, wide));
    auto fits = [&](int ks, int max_w) { return ks == 1 ? t.parts <= max_w : t.parts % 4 == 0 && t.parts / ks <= max_w; };
    // Columns to a wavefront and workgroups to a K range.  Packed: as few workgroups to a K range as hold the parts, and
    // the columns whose rounds cost least.  Planes: 64 columns (a lane loads four), K spread over more workgroups
    // while every one of them still gets a CU and, from two row tiles on, a part has six chunks: their partial tiles then
    // cost more than what a short loop gains (six products of C = 768, M = 33: 69 us spread, 53 not; C = 2560, five chunks
    // a part, M = 48: 90.8 / 85.8; C = 4096, eight, M = 64: 133 / 141; one row tile, C = 2560, M = 1: 59.6 / 64.7).
    int64_t best = 0;
    for (int nt = packed ? 1 : 4; nt <= 4; nt *= 2) {
        if (t.mt > 2 && nt < 4) continue;
        const int max_w = t.mt == 1 || (t.mt == 2 && nt == 1) ? 16 : 8 / t.cw;
        int ks = 1;
        while (ks < most && !fits(ks, max_w)) ks *= 2;
        if (!fits(ks, max_w)) continue;
        if (!packed)
            while (ks * 2 <= most && fits(ks * 2, max_w) && t.parts / (ks * 2) >= 4 && w4 * ks * 2 <= cus &&
                   (t.mt == 1 || chunks >= 6 * t.parts))
                ks *= 2;
        const int64_t cost = rounds(wgs(t.mt, nt * t.cw) * ks) * (2 * nt + 3 * t.mt);
        if (!best || cost < best) best = cost, t.nt = nt, t.ks = ks;
    }
    // Planes, one row tile, 128 columns to a workgroup where that leaves every CU one: eight columns a lane, half the load
    // instructions (us, four / eight columns: K = 4096, M = 16, N = 65536 58.5 / 44.0, 32768 31.7 / 24.4, 16384 19.1 / 21.7).
    // (Two parts at least: the outputs take a thread a column.)
    if (!packed && t.mt == 1 && t.ks == 1 && t.parts >= 2 && t.parts <= 8 && wgs(1, 8) >= cus) t.nt = 8;
    // Planes, deep K, a single round of workgroups of two row tiles: half as many groups of rows, of up to twice the rows, and
    // the same parts over two workgroups, since the planes' loads are what takes the time there (K = 16384, N = 4096, us, two
    // row tiles / three or four: M = 65 47.7 / 36.6, 128 48.1 / 42.4; K = 8192: 25.9 / 25.7, 26.8 / 29.4).
    if (!packed && t.mt == 2 && t.ks == 1 && t.parts == 8 && most >= 2 && chunks >= 256)
        for (int mt = 3; mt <= 4; ++mt)
            if (wgs(mt, 4) * 2 <= cus && groups(mt) * 2 <= groups(2) + 1 &&
                (size_t)wgs(mt, 4) * 2 * 16 * mt * 64 * 4 <= l.partial_bytes) {
                t.mt = mt, t.ks = 2;
                break;
            }
    // Planes whose 32 rows span 2 GB, rows of A of which 64 do: 16 rows and 64 columns to a workgroup, with 64-bit
    // addresses, and the same parts, so the same bits as for the same rows packed or side by side.  (More than 16 parts
    // come only with few tiles, whose counters and partial tiles have room.)
    t.far = (!packed && a->N >= (1 << 26)) || (a->M > 1 ? a->a_row_stride : a->K) >= (1 << 24);
    if (t.far) t.mt = 1, t.nt = 4, t.cw = 1, t.ks = t.parts > 16 ? 2 : 1;
    return t;
}

// Whether a call runs the wide kernel: the sizes decide, not the format, so that planes and packed weights give the same
// bits.  145..256 rows (of three groups of 64 the last then has 17 rows or more; K = 4096, N = 32768, us, planes / packed,
// tile against wide: M = 144 83.4 / 70.8 against 95.3 / 78.9, 145 88.9 / 79.5 against 89.6 / 79.2, 176 92.3 / 83.0 against 93.5
// / 77.1), eight chunks (with four as fast), two tiles and more to a CU, of which the last two rounds fill a quarter (K =
// 4096, M = 193, tile against wide: N = 16384 59.2 / 55.3 against 56.7 / 48.0, 17408 78.0 / 65.6 against 87.9 / 73.0, 20480
// 88.2 / 77.0 against 88.7 / 73.7), and planes and scales that a buffer covers (below 2 GB).
inline bool wide_call(const w6a16_args* a, const Layout& l, int64_t cus) {
    if (l.big || a->M <= 144 || a->M > 256 || a->K < 512) return false;
    const int64_t tiles = (int64_t)a->B * l.m_groups * l.n_strips, twice = 2 * cus, last = tiles % twice;
    if (tiles < twice || (last > 0 && 4 * last < twice)) return false;
    const int64_t limit = 0x7FFFFFFF;
    return (int64_t)(a->K / 2) * a->N < limit && (int64_t)(a->K / a->group_k) * a->N * 2 < limit;
}

}  // namespace w6
