// How a prefill launch is laid out: rows per workgroup, heads per set of packed rows, slices along the keys. Host code.
#ifndef GI_PREFILL_PLAN_H
#define GI_PREFILL_PLAN_H

#include <algorithm>
#include <cstddef>
#include <cstdint>

constexpr int kPrefillCUs = 256;      // compute units of a gfx950 device; a prefill workgroup takes one of its own
constexpr int kPrefillKeys = 64;      // keys per prefill tile; must match the kernels' PF_BK
constexpr int kPrefillMaxSlices = 64; // must match the kernels' PFC_MAXS

// The kernels of a launch: MFMA kernels over tiles staged as they are in memory (two sizes of workgroup), MFMA kernels that
// widen each int8 or 4-bit tile as they stage it (the larger workgroup only), and the f32 kernels (8 waves of 16 rows).
enum PrefillKind { kPrefillStaged, kPrefillTile, kPrefillF32 };

struct PrefillPlan {
    int waves;      // per workgroup: 8 or 4; head size 256: 4 or 2; f32: 8
    int group;      // query heads that share row tiles
    int rows;       // of a row tile: the workgroup's, or where an uncut launch leaves CUs idle half of them or fewer
    int tiles;      // key tiles per slice
    int nslice;     // slices of the longest row tile
};

inline int prefill_row_tiles(long long rows, int per) { return (int)((rows + per - 1) / per); }
inline int prefill_wave_rows(PrefillKind kind) { return kind == kPrefillF32 ? 16 : 32; }
inline int prefill_most_waves(PrefillKind kind, int hd) { return hd == 256 && kind != kPrefillF32 ? 4 : 8; }
// waves of a row tile of `rows` that hold any of P rows
inline int prefill_pwaves(long long P, int rows, int rw) { return P > rows ? rows / rw : (int)((P + rw - 1) / rw); }
// Bytes of a sliced launch's partials
inline size_t prefill_part_bytes(int nslice, int waves, PrefillKind kind, int n, int n_heads, int n_kv, int hd) {
    if (nslice == 1) return 0;
    const int rw = prefill_wave_rows(kind), rows = rw * waves;
    const long long P = (long long)n * (n_heads / n_kv);
    const size_t b = (size_t)prefill_row_tiles(P, rows) * n_kv * nslice * prefill_pwaves(P, rows, rw) * rw * (hd + 2) * 4;
    return (b + 255) / 256 * 256;
}

// Rows per kv head from which the int8 keys are widened into the workspace first (one pass over all keys, ~6 bytes moved
// per value) rather than tile by tile in the prefill: above one row tile (of 8 waves), every tile would be widened again for each.
// 32/8 heads of 128, tile by tile / widened: 16 tokens at a 2000-token prefix 17.6 / 21.5 us, at 16000 29.6 / 43.5; 64
// tokens at 2000 27.7 / 26.7, at 16000 48 / 51; 256 tokens at 2000 84 / 55; 8192 tokens 634 / 588.
constexpr int kPrefillWidenRows = 256;
inline bool prefill_widens(int n, int n_heads, int n_kv, int hd) {
    return hd == 256 || (long long)n * (n_heads / n_kv) > kPrefillWidenRows;
}

// A launch has one workgroup per (kv head, tile of packed query rows), and a CU holds one workgroup.
//  - Waves: 8 (256 rows, two waves per SIMD) or 4 (128 rows, one per SIMD). One wave takes a key tile in about 0.7 of
//    the time that two on its SIMD take for theirs together, so 4 waves win where the workgroups are few or unequal
//    (1024 tokens of 32/8 heads of 128, f16: 33.9 us with 8, 23.7 with 4; 512 at a 2000-token prefix 64 and 44) and
//    8 where they fill the chip several times over (8192 tokens: 505 and 580). Head size 256: 4 or 2.
//  - Slices: a short batch over a long prefix leaves most of the chip idle while each workgroup walks all of its keys
//    (512 tokens of 32/4 heads at a 16K prefix: 64 workgroups of 264 key tiles, 350 us). Such a launch cuts the key
//    tiles of every row tile into slices, one workgroup each, whose partial results a second launch merges (137 us).
//    An f32 tile takes three to five times as long, so those launches gain from shorter spans on (200 tokens of 32/32
//    heads of 96 at 1800: 64 workgroups of 32 tiles, 227 us; sliced 69 us).
//  - Tiles widened through registers have the larger workgroup only. Where a call with a workspace would stage widened
//    keys, the slices are those of that call, rated by its forms, so that both give the same bits. Up to kPrefillWidenRows
//    no call does, and the slices are rated by what such a tile takes: 1.9 us (57 tokens of 32/8 heads of 128 at 16000
//    int8 keys, 2 slices 242 us), 1.27 of a staged one, and 0.09 us a slice in the merge (rated by the staged forms: 57
//    tokens at 6100 keys took 14 slices, 32.2 us, now 20, 30.8; 64 of 32/8 heads of 64 at 16000 33.3, now 30.2; 40 of 9/3
//    at 6100 19.1, now 17.4; at worst 40 of 9/3 at 40000 31.3, now 32.6). Over 40 calls of 16 to 64 tokens, prefixes 1000 to
//    40000, that is 0.8% in the mean above the best of 1 to 64 slices, 5% at most; it was 2.2 and 13.
// A row's arithmetic does not depend on the waves, the set or the rows of its tile, only on the slices. Of a sliced launch the partials fit
// `room` bytes.
inline PrefillPlan prefill_rate(int pos0, int n, int n_heads, int n_kv, int hd, PrefillKind kind, size_t room) {
    const bool f32 = kind == kPrefillF32;
    const int G = n_heads / n_kv, cus = kPrefillCUs, tmax = (pos0 + n + kPrefillKeys - 1) / kPrefillKeys;
    const long long P = (long long)n * G;
    const int most = prefill_most_waves(kind, hd), rw = prefill_wave_rows(kind);
    const bool tile_only = kind == kPrefillTile && !prefill_widens(n, n_heads, n_kv, hd);
    PrefillPlan p{most, G, rw * most, tmax, 1};
    if ((long long)prefill_row_tiles(P, rw * most) * n_kv >= 2 * cus) return p; // longest tiles first balances these
    // Below 16 key tiles slices save less than the merge launch costs. A prompt of up to 4096 keys taken in chunks of
    // 256 tokens or more keeps each row's arithmetic independent of the chunking (one slice always); beyond, and in
    // shorter chunks, rows differ from the uncut ones by f16's step (each slice rounds its P against its own maximum).
    // What that costs such chunks, 255 (cut) and 256 tokens (not): 32/8 heads of 128, f16, at 1500 keys 25 and 32 us, at
    // 3000 30 and 51; 16/2 heads of 256 at 3000 37 and 83; in f32 (32/8 heads of 128) at 500 50 and 117, at 3000 135 and
    // 462. (Never cut, 256 tokens took 49, 80, 99, 117 and 462 before the row tiles were packed.)
    const bool may_slice = room && tmax >= (f32 ? 4 : 16) && (n < 256 || pos0 + n > 4096);
    // Costs in units of one key tile of an 8-wave workgroup (1.4 to 1.9 us; head size 256: of a 4-wave one): rounds of
    // workgroups over the CUs, each with a fixed cost until its first tile is in and for its output (~6 us), and for a
    // sliced launch the merge launch (~5 us) and its read of the partials (~4 TB/s).
    const double tile_s = f32 ? 5e-6 : 1.5e-6, per_wg = f32 ? 1.2 : 4.0, merge = f32 ? 1.0 : 3.3;
    const double per_slice = tile_only ? 0.06 : 0.0, less = tile_only ? 0.97 : 0.95;
    double best = 0, uncut = 0;
    int uncut_waves = most;
    for (int waves = most; waves >= (f32 || tile_only ? most : most / 2); waves -= most / 2) {
        const int rows = rw * waves, items = prefill_row_tiles(P, rows);
        const long long wgs = (long long)items * n_kv;
        const double tile = tile_only ? 1.27 : waves == most ? 1.0 : hd == 256 ? 0.85 : 0.7;
        auto tiles_of = [&](int i) { // key tiles of row tile i
            const long long last = std::min<long long>(n - 1, ((long long)(i + 1) * rows - 1) / G);
            return (int)((pos0 + last) / kPrefillKeys + 1);
        };
        // one slice: the longest workgroup, or the mean load of a CU where there are several rounds
        const double mean = (double)wgs / cus * (tile * (tiles_of(0) + tmax) / 2 + (wgs > cus ? per_wg : 0));
        const double one = std::max(tile * tmax, mean) + per_wg;
        // and where one round of them is about as long as the next (a long prefix under them all): r + 1 rounds take r + 1
        // times what the longest workgroup of the last of them does. (f16, uncut, 4 / 8 waves: 1500 tokens at 3000, 32/8
        // heads of 128, 376 workgroups or 192, 123 / 114 us; 4096 at 16000, 9/3 heads of 64, 288 or 144, 352 / 283; at
        // position 0 2000 tokens of 32/8 heads of 128 44 / 53. Of 250 calls, 1050 to 4096 tokens at 0 to 12000, five head
        // shapes, f16 and int8, the size taken costs 0.2% over the better one in the mean, 5.5% at most; with the mean load
        // alone it was 5.8 and 75.) It decides between the two sizes only: whether a launch is cut does not depend on it.
        const double later = hd == 64 && waves != most ? 0.75 : tile;
        double rounds = one;
        for (int r = 1; (long long)r * cus < wgs; r++)
            rounds = std::max(rounds, (r + 1) * (later * tiles_of(items - 1 - r * cus / n_kv) + per_wg));
        if (waves == most || rounds < 1.05 * uncut) uncut = rounds, uncut_waves = waves; // (rounds overlap a little)
        if (waves == most || one < 0.95 * best) best = one, p = PrefillPlan{waves, G, rows, tmax, 1};
        if (!may_slice) continue;
        const double part = std::min<long long>(P, rows) * (hd + 2) * 4.0 / 4e12 / tile_s;
        for (int S = 2; S <= std::min(kPrefillMaxSlices, tmax / 2) && wgs * S <= 4 * cus; S++) {
            const int C = (tmax + S - 1) / S, slices = (tmax + C - 1) / C;
            if (prefill_part_bytes(slices, kind == kPrefillTile ? most : waves, kind, n, n_heads, n_kv, hd) > room) continue;
            long long u = 0; // workgroups with keys
            if (tiles_of(0) + C > tmax) u = wgs * slices; // (every row tile has tmax tiles or nearly)
            else
                for (int i = 0; i < items; i++) u += (long long)n_kv * ((tiles_of(i) + C - 1) / C);
            const double cost = (double)((u + cus - 1) / cus) * (tile * C + per_wg) + merge + per_slice * slices + u * part;
            if (cost < less * best) best = cost, p = PrefillPlan{waves, G, rows, C, slices};
        }
    }
    if (p.nslice == 1) p.waves = uncut_waves, p.rows = rw * p.waves;
    return p;
}

// The plan of a call whose workspace has `room` bytes for partials.
// A launch that is not cut and leaves CUs idle takes the smaller workgroup, splits the group of a kv head's query heads into
// sets with row tiles of their own, and gives a workgroup fewer rows than its waves hold (half, a quarter, 32; the waves
// without rows stage tiles), each where that gives more workgroups, at most one each CU: a workgroup loads its rows'
// queries and stores its outputs by itself, and 128 rows of 256 f32 take it 7 us longer than 16. A step has to give a
// quarter more over a few key tiles (16/2 heads of 256, 200 tokens 15.1 / 13.6 us, 64 workgroups for 50), half as many
// again over longer spans, where that share counts for less (32/4 heads of 128, 300 tokens at 1500: 96 workgroups for 76
// take 33.4 us, 76 32.2). Replayed graph, whole groups / sets / sets and fewer rows: 32/8 heads of 128, f16, position 0, 64
// tokens 8.8 / 7.1 / 6.3 us, 250 tokens - / 11.1 / 8.8; int8 without a workspace, 250 tokens - / 18.9 / 12.0, 512 at
// 3000 - / 112 / 81; 16/2 heads of 256, f16, 16 tokens 14.2 / 8.4 / 8.4, 64 tokens 14.5 / 10.4 / 8.9.
// The f32 kernels, bound by their MFMAs with two waves a SIMD, always take one head a set: waves of a tile of 128 tokens of
// one head skip the key tiles past their own last row, where 128 rows of 4 heads all end at the same one (32/8 heads of
// 96, whole groups / sets: 32 tokens 19.3 / 10.0 us, 256 tokens 40.2 / 36.3, 4096 tokens 867 / 864).
inline PrefillPlan prefill_plan(int pos0, int n, int n_heads, int n_kv, int hd, PrefillKind kind, size_t room) {
    PrefillPlan p = prefill_rate(pos0, n, n_heads, n_kv, hd, kind, room ? SIZE_MAX : 0);
    const int most = prefill_most_waves(kind, hd), G = n_heads / n_kv;
    if (kind == kPrefillTile) p.waves = most, p.rows = prefill_wave_rows(kind) * most;
    if (prefill_part_bytes(p.nslice, p.waves, kind, n, n_heads, n_kv, hd) > room) {
        p = prefill_rate(pos0, n, n_heads, n_kv, hd, kind, room);
        if (kind == kPrefillTile) p.waves = most, p.rows = prefill_wave_rows(kind) * most;
    }
    if (p.nslice > 1) return p;
    if (kind == kPrefillF32) {
        p.group = 1;
        return p;
    }
    auto wgs = [&](int rows, int group) { return (long long)n_heads / group * prefill_row_tiles((long long)n * group, rows); };
    long long have = wgs(p.rows, p.group);
    const int gain = p.tiles < 16 ? 25 : 50; // percent more workgroups that a split has to give
    auto better = [&](long long w) { return w <= kPrefillCUs && w * 100 >= have * (100 + gain); };
    const int half = prefill_wave_rows(kind) * most / 2;
    if (kind == kPrefillStaged && p.waves == most && better(wgs(half, G))) p.waves = most / 2, p.rows = half, have = wgs(half, G);
    for (int g = G - 1; g >= 1; g--)
        if (G % g == 0 && better(wgs(p.rows, g))) p.group = g, have = wgs(p.rows, g);
    for (int rows = p.rows / 2; rows >= prefill_wave_rows(kind); rows /= 2)
        if (better(wgs(rows, p.group))) p.rows = rows, have = wgs(rows, p.group);
    return p;
}

#endif
