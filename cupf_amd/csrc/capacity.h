// capacity.h -- worst-case entries of a step's work lists, recomputed from
// the grid and the chunk depth alone (not from the values pf_create derived
// and stored), for the host check before every launch; and the range of the
// epochs.  Plain C++: the CPU tests compile it on its own.
#pragma once

namespace cupf {

// Column tiles are 64 x 4 interior points; a leftover strip at the +x end at
// least partial_min wide is a partial tile, a narrower one goes to the strip's
// waves (which are computed, never listed).
inline int cap_tiles_x(int fnx, int partial_min)
{
    const int n = fnx - 2, t = n / 64;
    return (n - 64 * t >= partial_min) ? t + 1 : t;
}

inline int cap_tiles_y(int fny) { return (fny - 2 + 3) / 4; }

inline int cap_nzchunk(int fnz, int kchunk) { return (fnz - 2 + kchunk - 1) / kchunk; }

// Entries the plan kernel may list in one step: each (column tile, z chunk)
// pair at most once.
inline long long worst_list_items(int fnx, int fny, int fnz, int kchunk, int partial_min)
{
    return (long long)cap_tiles_x(fnx, partial_min) * cap_tiles_y(fny) * cap_nzchunk(fnz, kchunk);
}

// Entries of the overflow fix-up list in one step: each interior point at
// most once.
inline long long worst_fix_entries(int fnx, int fny, int fnz)
{
    return (long long)(fnx - 2) * (fny - 2) * (fnz - 2);
}

// Entries of one of `segs` (a power of two up to 64) segments of that list: the
// interior rows, y-major ((j - 1) * (fnz - 2) + k - 1), are cut into 64 equal
// parts, and a wave's points (the columns of a row of a tile, or its part of
// the strip: 64 / width rows) go to the part of its first row.  A quarter as
// many segments hold four parts each, so every split fits the full one's list.
// (64 entries to a wave, whatever its columns, made the list 2.05 times the
// interior at 32^3 and 4 times for 16 columns; now 1.06 and 1.0.)
inline long long fix_segment_cap(int fnx, int fny, int fnz, int partial_min, int segs)
{
    const long long ny = fny - 2, nz = fnz - 2, part = (ny * nz + 63) / 64;
    const int tiled = 64 * cap_tiles_x(fnx, partial_min), ex = fnx - 2 - tiled;
    long long points = part * (ex > 0 ? tiled : fnx - 2);
    if (ex > 0) {
        const long long per = 64 / ex;  // y rows of a strip wave
        const long long js = (part + nz - 1) / nz + 1;  // y rows that a part touches at most
        const long long waves = (js + per - 1) / per * nz;
        points += (waves < part ? waves : part) * ex * (per < ny ? per : ny);
    }
    return points * (64 / segs);
}

// First entry of segment `seg` of 2^shift parts of `cap` entries.  The list of a
// narrow, long grid (4 x 66 x 1.6 M points, one strip) passes 32 bits.
constexpr unsigned long long fix_segment_base(int seg, int shift, unsigned cap)
{
    return ((unsigned long long)seg << shift) * cap;
}

// Elements of a context's large arrays: a slot buffer's phi or ids, a field, the
// fix-up list, a buffer's activity and row maps, the work list.
struct ContextSizes {
    long long slots, field, fix, act, row, items;
};
inline ContextSizes context_sizes(int fnx, int fny, int fnz, int K, int kchunk, int partial_min)
{
    const long long field = (long long)fnx * fny * fnz, columns = (fnx - 2 + 63) / 64;
    return {K * field,
            field,
            64 * fix_segment_cap(fnx, fny, fnz, partial_min, 64),
            columns * cap_tiles_y(fny) * fnz,
            columns * fny * fnz,
            worst_list_items(fnx, fny, fnz, kchunk, partial_min) + 1};
}

// The epoch counter's limit: row words hold an epoch and 4 bits of bound, and
// a few epochs are taken between two looks at the counter (new states).
constexpr unsigned kEpochMax = 0x07ffffffu;

// Whether the counter may still take `ahead` epochs; the maps are renewed
// otherwise, and it starts again.
inline bool epochs_left(unsigned ctr, unsigned ahead) { return ahead < kEpochMax && ctr < kEpochMax - ahead; }

// Steps of a batched run that has `left` to go before the next look at its
// members' counters (a run takes an epoch per step).
inline int epoch_run(int left) { return left < (1 << 26) ? left : 1 << 26; }

}  // namespace cupf
