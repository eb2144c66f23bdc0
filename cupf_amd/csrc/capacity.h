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

// Waves of the +x strip of one plane (its columns, 64 / width rows to a wave).
inline int cap_strip_waves(int fnx, int fny, int partial_min)
{
    const int ex = (fnx - 2) - 64 * cap_tiles_x(fnx, partial_min);
    return ex > 0 ? (fny - 2 + 64 / ex - 1) / (64 / ex) : 0;
}

// Entries of one of `segs` (a power of two up to 64) segments of that list: the
// interior rows, y-major ((j - 1) * (fnz - 2) + k - 1), are cut into 64 equal
// parts, and a wave's points (64 at most: a row of a tile, or its part of the
// strip) go to the part of its first row.  A quarter as many segments hold four
// parts each, so every split fits the full one's list.
inline long long fix_segment_cap(int fnx, int fny, int fnz, int partial_min, int segs)
{
    const long long nz = fnz - 2, part = ((fny - 2) * nz + 63) / 64;
    long long waves = cap_tiles_x(fnx, partial_min) * part;
    if (cap_strip_waves(fnx, fny, partial_min)) {
        const int per = 64 / ((fnx - 2) % 64);  // y rows of a strip wave
        const long long js = (part + nz - 1) / nz + 1;  // y rows that a part touches at most
        const long long strip = (js + per - 1) / per * nz;
        waves += strip < part ? strip : part;
    }
    return waves * 64 * (64 / segs);
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
