// apt_rows.h -- the step's main path (APTrhs_psi,
// 3DgrainMPI/APTPhaseField.cu:178-354): one wave per row of 64 points, straight
// from global memory, no LDS and no barriers.
//
// A row reads only the slots that its neighbourhood's row words say are filled
// (StepArgs::row_src): a grown microstructure holds 1-3 of its 8 slots, an
// initial one all of them.  Rows bounded by 4 slots take narrow_plane, whose
// loads all go out together; the others wide_plane, whose loads run one
// neighbour ahead of the compares.  Everything is indexed statically, so the
// gathered values live in registers.
//
// Bound by VALU issue in the general path (256x256x512 start-up: ~3,300
// instructions per row plane, 16 waves per CU) and by latency and launches in
// small grids.  Measured against 64x4 tiles with their halo in a three-plane
// LDS ring (76 KB, 203 registers: 8 waves per CU, every slot staged), step
// kernel: 256x256x512 at step 6 450 -> 215 us, at 150 259 -> 130, at 450 87 ->
// 36, at 1500 128 -> 55; 64^3 at step 10 108 -> 32, at 900 56 -> 21; 32^3 K=5
// 62 -> 16; a 78 % solid 256^3 window 1340 -> 1000.  The general path with its
// values in LDS (14 KB a wave, 10 waves per CU) took 1530 us for that window.
#pragma once

#include "apt_device.h"

namespace cupf {

namespace {

constexpr int kRowLanes = 64;  // one wave per workgroup: rows need no barrier

// Step arguments through a pointer the compiler cannot look through: fields
// are scalar loads where they are used, instead of ~100 uniform values held in
// (and spilled from) scalar registers across the whole kernel (174 scalar
// spills at first).  apt_step now, by the compiler's report, under the 128
// vector registers of 4 waves per SIMD: K = 5 115 registers and 5 scalar spills
// (27 points 111 and none); K = 8 128 with 24 scalar and 4 vector spills, 20 B of
// scratch a lane (27 points 5, 5 and 24 B).
typedef const __attribute__((address_space(4))) StepArgs CArgs;
__device__ __forceinline__ const StepArgs* args_ref(CArgs* p)
{
    asm volatile("" : "+s"(p));
    return (const StepArgs*)p;
}

// A wave's 64 points of one plane: column of the lane, and the element
// offsets of its x and y neighbours through the boundary maps.  Lanes past
// the end of a partial tile repeat the last column (on = false: they compute
// and do not store, mark or hand over).
struct RowLane {
    int i, j;
    int xm, xp, ym, yp;
    bool on;
};

__device__ __forceinline__ RowLane row_lane(const StepArgs& a, int i, int j, bool on)
{
    RowLane r;
    r.i = i;
    r.j = j;
    r.on = on;
    r.xm = bc_map(i - 1, a.fnx, a.bcx) - i;
    r.xp = bc_map(i + 1, a.fnx, a.bcx) - i;
    r.ym = (bc_map(j - 1, a.fny, a.bcy) - j) * a.fnx;
    r.yp = (bc_map(j + 1, a.fny, a.bcy) - j) * a.fnx;
    return r;
}

// Element at byte offset off (32 bits, per lane) from a wave-uniform base.
template <class T>
__device__ __forceinline__ T at_off(const T* base, unsigned off)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}
template <class T>
__device__ __forceinline__ void put_off(T* base, unsigned off, T v)
{
    *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off) = v;
}

// Plane terms (wave-uniform element offsets) and in-plane byte offsets (per
// lane) of the seven stencil points, order D,B,L,C,R,T,U.
struct RowStencil {
    int zD, zC, zU;
    unsigned c, xm, xp, ym, yp;
    __device__ __forceinline__ int plane(int s) const { return s == 0 ? zD : s == 6 ? zU : zC; }
    __device__ __forceinline__ unsigned off(int s) const
    {
        return s == 1 ? ym : s == 2 ? xm : s == 4 ? xp : s == 5 ? yp : c;
    }
};

__device__ __forceinline__ RowStencil row_stencil(const StepArgs& a, const RowLane& r, int k)
{
    const int A = a.fnx * a.fny;
    const int c = r.i + r.j * a.fnx;
    RowStencil t;
    t.zD = bc_map(k - 1, a.fnz, a.bcz) * A;
    t.zC = k * A;
    t.zU = bc_map(k + 1, a.fnz, a.bcz) * A;
    t.c = 4u * (unsigned)c;
    t.xm = 4u * (unsigned)(c + r.xm);
    t.xp = 4u * (unsigned)(c + r.xp);
    t.ym = 4u * (unsigned)(c + r.ym);
    t.yp = 4u * (unsigned)(c + r.yp);
    return t;
}

// Largest lane value of v (0..K) in the wave.
template <int K>
__device__ __forceinline__ int wave_max(int v)
{
    int m = 0;
#pragma unroll
    for (int q = 0; q < K; ++q) m += __ballot(v > q) != 0ull ? 1 : 0;
    return m;
}

// Destination maps of one row plane, m filled slots (K where the fix-up will
// fill them): the row of column tile tx, or (a strip) each lane's own row.
__device__ __forceinline__ void row_mark_tile(const StepArgs& a, const RowLane& r, int k, int tx, int m)
{
    if (m > 0 && threadIdx.x == 0) {
        a.act_dst[k * a.ntiles + act_tile_y(r.j) * a.ntx + tx] = a.ep_new;
        a.row_dst[(k * a.fny + r.j) * a.ntx + tx] = a.ep_new << 4 | (unsigned)m;
    }
}
__device__ __forceinline__ void row_mark_strip(const StepArgs& a, const RowLane& r, int k, int m)
{
    if (m > 0) {
        const int x = act_tile_x(r.i);
        a.act_dst[k * a.ntiles + act_tile_y(r.j) * a.ntx + x] = a.ep_new;
        atomicMax(a.row_dst + (k * a.fny + r.j) * a.ntx + x, a.ep_new << 4 | (unsigned)m);
    }
}

// One filled slot's new pair, and the stores of slot q.
__device__ __forceinline__ void row_store(const StepArgs& a, const RowStencil& t, int q, bool st, int id, float ph)
{
    if (st) {
        const long long b = (long long)q * a.L + t.zC;
        put_off(a.arg_new + b, t.c, id);
        put_off(a.ph_new + b, t.c, ph);
    }
}

// Gather of one row: ids in first-appearance order and, by list position and
// stencil row (D,B,L,C,R,T,U), the phi of the last entry holding the id (-1
// where the row has none).  Static registers throughout: an entry is compared
// with every list position and its phi selected into each.
// Which lanes have position q filled is a wave mask in scalar registers: a new
// id's lanes then find their free position with scalar ands, and only the
// positions that some of them take cost vector work (a new id takes 2-3 of the
// 8 over a wave; with a count per lane every new id went through all 8).
template <int K>
struct RowList {
    int la[K];
    float v[7][K];
    unsigned long long filled[K];  // lanes whose list reaches position q
    unsigned long long ovf;        // lanes with more ids than positions
    float outside;                 // largest phi of an entry whose id found no room
};

__device__ __forceinline__ bool in_mask(unsigned long long m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

template <int K>
__device__ __forceinline__ void list_init(RowList<K>& g)
{
#pragma unroll
    for (int q = 0; q < K; ++q) {
        g.la[q] = kNoKey;  // never a grain id
        g.filled[q] = 0ull;
#pragma unroll
        for (int s = 0; s < 7; ++s) g.v[s][q] = -1.0f;
    }
    g.outside = -__builtin_huge_valf();
    g.ovf = 0ull;
}

// Entry (x, f) of a neighbour point, its slot `slot`, the (before + 1)th of the
// gather; S: its stencil row, -1 for none; SKIP: leave at once where no lane has an id (pays
// with the 7 points, whose entries run up to the largest bound around: 1060 ->
// 1020 us for a 78 % solid 256^3 window; the 27 points lose 5 %).
// Only positions that earlier entries can have filled are looked at.  Positions
// fill in order, so a pair whose second one is filled in every lane that meets
// a new id has nothing to take: one branch per pair (256x256x512 at step 150:
// 162 us with a branch per position or one for all 8, 157 with pairs).
template <int K, int S, bool SKIP>
__device__ __forceinline__ void list_entry(int x, float f, int before, int slot, RowList<K>& g)
{
    unsigned long long left = __ballot(x != -1);  // lanes that meet a new id
    if (SKIP && left == 0ull) return;
    // A point and the one above it hold their ids in the order in which the
    // point below listed them a step ago: their slot's own position first, and
    // mostly nothing is left to look for (9 of 10 entries in a solid window, 2
    // of 3 in a start-up; 982 -> 957 us, 227 -> 215; the narrow path loses 4 %,
    // and as an exit of its own, before the compares, it cost 20 % in copies).
    constexpr bool HINT = SKIP && (S == 3 || S == 6) && K > 4;
    if (HINT) {
        const bool e = g.la[slot] == x;
        g.v[S < 0 ? 0 : S][slot] = e ? f : g.v[S < 0 ? 0 : S][slot];
        left &= ~__ballot(e);
        if (left == 0ull) return;
    }
#pragma unroll
    for (int q = 0; q < K; ++q) {
        if (q >= before) break;
        if (HINT && q == slot) continue;
        const bool e = g.la[q] == x;
        if (S >= 0) g.v[S < 0 ? 0 : S][q] = e ? f : g.v[S < 0 ? 0 : S][q];
        left &= ~__ballot(e);
    }
    if (left != 0ull) {
#pragma unroll
        for (int b = 0; b < K; b += 2) {
            if (b > before) break;
            if ((left & ~g.filled[b + 1 < K ? b + 1 : b]) == 0ull) continue;
#pragma unroll
            for (int q = b; q < b + 2 && q < K; ++q) {
                if (q > before) break;
                const unsigned long long t = left & ~g.filled[q];
                const bool w = in_mask(t);
                g.la[q] = w ? x : g.la[q];
                if (S >= 0) g.v[S < 0 ? 0 : S][q] = w ? f : g.v[S < 0 ? 0 : S][q];
                g.filled[q] |= t;
                left &= ~t;
            }
        }
        if (before >= K && left != 0ull) {
            const bool full = in_mask(left);
            g.ovf |= left;
            g.outside = full && f > g.outside ? f : g.outside;
        }
    }
}

// Positions filled in any lane of the wave, and in this lane.
template <int K>
__device__ __forceinline__ int list_max(const RowList<K>& g)
{
    int m = 0;
#pragma unroll
    for (int q = 0; q < K; ++q) m += g.filled[q] != 0ull ? 1 : 0;
    return m;
}
template <int K>
__device__ __forceinline__ int list_len(const RowList<K>& g)
{
    int n = 0;
#pragma unroll
    for (int q = 0; q < K; ++q) n += in_mask(g.filled[q]) ? 1 : 0;
    return n;
}

template <int P>
struct RowEntries {
    int x[P];
    float f[P];
};

template <int P>
__device__ __forceinline__ void entries_load(const StepArgs& a, int z, unsigned o, RowEntries<P>& e)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const long long b = (long long)p * a.L + z;
        e.x[p] = at_off(a.arg + b, o);
        e.f[p] = at_off(a.ph + b, o);
    }
}

// (SKIP comes with the 7-point order, whose S * P + p entries came before.)
template <int K, int P, int S, bool SKIP = true>
__device__ __forceinline__ void entries_list(const RowEntries<P>& e, RowList<K>& g)
{
#pragma unroll
    for (int p = 0; p < P; ++p) list_entry<K, S, SKIP>(e.x[p], e.f[p], SKIP ? S * P + p : K, p, g);
}

// The same, each entry's registers refilled with the next point's (plane term
// z, offset o) as it is taken: a whole point's loads stay in flight behind the
// compares, in one point's registers.
template <int K, int P, int S>
__device__ __forceinline__ void entries_list_next(const StepArgs& a, int z, unsigned o, RowEntries<P>& e,
                                                  RowList<K>& g)
{
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int x = e.x[p];
        const float f = e.f[p];
        list_entry<K, S, true>(x, f, S * P + p, p, g);
        const long long b = (long long)p * a.L + z;
        e.x[p] = at_off(a.arg + b, o);
        e.f[p] = at_off(a.ph + b, o);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// List positions of the narrow path: a row bounded by P <= 4 slots hardly
// ever gathers a fifth id (0.2 % of the rows of a grown 256x256x512 state).
constexpr int kNarrowList = 4;

// One plane of a row whose neighbourhood holds nothing above slot P - 1
// (7-point gather).  False if some lane gathers more than kNarrowList ids:
// nothing is written then and the wave takes the general path.
template <int K, int P>
__device__ __forceinline__ bool narrow_plane(const StepArgs& a, const RowLane& r, int k, int tx, int D,
                                             float xi, float yj, float a_s, float epsv)
{
    constexpr int M = kNarrowList;
    const RowStencil t = row_stencil(a, r, k);
    RowEntries<P> e[7];
#pragma unroll
    for (int s = 0; s < 7; ++s) entries_load(a, t.plane(s), t.off(s), e[s]);
    RowList<M> g;
    list_init(g);
    entries_list<M, P, 0>(e[0], g);
    entries_list<M, P, 1>(e[1], g);
    entries_list<M, P, 2>(e[2], g);
    entries_list<M, P, 3>(e[3], g);
    entries_list<M, P, 4>(e[4], g);
    entries_list<M, P, 5>(e[5], g);
    entries_list<M, P, 6>(e[6], g);
    if (g.ovf != 0ull) return false;
    const int nm = list_max(g);
    const int nst = max(nm, D);
    if (nst == 0) return true;
    bool skip = false;
    float Up = 0.0f;
    float rw[M];
    if (nm > 0) {
        float T;
        skip = thermal_Tv(a, xi, yj, a.z[k], T);
        Up = T / a.L_cp;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const float w = g.v[3][q] + 1.0f;
            rw[q] = 0.25f * w * w;
        }
    }
    // every slot's orientation rows in one round trip; a lane without a
    // gradient needs none (its anisotropy is 1 under any rotation)
    Rot m[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
        if (q < nm) {
            const bool flat = g.v[4][q] == g.v[2][q] && g.v[5][q] == g.v[1][q] && g.v[6][q] == g.v[0][q];
            m[q] = slot_rot(a, in_mask(g.filled[q]) ? g.la[q] : 0, flat ? -1.0f : g.v[3][q]);
        }
    }
#pragma unroll
    for (int q = 0; q < M; ++q) {
        if (q < nst) {
            int oid = -1;
            float oph = -1.0f;
            const bool in = in_mask(g.filled[q]);
            if (q < nm) {
                float repul = 0.0f;  // unfilled slots add exactly +0
#pragma unroll
                for (int p = 0; p < M; ++p)
                    if (p != q) repul += rw[p];
                const float nv = slot_update_r(a, m[q], g.v[0][q], g.v[1][q], g.v[2][q], g.v[3][q], g.v[4][q],
                                               g.v[5][q], g.v[6][q], repul, Up, a_s, epsv);
                oph = in ? nv : -1.0f;
                oid = in && !(nv < kKillf) ? g.la[q] : -1;
            }
            row_store(a, t, q, r.on && !(skip && in), oid, oph);
        }
    }
#pragma unroll 1
    for (int q = M; q < nst; ++q) row_store(a, t, q, r.on, -1, -1.0f);
    if (tx >= 0) row_mark_tile(a, r, k, tx, nm);
    else row_mark_strip(a, r, k, r.on ? list_len(g) : 0);
    return true;
}

template <int K, bool G27, int P>
__device__ __forceinline__ void row_gather(const StepArgs& a, const RowStencil& t, RowList<K>& g)
{
    if (!G27) {
        RowEntries<P> e;
        entries_load(a, t.zD, t.c, e);
        entries_list_next<K, P, 0>(a, t.zC, t.ym, e, g);
        entries_list_next<K, P, 1>(a, t.zC, t.xm, e, g);
        entries_list_next<K, P, 2>(a, t.zC, t.c, e, g);
        entries_list_next<K, P, 3>(a, t.zC, t.xp, e, g);
        entries_list_next<K, P, 4>(a, t.zC, t.yp, e, g);
        entries_list_next<K, P, 5>(a, t.zU, t.c, e, g);
        entries_list<K, P, 6>(e, g);
    } else {
        // z-major 27-point order (3Dgrain/APTPhaseField.cu:241-268): the
        // stencil rows keep phi, the other 20 positions only contribute ids
        // and run as loops of one position
        const int zD = t.zD, zC = t.zC, zU = t.zU;
        const unsigned c = t.c, xm = t.xm, xp = t.xp, ym = t.ym, yp = t.yp;
        auto ids = [&](int from, int to) {
#pragma unroll 1
            for (int u = from; u < to; ++u) {
                const int zi = u / 9, yi = (u - 9 * zi) / 3, xi = u - 9 * zi - 3 * yi;
                const int z = zi == 0 ? zD : zi == 2 ? zU : zC;
                const unsigned o = (xi == 0 ? xm : xi == 2 ? xp : c) + (yi == 0 ? ym - c : yi == 2 ? yp - c : 0u);
                int x[P];
#pragma unroll
                for (int p = 0; p < P; ++p) x[p] = at_off(a.arg + ((long long)p * a.L + z), o);
#pragma unroll
                for (int p = 0; p < P; ++p) list_entry<K, -1, false>(x[p], 0.0f, K, -1, g);
            }
        };
        RowEntries<P> e;
        ids(0, 4);
        entries_load(a, zD, c, e);
        entries_list<K, P, 0, false>(e, g);
        ids(5, 10);
        entries_load(a, zC, ym, e);
        entries_list<K, P, 1, false>(e, g);
        ids(11, 12);
        entries_load(a, zC, xm, e);
        entries_list<K, P, 2, false>(e, g);
        entries_load(a, zC, c, e);
        entries_list<K, P, 3, false>(e, g);
        entries_load(a, zC, xp, e);
        entries_list<K, P, 4, false>(e, g);
        ids(15, 16);
        entries_load(a, zC, yp, e);
        entries_list<K, P, 5, false>(e, g);
        ids(17, 22);
        entries_load(a, zU, c, e);
        entries_list<K, P, 6, false>(e, g);
        ids(23, 27);
    }
}

// One plane of a row, any neighbourhood: P and D bound the filled slots of
// the neighbourhood's source and of the destination.
template <int K, bool G27>
__device__ __forceinline__ void wide_plane(const StepArgs& a, const RowLane& r, int k, int tx, int P, int D,
                                           float xi, float yj, float a_s, float epsv, unsigned& nres)
{
    const RowStencil t = row_stencil(a, r, k);
    RowList<K> g;
    list_init(g);
    if (P <= 4) row_gather<K, G27, 4>(a, t, g);
    else if (K > 6 && P <= 6) row_gather<K, G27, 6>(a, t, g);
    else row_gather<K, G27, K>(a, t, g);
    const unsigned long long on = __ballot(r.on);
#pragma unroll
    for (int q = 0; q < K; ++q) g.filled[q] &= on;
    g.ovf &= on;
    // An overflowed point whose list ids all reach a phi above every entry
    // that found no room keeps its list: the list is the kept set of the
    // overflow policy, in its order.  (A list id's largest phi is taken over
    // the stencil rows' values; rows without the id count as -1, so a list
    // that does not rise above -1 goes to the fix-up.)
    if (!G27 && g.ovf != 0ull) {
        float low = __builtin_huge_valf();
#pragma unroll
        for (int q = 0; q < K; ++q) {
            float best = -__builtin_huge_valf();
#pragma unroll
            for (int s = 0; s < 7; ++s) best = g.v[s][q] > best ? g.v[s][q] : best;
            low = best < low ? best : low;
        }
        const unsigned long long keep = __ballot(low > -1.0f && g.outside < low) & g.ovf;
        nres += (unsigned)__popcll(keep);
        g.ovf &= ~keep;
    }
    // an overflowed point computes nothing here (fix-up kernel)
    const bool st = in_mask(on & ~g.ovf);
    const int nm = list_max(g);
    const int nst = max(nm, D);
    bool skip = false;
    float Up = 0.0f;
    float rw[K];
    if (nm > 0) {
        float T;
        skip = thermal_Tv(a, xi, yj, a.z[k], T);
        Up = T / a.L_cp;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            const float w = g.v[3][q] + 1.0f;
            rw[q] = 0.25f * w * w;
        }
    }
    // each slot's orientation rows are requested while the slot before it is
    // computed
    Rot m[2];
    if (nm > 0) m[0] = slot_rot(a, in_mask(g.filled[0]) ? g.la[0] : 0, g.v[3][0]);
#pragma unroll
    for (int q = 0; q < K; ++q) {
        if (q < nst) {
            int oid = -1;
            float oph = -1.0f;
            const bool in = in_mask(g.filled[q]);
            if (q < nm) {
                if (q + 1 < K && q + 1 < nm)
                    m[(q + 1) & 1] = slot_rot(a, in_mask(g.filled[(q + 1) % K]) ? g.la[(q + 1) % K] : 0,
                                              g.v[3][(q + 1) % K]);
                float repul = 0.0f;  // empty slots add exactly +0
#pragma unroll
                for (int p = 0; p < K; ++p)
                    if (p != q) repul += rw[p];
                const float nv = slot_update_r(a, m[q & 1], g.v[0][q], g.v[1][q], g.v[2][q], g.v[3][q], g.v[4][q],
                                               g.v[5][q], g.v[6][q], repul, Up, a_s, epsv);
                oph = in ? nv : -1.0f;
                oid = in && !(nv < kKillf) ? g.la[q] : -1;
            }
            row_store(a, t, q, st && !(skip && in), oid, oph);
        }
    }
    if (tx >= 0) row_mark_tile(a, r, k, tx, g.ovf != 0ull ? K : nm);
    else row_mark_strip(a, r, k, in_mask(g.ovf) ? K : list_len(g));
    if (g.ovf != 0ull) {
        // the row's, or a strip wave's first
        fixup_append(a, g.ovf, (unsigned)t.zC + (t.c >> 2), __builtin_amdgcn_readfirstlane(r.j), k);
    }
}

template <int K, bool G27>
__device__ __forceinline__ void row_plane(CArgs* args, const RowLane& r, int k, int tx, int P, int D, float xi,
                                          float yj, float a_s, float epsv, unsigned& nres)
{
    int done = 0;
    if (!G27) {
        if (P <= 2) done = narrow_plane<K, 2>(*args_ref(args), r, k, tx, D, xi, yj, a_s, epsv) ? 1 : 0;
        else if (P <= 4) done = narrow_plane<K, 4>(*args_ref(args), r, k, tx, D, xi, yj, a_s, epsv) ? 1 : 0;
        // the general path starts from a clean slate: nothing of the narrow
        // attempt stays in registers for it (177 vector registers otherwise)
        asm volatile("" : "+s"(done));
        if (done) return;
    }
    wide_plane<K, G27>(*args_ref(args), r, k, tx, P, D, xi, yj, a_s, epsv, nres);
}

__device__ __forceinline__ int word_bound(unsigned w, unsigned ep) { return (w >> 4) >= ep ? (int)(w & 15u) : 0; }

// Bounds of the filled slots around a row plane (P: source, its stencil's
// rows; D: the row's own in the destination), wave-uniform.  Words of the
// source's current epoch are the largest, so the maximum of the words holds
// the largest bound.
template <int K, bool G27>
__device__ __forceinline__ void row_bounds(const StepArgs& a, const RowLane& r, int k, int tx, int& P, int& D)
{
    const int jm = bc_map(r.j - 1, a.fny, a.bcy), jp = bc_map(r.j + 1, a.fny, a.bcy);
    const int km = bc_map(k - 1, a.fnz, a.bcz), kp = bc_map(k + 1, a.fnz, a.bcz);
    if (!G27 && tx >= 0) {
        // one row: uniform indices, scalar loads (this launch writes row_dst
        // words only after their own row has read them here)
        typedef const __attribute__((address_space(4))) unsigned CWord;
        CWord* w = (CWord*)a.row_src;
        const int j = __builtin_amdgcn_readfirstlane(r.j);
        const int ujm = __builtin_amdgcn_readfirstlane(jm), ujp = __builtin_amdgcn_readfirstlane(jp);
        const int i0 = 1 + tx * kTX;
        const int xl = act_tile_x(bc_map(i0 - 1, a.fnx, a.bcx));
        const int xr = act_tile_x(bc_map(min(i0 + kTX, a.fnx - 1), a.fnx, a.bcx));
        const int c = (k * a.fny + j) * a.ntx;
        const unsigned d = ((CWord*)a.row_dst)[c + tx];
        const unsigned m0 = max(max(w[c + tx], w[c + xl]), w[c + xr]);
        const unsigned m1 = max(w[(k * a.fny + ujm) * a.ntx + tx], w[(k * a.fny + ujp) * a.ntx + tx]);
        const unsigned m2 = max(w[(km * a.fny + j) * a.ntx + tx], w[(kp * a.fny + j) * a.ntx + tx]);
        P = min(word_bound(max(max(m0, m1), m2), a.ep_src), K);
        D = min(word_bound(d, a.ep_dst), K);
        return;
    }
    const int x = act_tile_x(r.i);
    const int xl = act_tile_x(bc_map(tx >= 0 ? 1 + tx * kTX - 1 : r.i - 1, a.fnx, a.bcx));
    const int xr = act_tile_x(bc_map(tx >= 0 ? min(1 + tx * kTX + kTX, a.fnx - 1) : r.i + 1, a.fnx, a.bcx));
    const unsigned d = a.row_dst[(k * a.fny + r.j) * a.ntx + x];
    unsigned m = 0u;
#pragma unroll
    for (int z = 0; z < 3; ++z) {
        const int kz = (z == 0 ? km : z == 2 ? kp : k) * a.fny;
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            const unsigned* w = a.row_src + (kz + (y == 0 ? jm : y == 2 ? jp : r.j)) * a.ntx;
            if (!G27 && z != 1 && y != 1) continue;
            m = max(m, w[x]);
            if (G27 || (z == 1 && y == 1)) m = max(m, max(w[xl], w[xr]));
        }
    }
    P = min(wave_max<8>(word_bound(m, a.ep_src)), K);
    D = min(wave_max<8>(word_bound(d, a.ep_dst)), K);
}

// One unit of the step: a wave's 64 points (a row of column tile tx, or with
// tx < 0 its part of the strip) over the planes k0 + bit of need.
struct RowUnit {
    int i, j, tx, k0;
    bool on;
    unsigned long long need;
};

// Strip unit s of a simulation (wseg waves per chunk, ex columns).
__device__ __forceinline__ RowUnit strip_unit(const StepArgs& a, int s, int wseg, int ex)
{
    RowUnit u;
    const int zc = s / wseg, seg = s - zc * wseg;
    const int lane = threadIdx.x;
    const int rows = 64 / ex, r0 = lane / ex;
    u.k0 = 1 + zc * a.kchunk;
    u.need = (1ull << (min(u.k0 + a.kchunk, a.fnz - 1) - u.k0)) - 1ull;
    u.tx = -1;
    u.i = a.fnx - 1 - ex + (lane - r0 * ex);
    u.j = 1 + seg * rows + r0;
    u.on = r0 < rows && u.j <= a.fny - 2;
    return u;
}

// Row `row` of listed chunk (item, need) of a simulation.
__device__ __forceinline__ RowUnit tile_unit(const StepArgs& a, int item, unsigned long long need, int row)
{
    RowUnit u;
    const int zc = item / a.items_chunk;
    const int t = item - zc * a.items_chunk;
    const int ty = t / a.tiles_x;
    u.tx = t - ty * a.tiles_x;
    u.k0 = 1 + zc * a.kchunk;
    u.i = 1 + u.tx * kTX + (int)threadIdx.x;
    u.j = 1 + ty * kTY + row;
    u.on = u.i <= a.fnx - 2;
    u.need = u.j <= a.fny - 2 ? need : 0ull;  // a partial tile's rows past the end
    return u;
}

template <int K, bool G27>
__device__ __forceinline__ void row_unit(CArgs* args, const RowUnit& u, unsigned& nres)
{
    const StepArgs& a = *args_ref(args);
    const RowLane r = row_lane(a, min(u.i, a.fnx - 2), min(u.j, a.fny - 2), u.on);
    const float xi = a.x[r.i], yj = a.y[r.j];
    const float a_s = 1.0f + 3.0f * a.kin_delta;
    const float epsv = -4.0f * a.kin_delta / a_s;
#pragma unroll 1
    for (unsigned long long need = u.need; need; need &= need - 1) {
        const StepArgs& b = *args_ref(args);
        const int k = u.k0 + __ffsll((long long)need) - 1;
        int P = K, D = K;
        if (b.use_act) row_bounds<K, G27>(b, r, k, u.tx, P, D);
        if (P + D == 0) continue;
        row_plane<K, G27>(args, r, k, u.tx, P, D, xi, yj, a_s, epsv, nres);
    }
}

}  // namespace

}  // namespace cupf
