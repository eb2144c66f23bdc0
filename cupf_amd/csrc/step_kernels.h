// step_kernels.h -- the step and fix-up kernels (single simulation
// and batched), instantiated once per (K, gather variant) by the step_k*_g*.hip
// files so the large template instantiations compile in parallel.
#pragma once

#include <algorithm>

#include "apt_device.h"
#include "apt_rows.h"

namespace cupf {

namespace {

// A wave's place among W waves that take units u, u + W, ...: kXcdRun
// neighbouring places on one XCD (workgroups go to the 8 XCDs in turn), so that
// the rows of a tile plane and its neighbours in x meet in one L2, and every
// XCD has the same share of a last, partly filled round.  (Runs of 4 / 16 / 64 /
// 128 / 512: 243 / 241 / 249 / 284 / 305 us for the 256x256x512 start-up, 57 /
// 55 / 57 / 64 / 66 at step 1500, 1014 / 1000 / 987 / 987 / 1168 for a solid
// 256^3 window, whose line fetches beyond the L2s fall by 39 %.)
constexpr unsigned kXcdRun = 16u;
__device__ __forceinline__ unsigned row_place(unsigned W)
{
    const unsigned b = blockIdx.x, x = b % 8u, m = b / 8u;
    return W % (8u * kXcdRun) == 0u ? (m / kXcdRun * 8u + x) * kXcdRun + m % kXcdRun : b;
}

// APTrhs_psi (3DgrainMPI/APTPhaseField.cu:178-354) over every interior point:
// one-wave workgroups, a few rounds of them, over units, the strip's first, then
// row r of listed chunk e as unit 4 e + r.  Waves take units by position: an
// atomic claim per unit (or only for the last two rounds) costs ~17 ns each on
// one address, which the start-up's 36,000 row planes of 4 us do not afford
// (256x256x512, before the entries got cheaper: 407 us by position, 498 with
// claims in the last two rounds).
template <int K, bool G27>
__global__ __launch_bounds__(kRowLanes, 4) void apt_step(StepArgs)
{
    CArgs* args = (CArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    const StepArgs& a = *args_ref(args);
    const int ex = strip_width(a.fnx, a.tiles_x);
    const int wseg = strip_waves(ex, a.fny);
    const unsigned ns = (unsigned)(wseg * a.nzchunk);
    const unsigned n = ns + 4u * __atomic_load_n(a.wl_count, __ATOMIC_RELAXED);
    const unsigned W = gridDim.x;
    const unsigned place = row_place(W);
    unsigned nres = 0u;  // overflowed points settled here
#pragma unroll 1
    for (unsigned u = place; u < n; u += W) {
        const StepArgs& b = *args_ref(args);
        RowUnit w;
        if (u < ns) {
            w = strip_unit(b, (int)u, wseg, ex);
        } else {
            const unsigned e = (u - ns) >> 2;
            w = tile_unit(b, b.wl_item[e], b.wl_need[e], (int)((u - ns) & 3u));
        }
        row_unit<K, G27>(args, w, nres);
    }
    if (threadIdx.x == 0 && nres)
        atomicAdd(a.overflow + kLineWords / 2 * (place % kSpread), (unsigned long long)nres);
}

// The units of kPoints list entries that wave w of workgroup blk takes: an
// eighth of the list, in order, for each XCD (workgroups go to the 8 XCDs in
// turn), because the 8 units of a row's 64 points share their neighbours'
// lines; and within the eighth the first wave of every workgroup before the
// second of any, so a short list is spread over the CUs.  (Units in order over
// all workgroups met in no L2: 7.5 M line fetches against 6.3 M, and 130 against
// 119 us, for the 270,000 points of the 256x256x512 start-up.)
struct FixShare {
    unsigned first, end, step;
};
__device__ __forceinline__ FixShare fix_share(unsigned units, int blk, int nblk, int w)
{
    const unsigned X = nblk % 8 == 0 ? 8u : 1u;
    const unsigned x = (unsigned)blk % X, per = (unsigned)nblk / X;
    const unsigned lo = (unsigned)((unsigned long long)units * x / X);
    return {lo + (unsigned)w * per + (unsigned)blk / X, (unsigned)((unsigned long long)units * (x + 1u) / X),
            per * (kFixLanes / 64)};
}

// Fix-up pass for the points of the last apt_step launch whose neighbourhood
// overflowed K slots; adds their number to the overflow diagnostic.  The list
// lives in this step's counter set, which the next-but-one plan kernel
// clears, so nothing here has to wait for the other workgroups.
template <int K, bool G27>
__device__ __forceinline__ void fixup_run(const StepArgs& a, int blk, int nblk)
{
    using F = FixGroup<G27>;
    __shared__ unsigned s_fix[(kFixLanes / F::kLanes) * (kFixStride + F::kIds)];
    __shared__ unsigned s_pre[kSpread + 1], s_cnt[kSpread], s_wave[kFixLanes / 64];
    const unsigned units = fixup_units<F::kPoints>(
        kSpread, [&](int q) { return __atomic_load_n(a.fix_count + kLineWords * q, __ATOMIC_RELAXED); }, s_pre,
        s_cnt, s_wave);
    if (units == 0u) return;
    if (blk == 0 && threadIdx.x < kSpread && s_cnt[threadIdx.x])
        atomicAdd(a.overflow + kLineWords / 2 * threadIdx.x, (unsigned long long)s_cnt[threadIdx.x]);
    const float a_s = 1.0f + 3.0f * a.kin_delta;
    const float epsv = -4.0f * a.kin_delta / a_s;
    const int l = threadIdx.x & (F::kLanes - 1), grp = threadIdx.x / F::kLanes;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const FixShare sh = fix_share(units, blk, nblk, w);
#pragma unroll 1
    for (unsigned u = sh.first; u < sh.end; u += sh.step) {
        const int seg = fixup_find(s_pre, kSpread, u);
        const unsigned e0 = (u - s_pre[seg]) * F::kPoints;
        const unsigned e = e0 + (unsigned)(grp & (F::kPoints - 1));
        const bool on = e < s_cnt[seg];
        const unsigned* list = a.fix_list + fix_segment_base(seg, 0, a.fix_cap);
        fixup_group<K, G27>(a, list[on ? e : e0], on, l, s_fix + grp * (kFixStride + F::kIds), a_s, epsv);
    }
}

// Waves per SIMD that the registers of the 7-point fix-up have to leave room
// for: as many as its LDS lets in (unasked, the cold NaN branch took 8 more
// vector registers, 78, and a wave away).  The 27-point kernels get there by
// themselves (94 registers at K = 5) or not at all (143 at K = 8).
constexpr int fix_waves(bool g27) { return g27 ? 1 : 7; }

template <int K, bool G27>
__global__ __launch_bounds__(kFixLanes, fix_waves(G27)) void apt_fixup(StepArgs)
{
    CArgs* a = (CArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    fixup_run<K, G27>(*args_ref(a), (int)blockIdx.x, (int)gridDim.x);
}

// The fix-up of one step and the work-list plan of the next in one launch:
// blocks [0, fa.fix_blocks) run the fix-up with fa, the others the plan with
// pa.  The plan reads only activity words, which the fix-up does not write
// (the step kernel marks an overflowed point's tile), and the fix-up reads
// its own step's counter set while the plan fills the next one and clears
// the one after (three sets in turn), so the two halves need no order
// between them.  Saves one launch and its dispatch gap per step.
template <int K, bool G27>
__global__ __launch_bounds__(kBlock, fix_waves(G27)) void apt_fixplan(StepArgs, StepArgs)
{
    static_assert(kFixLanes == kBlock, "one workgroup size for both halves");
    CArgs* args = (CArgs*)__builtin_amdgcn_kernarg_segment_ptr();  // fa, pa
    const int nfix = args[0].fix_blocks;
    if ((int)blockIdx.x < nfix) fixup_run<K, G27>(*args_ref(args), (int)blockIdx.x, nfix);
    else plan_block(*args_ref(args + 1), (int)blockIdx.x - nfix);
}

// Batched APTrhs_psi: the strip units of every simulation, then the rows of
// the chunks the batched plan kernel listed, each with its own simulation's
// step arguments (batch_advance rewrites them only after this kernel).
template <int K, bool G27>
__global__ __launch_bounds__(kRowLanes, 4) void batch_step(BatchArgs b)
{
    typedef const __attribute__((address_space(4))) BatchSim CSim;
    const CSim* sims = (const CSim*)b.sims;
    const unsigned* cnt = b.cnt + 4 * __atomic_load_n(b.cnt + 8, __ATOMIC_RELAXED);
    const unsigned ns = (unsigned)b.strip_total;
    const unsigned n = ns + 4u * __atomic_load_n(cnt, __ATOMIC_RELAXED);
    const unsigned W = gridDim.x;
#pragma unroll 1
    for (unsigned u = row_place(W); u < n; u += W) {
        unsigned nres = 0u;
        int sim;
        RowUnit w;
        if (u < ns) {
            int lo = 0, hi = b.n - 1;  // last simulation whose units start at or before u
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (sims[mid].strip_base <= (int)u) lo = mid;
                else hi = mid - 1;
            }
            sim = lo;
            const StepArgs& a = *(const StepArgs*)&sims[sim].a;
            const int ex = strip_width(a.fnx, a.tiles_x);
            w = strip_unit(a, (int)u - sims[sim].strip_base, strip_waves(ex, a.fny), ex);
        } else {
            const unsigned e = (u - ns) >> 2;
            sim = __builtin_amdgcn_readfirstlane(b.wl_sim[e]);
            w = tile_unit(*(const StepArgs*)&sims[sim].a, b.wl_item[e], b.wl_need[e], (int)((u - ns) & 3u));
        }
        row_unit<K, G27>((CArgs*)&sims[sim].a, w, nres);
        if (threadIdx.x == 0 && nres)
            atomicAdd(sims[sim].a.overflow + kLineWords / 2 * (u % kSpread), (unsigned long long)nres);
    }
}

// Batched fix-up: the list segments of all simulations (fix_segs each) form
// one index space of wave units (prefix sums in LDS) that the grid strides
// over, so long and short lists alike are spread over every workgroup.
// (Four waves per SIMD: 126 registers for 27 points at K = 8, 138 unasked.)
template <int K, bool G27>
__global__ __launch_bounds__(kFixLanes, 4) void batch_fixup(BatchArgs b)
{
    using F = FixGroup<G27>;
    __shared__ unsigned s_fix[(kFixLanes / F::kLanes) * (kFixStride + F::kIds)];
    __shared__ unsigned s_pre[kMaxBatch + 1], s_cnt[kMaxBatch], s_wave[kFixLanes / 64];
    typedef const __attribute__((address_space(4))) BatchSim CSim;
    const CSim* sims = (const CSim*)b.sims;
    const int segs = b.fix_segs, m = b.n * segs;
    const unsigned units = fixup_units<F::kPoints>(
        m,
        [&](int q) {
            return __atomic_load_n(b.sims[q / segs].a.fix_count + kLineWords * (q % segs), __ATOMIC_RELAXED);
        },
        s_pre, s_cnt, s_wave);
    if (blockIdx.x == 0)
        for (int q = threadIdx.x; q < m; q += kFixLanes)
            if (s_cnt[q])
                atomicAdd(b.sims[q / segs].a.overflow + kLineWords / 2 * (q % segs), (unsigned long long)s_cnt[q]);
    const int l = threadIdx.x & (F::kLanes - 1), grp = threadIdx.x / F::kLanes;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const FixShare sh = fix_share(units, (int)blockIdx.x, (int)gridDim.x, w);
#pragma unroll 1
    for (unsigned u = sh.first; u < sh.end; u += sh.step) {
        const int q = fixup_find(s_pre, m, u);
        const StepArgs& a = *(const StepArgs*)&sims[q / segs].a;
        const unsigned e0 = (u - s_pre[q]) * F::kPoints;
        const unsigned e = e0 + (unsigned)(grp & (F::kPoints - 1));
        const float a_s = 1.0f + 3.0f * a.kin_delta;
        const float epsv = -4.0f * a.kin_delta / a_s;
        const bool on = e < s_cnt[q];
        const unsigned* list = a.fix_list + fix_segment_base(q % segs, a.fix_shift, a.fix_cap);
        fixup_group<K, G27>(a, list[on ? e : e0], on, l, s_fix + grp * (kFixStride + F::kIds), a_s, epsv);
    }
}

template <int K, bool G27>
hipError_t launch_step_t(const StepArgs& a, hipStream_t stream, hipEvent_t ev_begin, hipEvent_t ev_planned,
                         hipEvent_t ev_mid, hipEvent_t ev_end, bool planned, const StepArgs* next)
{
    if (ev_begin) (void)hipEventRecord(ev_begin, stream);
    hipError_t e;
    if (!planned && (e = launch_plan(a, stream)) != hipSuccess) return e;
    if (ev_planned) (void)hipEventRecord(ev_planned, stream);
    hipLaunchKernelGGL((apt_step<K, G27>), dim3(a.step_blocks), dim3(kRowLanes), 0, stream, a);
    if (ev_mid) (void)hipEventRecord(ev_mid, stream);
    if (next) {  // this step's fix-up and the next step's plan in one launch
        const int pblocks = max(1, cdiv(plan_waves(next->kchunk, next->nzchunk, next->items_chunk), kBlock / 64));
        hipLaunchKernelGGL((apt_fixplan<K, G27>), dim3(a.fix_blocks + pblocks), dim3(kBlock), 0, stream, a, *next);
    } else {
        hipLaunchKernelGGL((apt_fixup<K, G27>), dim3(a.fix_blocks), dim3(kFixLanes), 0, stream, a);
    }
    if (ev_end) (void)hipEventRecord(ev_end, stream);
    return hipGetLastError();
}

template <int K, bool G27>
hipError_t launch_batch_t(const BatchArgs& b, hipStream_t stream)
{
    hipError_t e = launch_batch_plan(b, stream);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((batch_step<K, G27>), dim3(b.step_blocks), dim3(kRowLanes), 0, stream, b);
    hipLaunchKernelGGL((batch_fixup<K, G27>), dim3(b.fix_blocks), dim3(kFixLanes), 0, stream, b);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_batch_advance(b, stream);
}

// Workgroups that fit the device at once: which = 0 step, 1 batched step,
// 2 fix-up, 3 batched fix-up.
template <int K, bool G27>
int slots_t(int device, int which)
{
    int ncu = 0, per = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return 0;
    hipError_t e;
    switch (which) {
    case 0: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, apt_step<K, G27>, kRowLanes, 0); break;
    case 1: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, batch_step<K, G27>, kRowLanes, 0); break;
    case 2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, apt_fixup<K, G27>, kFixLanes, 0); break;
    default: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, batch_fixup<K, G27>, kFixLanes, 0); break;
    }
    if (e != hipSuccess || per < 1) return 0;
    return per * ncu;
}

}  // namespace

}  // namespace cupf
