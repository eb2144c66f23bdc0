// step_kernels.h -- the persistent step and fix-up kernels (single simulation
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
// XCD has the same share of a last, partly filled round.  (1 / 4 / 16: 407 /
// 405 / 401 us for the 256x256x512 start-up, 79 / 79 / 77 us at step 1500; one
// run of W / 8 per XCD: 460 and 86 us, the last round falls on few XCDs.)
constexpr unsigned kXcdRun = 16u;
__device__ __forceinline__ unsigned row_place(unsigned W)
{
    const unsigned b = blockIdx.x, x = b % 8u, m = b / 8u;
    return W % (8u * kXcdRun) == 0u ? (m / kXcdRun * 8u + x) * kXcdRun + m % kXcdRun : b;
}

// APTrhs_psi (3DgrainMPI/APTPhaseField.cu:178-354) over every interior point:
// a persistent grid of one-wave workgroups over units, the strip's first, then
// row r of listed chunk e as unit 4 e + r.  Waves take units by position: an
// atomic claim per unit (or only for the last two rounds) costs ~17 ns each on
// one address, which the start-up's 36,000 row planes of 4 us do not afford
// (256x256x512: 407 us by position, 498 with claims in the last two rounds).
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
    unsigned nres = 0u;  // overflowed points settled here
#pragma unroll 1
    for (unsigned u = row_place(W); u < n; u += W) {
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
    if (threadIdx.x == 0 && nres) atomicAdd(a.overflow, (unsigned long long)nres);
}

// Fix-up pass for the points of the last apt_step launch whose neighbourhood
// overflowed K slots; adds their number to the overflow diagnostic.  The list
// lives in this step's counter set, which the next-but-one plan kernel
// clears, so nothing here has to wait for the other workgroups.
template <int K, bool G27>
__device__ __forceinline__ void fixup_run(const StepArgs& a, int blk, int nblk)
{
    const unsigned n = __atomic_load_n(a.fix_count, __ATOMIC_RELAXED);
    if (n == 0u) return;
    if (blk == 0 && threadIdx.x == 0) atomicAdd(a.overflow, (unsigned long long)n);
    const float a_s = 1.0f + 3.0f * a.kin_delta;
    const float epsv = -4.0f * a.kin_delta / a_s;
    using F = FixGroup<G27>;
    __shared__ unsigned s_fix[(kFixLanes / F::kLanes) * kFixStride];
    const int l = threadIdx.x & (F::kLanes - 1), grp = threadIdx.x / F::kLanes;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // wave units of kPoints entries, the first of every workgroup before the
    // second of any, so a short list is spread over the CUs
#pragma unroll 1
    for (unsigned u = (unsigned)(w * nblk + blk); u * F::kPoints < n; u += (unsigned)(nblk * (kFixLanes / 64))) {
        const unsigned e = u * F::kPoints + (unsigned)(grp & (F::kPoints - 1));
        const bool on = e < n;
        fixup_group<K, G27>(a, a.fix_list[on ? e : u * F::kPoints], on, l, s_fix + grp * kFixStride, a_s, epsv);
    }
}

template <int K, bool G27>
__global__ __launch_bounds__(kFixLanes) void apt_fixup(StepArgs a)
{
    fixup_run<K, G27>(a, (int)blockIdx.x, (int)gridDim.x);
}

// The fix-up of one step and the work-list plan of the next in one launch:
// blocks [0, fa.fix_blocks) run the fix-up with fa, the others the plan with
// pa.  The plan reads only activity words, which the fix-up does not write
// (the step kernel marks an overflowed point's tile), and the fix-up reads
// its own step's counter set while the plan fills the next one and clears
// the one after (three sets in turn), so the two halves need no order
// between them.  Saves one launch and its dispatch gap per step.
template <int K, bool G27>
__global__ __launch_bounds__(kBlock) void apt_fixplan(StepArgs fa, StepArgs pa)
{
    static_assert(kFixLanes == kBlock, "one workgroup size for both halves");
    if ((int)blockIdx.x < fa.fix_blocks) fixup_run<K, G27>(fa, (int)blockIdx.x, fa.fix_blocks);
    else plan_block(pa, (int)blockIdx.x - fa.fix_blocks);
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
        if (threadIdx.x == 0 && nres) atomicAdd(sims[sim].a.overflow, (unsigned long long)nres);
    }
}

// Batched fix-up: the overflow lists of all simulations form one index space
// (prefix sums of their lengths, in LDS) that the grid strides over, so long
// and short lists alike are spread over every workgroup.
template <int K, bool G27>
__global__ __launch_bounds__(kFixLanes) void batch_fixup(BatchArgs b)
{
    using F = FixGroup<G27>;
    __shared__ unsigned s_fix[(kFixLanes / F::kLanes) * kFixStride];
    __shared__ unsigned s_pre[kMaxBatch + 1];  // wave units of the simulations before each
    for (int t = threadIdx.x; t < b.n; t += kFixLanes)
        s_pre[t + 1] = __atomic_load_n(b.sims[t].a.fix_count, __ATOMIC_RELAXED);
    __syncthreads();
    if (threadIdx.x == 0) {
        s_pre[0] = 0u;
        for (int t = 0; t < b.n; ++t) {
            const unsigned c = s_pre[t + 1];
            if (blockIdx.x == 0 && c) atomicAdd(b.sims[t].a.overflow, (unsigned long long)c);
            s_pre[t + 1] = s_pre[t] + (c + F::kPoints - 1) / F::kPoints;
        }
    }
    __syncthreads();
    const unsigned units = s_pre[b.n];
    const int l = threadIdx.x & (F::kLanes - 1), grp = threadIdx.x / F::kLanes;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    typedef const __attribute__((address_space(4))) BatchSim CSim;
    const CSim* sims = (const CSim*)b.sims;
#pragma unroll 1
    for (unsigned u = (unsigned)(w * (int)gridDim.x + (int)blockIdx.x); u < units;
         u += (unsigned)((int)gridDim.x * (kFixLanes / 64))) {
        int lo = 0, hi = b.n - 1;  // last simulation whose units start at or before u
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_pre[mid] <= u) lo = mid;
            else hi = mid - 1;
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        const StepArgs& a = *(const StepArgs*)&sims[lo].a;
        const unsigned n = __atomic_load_n(a.fix_count, __ATOMIC_RELAXED);
        const unsigned e0 = (u - s_pre[lo]) * F::kPoints;
        const unsigned e = e0 + (unsigned)(grp & (F::kPoints - 1));
        const float a_s = 1.0f + 3.0f * a.kin_delta;
        const float epsv = -4.0f * a.kin_delta / a_s;
        const bool on = e < n;
        fixup_group<K, G27>(a, a.fix_list[on ? e : e0], on, l, s_fix + grp * kFixStride, a_s, epsv);
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
