// apt_internal.h -- device-side argument blocks shared by the kernels and the
// C-ABI layer of cupf_amd.  Not part of the public interface.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "capacity.h"

namespace cupf {

// LS = -0.995 (3DgrainMPI/APTPhaseField.cu:25) is a double literal in the
// reference: every `phi > LS` test compares in double.
constexpr double kLS = -0.995;
// The same comparison and that with the slot kill threshold -0.9999
// (3DgrainMPI/APTPhaseField.cu:341, also a double) in float, exact for every
// float x: (double)x > -0.995 <=> x > -0.995f, because -0.995f is the largest
// float not above -0.995; (double)x < -0.9999 <=> x < -0.9999f, because -0.9999f
// is the smallest float not below -0.9999 (checked exhaustively on [-1, -0.99]
// by tests/test_oracle.py).
constexpr float kLSf = -0.995f;
constexpr float kKillf = -0.9999f;

// Leftover columns at the +x end narrower than this form a strip, whose rows
// share waves (64 / width rows each); wider ones form a partial tile, one row
// per wave.
constexpr int kPartialMin = 16;

// Atomics of a whole grid on one address go through one at a time, ~17 ns each
// (the start-up of a 256x256x512 simulation hands over points from ~25,000 row
// planes of a 400 us step), so the fix-up list and the overflow count are
// spread over kSpread counters on cache lines of their own: the list's by
// equal shares of the rows, y-major (capacity.h).  (One counter each
// before; step kernel at step 6: 400 -> 266 us; 64^3 at step 10 45 -> 34; the
// 27-point gather at 96x96x128 115 -> 80.)
constexpr int kSpread = 64;
constexpr int kLineWords = 32;             // 128 bytes
constexpr int kWlWord = kSpread * kLineWords;           // a set's work-list counter
constexpr int kSetWords = (kSpread + 1) * kLineWords;   // a step's counter set
// Counters over all members of a batch (kMaxBatch at most).
constexpr int kBatchSpread = 256;

// Everything one APT step launch reads.  Passed by value (kernel argument
// segment -> SGPRs), so no constant-memory upload per step.
struct StepArgs {
    const float* ph;       // source buffer, K slot planes
    const int* arg;
    float* ph_new;         // destination buffer
    int* arg_new;
    const float* x;
    const float* y;
    const float* z;
    const float* R12;      // orientation rows, 12 floats per grain (9 used)
    const float* psi_mac;  // type-4 thermal field
    unsigned long long* overflow;  // points with > K distinct ids: the sum of kSpread counts,
                                   // kLineWords / 2 apart
    // Interior points left to the fix-up pass: 64 equal parts of fix_cap entries
    // by the index of a row plane (capacity.h), a segment of the list each, or
    // (a batch) 2^fix_shift of them to a segment.
    unsigned* fix_list;
    int fix_shift;
    unsigned fix_cap;
    // Counters of this step: fix_count[kLineWords * s] entries in segment s;
    // wl_count (below) points into the same set (kSetWords).  Steps take three sets in turn;
    // cnt_next is the next step's, cleared by this step's plan kernel (its
    // last user, two steps back, has finished; this step's fix-up, which may
    // run beside the next step's plan, keeps its own).
    unsigned* fix_count;
    unsigned* cnt_next;
    // Activity map: one word per (column tile, z plane) and buffer.  A tile
    // plane of a buffer may hold a slot other than the empty pair (-1, -1.0f)
    // only if its word is >= that buffer's epoch.  Epochs come from one
    // increasing counter, so stale words never need clearing.
    const unsigned* act_src;
    unsigned* act_dst;
    unsigned ep_src;       // epoch of the source buffer
    unsigned ep_dst;       // epoch the destination buffer had before this step
    unsigned ep_new;       // epoch the destination buffer gets from this step
    int use_act;           // 0: process every plane (the map is still maintained)
    // unused0 and unused1 keep the fields behind them where scalar loads fetch
    // several at once (apt_step without them: 43.6 us in place of 42.9 for
    // 139x74x101 in a cylinder's field, 21.1 in place of 20.9 at 64^3).
    int ntx, unused0, ntiles;  // activity tiles in x and in all (64x4, partial ones included)
    // Row map: one word per (row of a column tile, z plane) and buffer, epoch
    // << 4 | bound.  A row of a buffer may hold anything but empty pairs only
    // if its word's epoch is >= the buffer's, and then only in slots below
    // the bound.  Index (k * fny + j) * ntx + column tile.
    const unsigned* row_src;
    unsigned* row_dst;
    // Work of one step: the strip's units (see apt_step), then the tile chunks
    // listed by the plan kernel: wl_item = z chunk * items_chunk + tile, with
    // the chunk's plane mask, wl_count[0] of them (word kWlWord of the counter set).
    int* wl_item;
    unsigned long long* wl_need;
    unsigned* wl_count;
    int items_chunk;       // tiles per z chunk
    int step_blocks;       // one-wave workgroups of the step kernel
    int fix_blocks;        // workgroups of the overflow fix-up kernel
    int fnx, fny, fnz;
    int L;                 // slot stride fnx*fny*fnz
    int nzchunk, kchunk;   // z-chunks per column, planes per chunk
    int tiles_x, unused1;  // 64x4 column tiles in x (one partial at the +x end included;
                           // see kPartialMin)
    int bcx, bcy, bcz;
    int num_theta;
    int thermal_type;
    int use_iuc;
    float t;
    float dt, hi, lamd, L_cp, kin_delta, eps;
    float G, R, uc, uc0, z0, r0, lyd, lzd, V, mp_len, x0, order;
    float tan_angle, cos_angle;
    int Nx, Ny, Nz;
    float X0_mac, Y0_mac, Z0_mac, Dx_mac;
};

// One simulation of a batch, in device memory.  `a` holds the arguments of
// its next step; after every step the advance kernel swaps the buffers, moves
// the epochs and the step index and recomputes t, exactly as the host does
// between two single-simulation launches.
struct BatchSim {
    StepArgs a;
    float* ph[2];
    int* arg[2];
    unsigned* act[2];
    unsigned* row[2];
    unsigned ep[2];        // epochs of the two buffers
    unsigned ep_ctr;       // epoch counter of the simulation
    int cur;               // source buffer of the next step
    int step;              // index s of the next step (t = (float)s*dt*tau0)
    int parity;            // counter set of the next step (0..2, in turn)
    unsigned* cnt;         // the simulation's three counter sets
    float tau0;
    int plan_base;         // first plan wave of this simulation
    int strip_base;        // first strip unit of this simulation
};

// Plan waves: a wave's 64 lanes cover plan_tiles tiles, plan_rows lanes (z
// planes) each: a group of plan_group z chunks plus one halo plane at each
// end (kchunk <= 61).
__host__ __device__ inline int plan_rows(int kchunk) { return kchunk <= 14 ? 16 : (kchunk <= 30 ? 32 : 64); }
__host__ __device__ inline int plan_tiles(int kchunk) { return 64 / plan_rows(kchunk); }
__host__ __device__ inline int plan_group(int kchunk) { return (plan_rows(kchunk) - 2) / kchunk; }
// Plan waves of a simulation with nzchunk chunks of items_chunk tiles.
__host__ __device__ inline int plan_waves(int kchunk, int nzchunk, int items_chunk)
{
    const int g = plan_group(kchunk), tw = plan_tiles(kchunk);
    return ((nzchunk + g - 1) / g) * ((items_chunk + tw - 1) / tw);
}

// Waves of the +x strip per z chunk: ex columns of fny - 2 rows (ex <= 0: no
// strip), 64 / ex rows to a wave.
__host__ __device__ inline int strip_width(int fnx, int tiles_x) { return (fnx - 2) - 64 * tiles_x; }
__host__ __device__ inline int strip_waves(int ex, int fny)
{
    return ex > 0 ? (fny - 2 + 64 / ex - 1) / (64 / ex) : 0;
}

// Most simulations one batch may hold.
constexpr int kMaxBatch = 1024;

// A batched step over n simulations sharing K and the gather variant.  The
// work list holds tile chunks of every simulation; cnt holds the chunks listed
// by alternate steps (words 0 and 4), selected by cnt[8].
struct BatchArgs {
    BatchSim* sims;
    int n;
    int plan_total;        // waves of the plan kernel (all simulations)
    int strip_total;       // strip units of all simulations
    int* wl_sim;
    int* wl_item;
    unsigned long long* wl_need;
    unsigned* cnt;
    int fix_segs;          // fix-up list segments of each simulation
    int step_blocks;
    int fix_blocks;        // workgroups of the batched fix-up kernel
};

// Nucleation launch block (3DgrainMPI/APTPhaseField.cu:459-536).
struct NuclArgs {
    float* ph;
    int* arg;
    int* status;
    const float* x;
    const float* y;
    const float* z;
    const float* T3d;
    const float* ball;     // (2p+1)^3 tanh template
    unsigned long long* events;
    unsigned* act;         // activity and row maps of the buffer nucleated into, and its epoch
    unsigned* row;
    unsigned ep;
    int ntx, ntiles;
    int fnx, fny, fnz, L, K;
    int cnx, cny, cnz, p;
    int use_iuc;
    float t, dt;
    float uc0, undcool_mean, undcool_std, nuc_Nmax, nuc_Nmax0, nuc_rad;
    int Nx, Ny, Nz, Nt;
    float X0_mac, Y0_mac, Z0_mac, t0_mac, Dx_mac, Dt_mac;
    uint64_t seed;
    uint64_t call;
};

// Launchers (apt_misc.hip, step_k*_g*.hip).  All enqueue on
// `stream` and return the hipError_t of the launch.
// Step waves launched per wave that fits the device: the dispatcher gives a CU
// whose wave has ended the next one, which evens out units of unequal cost (a
// grid of only the waves that fit, each with its share of the units, had its
// waves done for 10 % of the launch on average); a wave that finds no unit
// costs ~0.17 ns.  Rounds 1 / 2 / 4 / 6 / 8 / 16 / 64: 256x256x512 at step 150
// 155 / 154 / 140 / 136 / 138 / 135 / 172 us, at step 450 36 / 34 / 33 / 34 /
// 34 / 40 / 81; 78 % solid 256^3 window 1003 / 998 / 988 / 983 / 972 / 961 / 994.
constexpr int kStepRounds = 6;

// Workgroups of the step kernel that fit the device at once.
int step_kernel_slots(int K, int gather27, int device);
int batch_kernel_slots(int K, int gather27, int device);
// Workgroups of the (single or batched) overflow fix-up kernel that fit at once.
int fixup_kernel_slots(int K, int gather27, int device, bool batch);
// Batched step: plan, step, fix-up and advance kernels.
hipError_t launch_batch_step(const BatchArgs& b, int K, int gather27, hipStream_t stream);
// Pieces shared by the per-K launchers.
hipError_t launch_plan(const StepArgs& a, hipStream_t stream);
hipError_t launch_batch_plan(const BatchArgs& b, hipStream_t stream);
hipError_t launch_batch_advance(const BatchArgs& b, hipStream_t stream);
hipError_t launch_step_k5_g7(const StepArgs& a, hipStream_t stream,
                             hipEvent_t e0, hipEvent_t e1, hipEvent_t e2, hipEvent_t e3,
                             bool planned, const StepArgs* next);
hipError_t launch_batch_k5_g7(const BatchArgs& b, hipStream_t stream);
int step_slots_k5_g7(int device, int which);
hipError_t launch_step_k5_g27(const StepArgs& a, hipStream_t stream,
                             hipEvent_t e0, hipEvent_t e1, hipEvent_t e2, hipEvent_t e3,
                             bool planned, const StepArgs* next);
hipError_t launch_batch_k5_g27(const BatchArgs& b, hipStream_t stream);
int step_slots_k5_g27(int device, int which);
hipError_t launch_step_k8_g7(const StepArgs& a, hipStream_t stream,
                             hipEvent_t e0, hipEvent_t e1, hipEvent_t e2, hipEvent_t e3,
                             bool planned, const StepArgs* next);
hipError_t launch_batch_k8_g7(const BatchArgs& b, hipStream_t stream);
int step_slots_k8_g7(int device, int which);
hipError_t launch_step_k8_g27(const StepArgs& a, hipStream_t stream,
                             hipEvent_t e0, hipEvent_t e1, hipEvent_t e2, hipEvent_t e3,
                             bool planned, const StepArgs* next);
hipError_t launch_batch_k8_g27(const BatchArgs& b, hipStream_t stream);
int step_slots_k8_g27(int device, int which);
// Work-list plan (unless `planned`: the previous launch's apt_fixplan made
// it), main step kernel, then the overflow fix-up, or with `next` the fix-up
// together with the plan of the step `next` describes (apt_fixplan).
// Optional events are recorded before the plan, after it, after the main
// kernel and after the fix-up.
hipError_t launch_step(const StepArgs& a, int K, int gather27, hipStream_t stream,
                       hipEvent_t ev_begin = nullptr,
                       hipEvent_t ev_planned = nullptr, hipEvent_t ev_mid = nullptr,
                       hipEvent_t ev_end = nullptr, bool planned = false,
                       const StepArgs* next = nullptr);
// Device-side QoIs on a collected alpha field (qoi.hip).
hipError_t launch_qoi_volume(const int* alpha, int fnx, int fny, int fnz, int max_id, int* counts,
                             int* first, unsigned long long* above, hipStream_t stream);
// Junction rows in scan order: count pass into blk_cnt, scan into blk_off and
// *count, then (cap > 0) the rows; blk_cnt/blk_off hold qoi_junction_blocks words.
int qoi_junction_blocks(int fnx, int fny, int fnz);
hipError_t launch_qoi_junctions(const int* alpha, int fnx, int fny, int fnz, unsigned* blk_cnt,
                                unsigned* blk_off, int* rows, int cap, unsigned* count,
                                hipStream_t stream);
hipError_t launch_qoi_liquid_planes(const int* alpha, int fnx, int fny, int fnz, unsigned* liq,
                                   hipStream_t stream);
hipError_t launch_qoi_area(const int* alpha, int fnx, int fny, int fnz, int ng, int tip, int* total,
                           int* extra, hipStream_t stream);
hipError_t launch_bc_fill(float* ph, int* arg, int fnx, int fny, int fnz, int K, int bcx,
                          int bcy, int bcz, hipStream_t stream);
// The buffer's row words for launch_collect (row = nullptr: every slot is
// read); halo: it was filled from the buffer as it is.
struct CollectRows {
    const unsigned* row;
    unsigned ep;
    int halo;
    int fnx, fny, fnz, bcx, bcy, bcz, ntx;
};
hipError_t launch_collect(const float* ph, const int* arg, float* phi, int* alpha, int L, int K,
                          int clear_alpha, const CollectRows& rows, hipStream_t stream);
// Both buffers' maps (activity and row words, new epochs), marked while the
// buffers are initialised.
struct IniMaps {
    unsigned* act[2];
    unsigned* row[2];
    unsigned ep[2];
    int fnx, fny, fnz, ntx, ntiles;
};
hipError_t launch_ini(float* ph0, int* arg0, float* ph1, int* arg1, const float* phi0,
                      const int* alpha0, int L, int K, const IniMaps& maps, hipStream_t stream);
// Exact sums of planes k_from .. k_to-1 into sums[k_from .. k_to) (the rest untouched).
hipError_t launch_plane_sums(const float* ph, long long* sums, int fnx, int fny, int fnz, int K,
                             int k_from, int k_to, hipStream_t stream);
hipError_t launch_move_frame(float* ph_old, int* arg_old, float* ph_new, int* arg_new, float* z,
                             float* zbuf, const int* alpha, int* alpha_full, int* loss_area,
                             int move_count, int fnx, int fny, int fnz, int K, int num_theta,
                             hipStream_t stream);
hipError_t launch_nucl_status(const float* phi0, int* status, int cnx, int cny, int cnz, int p,
                              int fnx, int fny, hipStream_t stream);
hipError_t launch_nucl(const NuclArgs& a, hipStream_t stream);
// Activity and row maps of one buffer from its contents: every tile plane and
// row holding a non-empty slot gets `ep` (the row with its bound).
hipError_t launch_act_rebuild(const float* ph, const int* arg, unsigned* act, unsigned* row, unsigned ep, int fnx,
                              int fny, int fnz, int K, int ntx, int ntiles, hipStream_t stream);
hipError_t launch_copy(const void* src, void* dst, size_t bytes, hipStream_t stream);

}  // namespace cupf
