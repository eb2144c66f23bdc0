// apt_device.h -- device code of the APT step shared by the kernel translation
// units (included by apt_misc.hip and step_k*.hip; internal linkage).
//
// Field layout (3DgrainMPI/devicefunc.cu_inl:24-29): SoA slot planes,
// element (i,j,k,slot) at i + j*fnx + k*fnx*fny + slot*L, phi float32 and
// grain id int32 in separate arrays, -1 = empty slot.
//
// Arithmetic follows the reference source operation by operation (build with
// -ffp-contract=off): float everywhere except the reference's implicit double
// promotions (the 1e6 thermal factors, LS=-0.995 and the -0.9999 kill test).
#pragma once

#include "apt_internal.h"

namespace cupf {

namespace {

constexpr int kBlock = 256;        // 4 wave64 per workgroup
constexpr int kFixLanes = 256;     // fix-up workgroup

// Halo index -> interior source index along one axis (APTsetBC3D,
// 3DgrainMPI/APTPhaseField.cu:111-112,134-135,157-158): no-flux mirrors
// out[0]=in[2], out[n-1]=in[n-3]; periodic wraps out[0]=in[n-2], out[n-1]=in[1].
__device__ __forceinline__ int bc_map(int q, int n, int periodic)
{
    if (q == 0) return periodic ? n - 2 : 2;
    if (q == n - 1) return periodic ? 1 : n - 3;
    return q;
}

// kine_ani (3DgrainMPI/APTPhaseField.cu:36-52) with a row-major rotation;
// each row is (m0*ux + m1*uy) + m2*uz, which equals the reference's angle
// form bit for bit (a - b*c == a + (-b)*c; the "+ 0" only flips signs of zeros
// that are squared away).
__device__ __forceinline__ float kine_ani(float ux, float uy, float uz, float m0, float m1,
                                          float m2, float m3, float m4, float m5, float m6,
                                          float m7, float m8, float a_s, float epsv, float eps)
{
    float ux2 = m0 * ux + m1 * uy + m2 * uz;
    ux2 = ux2 * ux2;
    float uy2 = m3 * ux + m4 * uy + m5 * uz;
    uy2 = uy2 * uy2;
    float uz2 = m6 * ux + m7 * uy + m8 * uz;
    uz2 = uz2 * uz2;
    float mag = ux2 + uy2 + uz2;
    float mag2 = mag * mag;
    if (mag > eps) return a_s * (1.0f + epsv * (ux2 * ux2 + uy2 * uy2 + uz2 * uz2) / mag2);
    return 1.0f;
}

// interp3Dtemperature (3DgrainMPI/devicefunc.cu_inl:85-125), indices clamped
// into the macro grid (the reference reads out of bounds there).
__device__ __forceinline__ float interp3(const float* __restrict__ u, float x, float y, float z,
                                         int Nx, int Ny, int Nz, float Dx)
{
    int kx = (int)(x / Dx), ky = (int)(y / Dx), kz = (int)(z / Dx);
    float dx = x / Dx - kx, dy = y / Dx - ky, dz = z / Dx - kz;
    if (kx == Nx - 1) { kx = Nx - 2; dx = 1.0f; }
    if (ky == Ny - 1) { ky = Ny - 2; dy = 1.0f; }
    if (kz == Nz - 1) { kz = Nz - 2; dz = 1.0f; }
    kx = min(max(kx, 0), Nx - 2);
    ky = min(max(ky, 0), Ny - 2);
    kz = min(max(kz, 0), Nz - 2);
    int o = kx + ky * Nx + kz * Nx * Ny;
    int on = kx + ky * Nx + (kz + 1) * Nx * Ny;
    return ((1.0f - dx) * (1.0f - dy) * u[o] + (1.0f - dx) * dy * u[o + Nx]
            + dx * (1.0f - dy) * u[o + 1] + dx * dy * u[o + Nx + 1]) * (1.0f - dz)
         + ((1.0f - dx) * (1.0f - dy) * u[on] + (1.0f - dx) * dy * u[on + Nx]
            + dx * (1.0f - dy) * u[on + 1] + dx * dy * u[on + Nx + 1]) * dz;
}

// interp4Dtemperature (3DgrainMPI/devicefunc.cu_inl:32-83), clamped likewise.
__device__ __forceinline__ float interp4(const float* __restrict__ u, float x, float y, float z,
                                         float t, int Nx, int Ny, int Nz, int Nt, float Dx,
                                         float Dt)
{
    int kx = (int)(x / Dx), ky = (int)(y / Dx), kz = (int)(z / Dx), kt = (int)(t / Dt);
    float dx = x / Dx - kx, dy = y / Dx - ky, dz = z / Dx - kz, dt = t / Dt - kt;
    if (kx == Nx - 1) { kx = Nx - 2; dx = 1.0f; }
    if (ky == Ny - 1) { ky = Ny - 2; dy = 1.0f; }
    if (kz == Nz - 1) { kz = Nz - 2; dz = 1.0f; }
    if (kt == Nt - 1) { kt = Nt - 2; dt = 1.0f; }
    kx = min(max(kx, 0), Nx - 2);
    ky = min(max(ky, 0), Ny - 2);
    kz = min(max(kz, 0), Nz - 2);
    kt = min(max(kt, 0), Nt - 2);
    const int NN = Nx * Ny * Nz;
    int o = kx + ky * Nx + kz * Nx * Ny + kt * NN;
    int on = kx + ky * Nx + (kz + 1) * Nx * Ny + kt * NN;
    float up = ((1.0f - dx) * (1.0f - dy) * u[o] + (1.0f - dx) * dy * u[o + Nx]
                + dx * (1.0f - dy) * u[o + 1] + dx * dy * u[o + Nx + 1]) * (1.0f - dz)
             + ((1.0f - dx) * (1.0f - dy) * u[on] + (1.0f - dx) * dy * u[on + Nx]
                + dx * (1.0f - dy) * u[on + 1] + dx * dy * u[on + Nx + 1]) * dz;
    o += NN;
    on += NN;
    float un = ((1.0f - dx) * (1.0f - dy) * u[o] + (1.0f - dx) * dy * u[o + Nx]
                + dx * (1.0f - dy) * u[o + 1] + dx * dy * u[o + Nx + 1]) * (1.0f - dz)
             + ((1.0f - dx) * (1.0f - dy) * u[on] + (1.0f - dx) * dy * u[on + Nx]
                + dx * (1.0f - dy) * u[on + 1] + dx * dy * u[on + Nx + 1]) * dz;
    return (1.0f - dt) * up + dt * un;
}

// Thermal value of one point at coordinates (xi, yj, zk)
// (3DgrainMPI/APTPhaseField.cu:278-327; type 5: 3Dgrain/APTPhaseField.cu:303).
// Returns true where the reference `continue`s past the slot, leaving the
// destination untouched.
__device__ __forceinline__ bool thermal_Tv(const StepArgs& a, float xi, float yj, float zk, float& T)
{
    const float t = a.t;
    if (a.use_iuc) {
        T = -a.uc0 * 1e6 * t;
        return false;
    }
    switch (a.thermal_type) {
    case 1:
        T = a.G * (zk - a.z0) - a.uc * 1e6 * t;
        return false;
    case 2: {
        float dist = sqrtf((yj - 0.5f * a.lyd) * (yj - 0.5f * a.lyd)
                           + (zk - a.z0 - a.lzd) * (zk - a.z0 - a.lzd)) - a.r0;
        T = -a.G * dist - a.uc * 1e6 * t;
        return false;
    }
    case 3: {
        float lm = (a.r0 - a.z0) / a.tan_angle;
        float x_start = 0;
        float xl = xi - x_start;
        float r0_x = a.z0 + (a.r0 - a.z0) * xl / lm;
        float z_tilt = a.z0 + a.lzd - zk;
        float dist = a.cos_angle * (sqrtf((yj - 0.5f * a.lyd) * (yj - 0.5f * a.lyd)
                                          + z_tilt * z_tilt) - r0_x);
        if (xl > lm + a.V * t * 1e6) return true;
        T = -a.G * dist - a.uc * 1e6 * t;
        return false;
    }
    case 4: {
        float xq = xi - a.V * t * 1e6;
        if (xq > a.mp_len + a.x0 || xq < 0.0f) return true;
        float v = interp3(a.psi_mac, xq - a.X0_mac, yj - a.Y0_mac, zk - a.Z0_mac, a.Nx, a.Ny,
                          a.Nz, a.Dx_mac);
        T = (a.order == 100) ? -v : -a.G * v;
        return false;
    }
    case 5:
        T = a.G * (zk - a.R * 1e6 * t - 2);
        return false;
    default:
        T = 0.0f;
        return false;
    }
}

// The same at grid point (i, j, k), coordinates read from the x/y/z arrays.
__device__ __forceinline__ bool thermal_T(const StepArgs& a, int i, int j, int k, float& T)
{
    const int tt = a.thermal_type;
    const bool nx = !a.use_iuc && (tt == 3 || tt == 4);
    const bool ny = !a.use_iuc && (tt >= 2 && tt <= 4);
    return thermal_Tv(a, nx ? a.x[i] : 0.0f, ny ? a.y[j] : 0.0f, a.z[k], T);
}

// Orientation rows of a slot: the grain's rotation where its centre phi
// exceeds LS (double compare), the identity elsewhere
// (3DgrainMPI/APTPhaseField.cu:258-273).
struct Rot {
    float m0, m1, m2, m3, m4, m5, m6, m7, m8;
};

__device__ __forceinline__ Rot slot_rot(const StepArgs& a, int gid, float phC)
{
    Rot r{1.0f, 0.0f, 0.0f, 0.0f, 1.0f, 0.0f, 0.0f, 0.0f, 1.0f};
    if (phC > kLSf) {
        const int tid = gid <= a.num_theta ? gid : (gid % a.num_theta) + 1;
        const float4* p = reinterpret_cast<const float4*>(a.R12 + 12 * tid);
        const float4 r0 = p[0], r1 = p[1], r2 = p[2];
        r = Rot{r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x};
    }
    return r;
}

// Right-hand side and explicit Euler update of one filled slot
// (3DgrainMPI/APTPhaseField.cu:250-340) with its orientation rows.  repul is
// the ascending sum of 0.25*(phiC_p+1)^2 over the other filled slots (empty
// ones add exactly +0).
__device__ __forceinline__ float slot_update_r(const StepArgs& a, const Rot& m, float phD,
                                               float phB, float phL, float phC, float phR,
                                               float phT, float phU, float repul, float Up,
                                               float a_s, float epsv)
{
    const float phxn = (phR - phL) * 0.5f;
    const float phyn = (phT - phB) * 0.5f;
    const float phzn = (phU - phD) * 0.5f;
    const float A2 = kine_ani(phxn, phyn, phzn, m.m0, m.m1, m.m2, m.m3, m.m4, m.m5, m.m6, m.m7,
                              m.m8, a_s, epsv, a.eps);
    const float diff = phR + phL + phT + phB + phU + phD - 6.0f * phC;
    const float omc = 1.0f - phC * phC;
    const float rhs = diff * a.hi * a.hi + omc * phC
                    - a.lamd * Up * (omc * omc - 6.0f * (phC + 1.0f) * repul);
    const float dphi = rhs / A2;
    return phC + a.dt * dphi;
}

__device__ __forceinline__ float slot_update(const StepArgs& a, int gid, float phD, float phB,
                                             float phL, float phC, float phR, float phT,
                                             float phU, float repul, float Up, float a_s,
                                             float epsv)
{
    return slot_update_r(a, slot_rot(a, gid, phC), phD, phB, phL, phC, phR, phT, phU, repul, Up,
                         a_s, epsv);
}

// Overflow policy for a point whose neighbourhood holds more than K distinct
// ids (undefined behaviour in the reference, 3DgrainMPI/APTPhaseField.cu:222-231).
// Kept set: the K ids ranked first by (largest phi over their entries, then
// earliest entry reaching it), in first-appearance order.
//
// A group of lanes settles one point: lane l holds the K (id, phi) entries of
// neighbour l (8 lanes for the 7 points; 16 lanes with up to two positions
// each, l and l + 16, for the 27), all loaded in one round trip.  K rounds
// each pick the entry of largest phi (earliest among equals) that is left,
// which names the next id of the ranking, and drop that id's entries; lanes
// reduce by DPP within the group.  Then lane q updates slot q.
//
// Bound by latency for short lists, by VALU issue and the fetches of the
// neighbours' lines for long ones (~800 instructions per wave of 8 points).
// Searching the maximum, its position and its id one after the other took 950,
// and passing the step's arguments by value spilled scalar registers (97 vector
// registers against 70): 64^3 K=8 13.4 -> 11.4 us, 96x96x128 K=5 with 27 points
// 127 -> 108, 256x256x512 133 -> 119 (89 with segments by region).  One point per lane with a streaming
// top-K (56 dependent pushes and a second pass over the neighbours) was one
// long chain of loads and compares, and left all but a few CUs idle: the
// fix-up of a 64^3 K=8 start-up fell from 53-62 to 12-13 us, of 32^3 K=5 from
// 27 to 9 us, of 96x96x128 K=5 with the 27-point gather from 121-148 to
// 51-122 us.  It gathers from the state; the records of the neighbours'
// entries that the step kernel used to write for it (448 B a point at K=8)
// cost the step more than they saved (256x256x512 start-up: step kernel 530 ->
// 449 us without them, fix-up 93 -> 127 us).
template <bool G27>
struct FixGroup {
    static constexpr int kLanes = G27 ? 16 : 8;   // lanes per point
    static constexpr int kPos = G27 ? 2 : 1;      // neighbour positions per lane
    static constexpr int kPoints = 64 / kLanes;   // points per wave
    static constexpr int kIds = G27 ? 256 : 64;   // scan positions (padded): LDS words of the ids
};

// LDS words of one group: the kept ids' phi at the 7 stencil rows by rank
// (8 x 8), then four rows of 8: ids and first positions by rank, rank by slot,
// repulsion by slot.  The stride keeps a wave's groups on different banks.
constexpr int kFixVal = 0, kFixId = 64, kFixPos = 72, kFixRank = 80, kFixRep = 88, kFixStride = 104;

template <int CTRL>
__device__ __forceinline__ int dpp_get(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}

// Smallest value over a group of 8 or 16 lanes, on every lane of it
// (all lanes of the wave active): xor 1, xor 2, half-row mirror, row mirror.
template <bool G27>
__device__ __forceinline__ int group_min(int v)
{
    v = min(v, dpp_get<0xB1>(v));
    v = min(v, dpp_get<0x4E>(v));
    v = min(v, dpp_get<0x141>(v));
    return G27 ? min(v, dpp_get<0x140>(v)) : v;
}

// phi, no NaN, as an integer of the same order (-0 as +0, below every float: kNoKey).
constexpr int kNoKey = (int)0x80000000;
__device__ __forceinline__ int phi_key(float x)
{
    const int b = __float_as_int(x + 0.0f);
    return b ^ ((b >> 31) & 0x7fffffff);
}

// Ranking keys of the fix-up: doubles 1.mantissa, or below 1.0 (never NaN).
constexpr unsigned kRankOne = 0x3ff00000u;
__device__ __forceinline__ double rank_key(unsigned hi, unsigned lo) { return __hiloint2double((int)hi, (int)lo); }
__device__ __forceinline__ double rank_max(double a, double b)
{
    double m;
    asm("v_max_f64 %0, %1, %2" : "=v"(m) : "v"(a), "v"(b));
    return m;
}
template <int CTRL>
__device__ __forceinline__ double rank_max_dpp(double a)
{
    return rank_max(a, rank_key((unsigned)dpp_get<CTRL>(__double2hiint(a)), (unsigned)dpp_get<CTRL>(__double2loint(a))));
}
template <bool G27>
__device__ __forceinline__ double group_rank_max(double a)
{
    a = rank_max_dpp<0xB1>(a);
    a = rank_max_dpp<0x4E>(a);
    a = rank_max_dpp<0x141>(a);
    return G27 ? rank_max_dpp<0x140>(a) : a;
}

// Orders a wave's LDS accesses (DS operations of a wave complete in order).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The overflow policy and pass B for one point per group; every lane of the
// wave calls it.  on: the group has a point (C, its element index).
template <int K, bool G27>
__device__ __forceinline__ void fixup_group(const StepArgs& a, unsigned C, bool on, int l, unsigned* sc,
                                            float a_s, float epsv)
{
    using F = FixGroup<G27>;
    constexpr int E = F::kPos * K;
    const int A = a.fnx * a.fny;
    const int k = (int)C / A;
    const int rem = (int)C - k * A;
    const int j = rem / a.fnx;
    const int i = rem - j * a.fnx;
    int id[E];
    float ph[E];
    double key[E];
    int row = -1, rowpos = 0;  // the lane's stencil row (D,B,L,C,R,T,U) and which of its positions it is
#pragma unroll
    for (int t = 0; t < F::kPos; ++t) {
        const int u = l + 16 * t;  // scan position
        int dx, dy, dz, s;
        bool in;
        if (!G27) {
            dx = u == 2 ? -1 : u == 4 ? 1 : 0;
            dy = u == 1 ? -1 : u == 5 ? 1 : 0;
            dz = u == 0 ? -1 : u == 6 ? 1 : 0;
            s = u;
            in = u < 7;
        } else {  // z-major 27-point order (3Dgrain/APTPhaseField.cu:241-268)
            dx = u % 3 - 1;
            dy = u / 3 % 3 - 1;
            dz = u / 9 - 1;
            s = u == 4 ? 0 : u == 10 ? 1 : (u >= 12 && u <= 14) ? u - 10 : u == 16 ? 5 : u == 22 ? 6 : -1;
            in = u < 27;
        }
        if (in && s >= 0) {  // at most one position of a lane
            row = s;
            rowpos = t;
        }
        in = in && on;
        const int b = in ? bc_map(i + dx, a.fnx, a.bcx) + bc_map(j + dy, a.fny, a.bcy) * a.fnx +
                               bc_map(k + dz, a.fnz, a.bcz) * A
                         : (int)C;
#pragma unroll
        for (int p = 0; p < K; ++p) {
            const int x = a.arg[b + p * a.L];
            ph[t * K + p] = a.ph[b + p * a.L];
            id[t * K + p] = in ? x : -1;
        }
    }
    // An entry's key is its phi's order (32 bits) and below it the scan position
    // counted backwards (8 bits) in a double's mantissa, so one maximum finds
    // the largest phi and the earliest entry holding it; entries out of the
    // ranking lie below 1.0.  Its id is then looked up in LDS.  A NaN ranks below
    // every other entry, but nothing is larger than it either: as the first
    // entry left it is taken, whatever the maximum (`nan`: the wave has one; the
    // tests for it cost 99.1 -> 100.4 us for 96x96x128 K=5 with 27 points, 11.6 ->
    // 11.7 at 64^3).
    const int pos0 = l * K;  // scan position of entry e: pos0 + (16 K for the second position) + slot
    unsigned* ids = sc + kFixStride;
    unsigned odd = 0u;  // this lane's NaN entries
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int pos = pos0 + (e / K) * 16 * K + e % K;
        const bool ordered = ph[e] == ph[e];
        const unsigned u = ordered ? (unsigned)phi_key(ph[e]) ^ 0x80000000u : 0u;
        odd |= id[e] != -1 && !ordered ? 1u << e : 0u;
        key[e] = rank_key(id[e] != -1 ? kRankOne | u >> 12 : 0u, u << 20 | (unsigned)(255 - pos) << 12);
        ids[pos] = (unsigned)id[e];
    }
    wave_lds_fence();
    const bool nan = __ballot(odd != 0u) != 0ull;
    int nk = 0;
#pragma unroll 1
    for (int r = 0; r < K; ++r) {
        double m = key[0];
#pragma unroll
        for (int e = 1; e < E; ++e) m = rank_max(m, key[e]);
        m = group_rank_max<G27>(m);
        const bool live = (unsigned)__double2hiint(m) >= kRankOne;
        int top = 255 - ((unsigned)__double2loint(m) >> 12 & 255u);
        if (nan) {
            unsigned left = 0u;  // its entries not taken
#pragma unroll
            for (int e = 0; e < E; ++e)
                left |= (unsigned)__double2hiint(key[e]) >= kRankOne ? 1u << e : 0u;
            // 2 * position of the first entry left, + 1 for a NaN
            const int e = __ffs((int)left) - 1;
            int first = left ? 2 * (pos0 + (e / K) * 16 * K + e % K) + (int)(odd >> e & 1u) : 0x7fffffff;
            first = group_min<G27>(first);
            if (live && (first & 1)) top = first >> 1;
        }
        const int kid = live ? (int)ids[top] : kNoKey;
        nk += live ? 1 : 0;
        // the id's entries leave the ranking; its phi at this lane's stencil
        // row is the last entry's, as the reference's overwrite gives it
        float v = -1.0f;
        int fp = 0x7fffffff;
#pragma unroll
        for (int e = E - 1; e >= 0; --e) {
            const bool h = id[e] == kid;
            fp = h ? pos0 + (e / K) * 16 * K + e % K : fp;
            key[e] = rank_key(h ? 0u : (unsigned)__double2hiint(key[e]), (unsigned)__double2loint(key[e]));
        }
#pragma unroll
        for (int t = 0; t < F::kPos; ++t)
#pragma unroll
            for (int p = 0; p < K; ++p)
                v = id[t * K + p] == kid && (F::kPos == 1 || rowpos == t) ? ph[t * K + p] : v;
        fp = group_min<G27>(fp);
        if (row >= 0) sc[kFixVal + 8 * r + row] = __float_as_uint(v);
        if (l == 0) {
            sc[kFixId + r] = (unsigned)kid;
            sc[kFixPos + r] = (unsigned)fp;
        }
    }
    wave_lds_fence();
    if (l < K) {  // lane r: the slot of rank r
        const unsigned mine = sc[kFixPos + l];
        int slot = 0;
#pragma unroll
        for (int r = 0; r < K; ++r) slot += sc[kFixPos + r] < mine ? 1 : 0;
        sc[kFixRank + slot] = (unsigned)l;
    }
    wave_lds_fence();
    // lane q: slot q
    const int q = min(l, K - 1);
    const bool in = on && l < nk;
    const int r = in ? (int)sc[kFixRank + q] : 0;
    float v[7];
#pragma unroll
    for (int s = 0; s < 7; ++s) v[s] = __uint_as_float(sc[kFixVal + 8 * r + s]);
    const int gid = (int)sc[kFixId + r];
    const float w = v[3] + 1.0f;
    if (l < K) sc[kFixRep + l] = in ? __float_as_uint(0.25f * w * w) : 0u;
    wave_lds_fence();
    float repul = 0.0f;  // empty slots add exactly +0
#pragma unroll
    for (int p = 0; p < K; ++p) repul += p != q ? __uint_as_float(sc[kFixRep + p]) : 0.0f;
    wave_lds_fence();  // the words are rewritten for the group's next point
    if (on && l < K) {
        const int o = (int)C + l * a.L;
        if (!in) {
            a.arg_new[o] = -1;
            a.ph_new[o] = -1.0f;
        } else {
            float T;
            if (!thermal_T(a, i, j, k, T)) {
                const float nv = slot_update(a, gid, v[0], v[1], v[2], v[3], v[4], v[5], v[6], repul,
                                             T / a.L_cp, a_s, epsv);
                a.ph_new[o] = nv;
                a.arg_new[o] = (nv < kKillf) ? -1 : gid;
            }
        }
    }
}

// Column tiles of the activity map and the work list: 64 x 4 interior points.
// Planes are skipped with the activity map.  If every tile plane that the
// stencil of plane k can reach (the 3 x 3 neighbouring tiles at k-1, k, k+1,
// through the boundary maps) holds only empty pairs in the source, every
// point of plane k gathers no id and its result is K empty pairs; if the
// destination tile plane is also all empty, writing them changes nothing.
// Such planes are neither read nor written.  The results are the same bits as
// processing everything.
constexpr int kTX = 64, kTY = 4;

__device__ __forceinline__ int act_tile_x(int i) { return (i - 1) / kTX; }
__device__ __forceinline__ int act_tile_y(int j) { return (j - 1) / kTY; }

// Append the lanes of a wave in m (not 0) to the fix-up list (one atomic per
// wave); j, k: its first row, wave-uniform.  A segment holds a few y rows of
// every plane (capacity.h), so the fix-up's XCDs, an eighth of the list each,
// meet most of their points' neighbours in their own L2 (segments of every 64th
// row: 640 MB fetched for the 256x256x512 start-up's list in 119 us, 356 in 89).
__device__ __forceinline__ void fixup_append(const StepArgs& a, unsigned long long m, unsigned point, int j, int k)
{
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)m) - 1;
    const unsigned nz = (unsigned)a.fnz - 2u;
    const unsigned part = ((unsigned)(a.fny - 2) * nz + 63u) / 64u;
    const int seg = (int)(((unsigned)(j - 1) * nz + (unsigned)(k - 1)) / part) >> a.fix_shift;
    unsigned base = 0;
    if (lane == leader) base = atomicAdd(a.fix_count + kLineWords * seg, (unsigned)__popcll(m));
    base = __shfl(base, leader);
    if ((m >> lane) & 1ull)
        a.fix_list[fix_segment_base(seg, a.fix_shift, a.fix_cap) + base + (unsigned)__popcll(m & ((1ull << lane) - 1ull))] = point;
}

// Counts of m fix-up segments (count(q), m <= kMaxBatch) into s_cnt and the
// exclusive prefix of the wave units they make (POINTS entries each) into
// s_pre[0 .. m]; every thread of a kFixLanes workgroup calls it.  Returns the
// number of units.
template <int POINTS, class Count>
__device__ __forceinline__ unsigned fixup_units(int m, Count&& count, unsigned* s_pre, unsigned* s_cnt,
                                                unsigned* s_wave)
{
    const int per = (m + kFixLanes - 1) / kFixLanes;
    const int q0 = min((int)threadIdx.x * per, m), q1 = min(q0 + per, m);
    unsigned own = 0u;
    for (int q = q0; q < q1; ++q) {
        const unsigned c = count(q);
        s_cnt[q] = c;
        own += (c + POINTS - 1) / POINTS;
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    unsigned x = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned v = __shfl_up(x, d);
        x += lane >= d ? v : 0u;
    }
    if (lane == 63) s_wave[w] = x;
    __syncthreads();
    unsigned run = x - own;
#pragma unroll
    for (int u = 0; u < kFixLanes / 64; ++u) run += u < w ? s_wave[u] : 0u;
    for (int q = q0; q < q1; ++q) {
        s_pre[q] = run;
        run += (s_cnt[q] + POINTS - 1) / POINTS;
    }
    if (threadIdx.x == kFixLanes - 1) s_pre[m] = run;
    __syncthreads();
    return s_pre[m];
}

// Last segment whose units start at or before u (wave-uniform).
__device__ __forceinline__ int fixup_find(const unsigned* s_pre, int m, unsigned u)
{
    int lo = 0, hi = m - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_pre[mid] <= u) lo = mid;
        else hi = mid - 1;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// The plan kernels' unit of work: wave gw of a simulation covers z-chunk
// group cg = gw / (waves per group) and plan_tiles consecutive full tiles.
// Lane l reads the activity of tile slot l / plan_rows at plane kb - 1 +
// l % plan_rows (kb: first plane of the group): the 3 x 3 source words and
// the tile's own destination word.  Two ballots then hold every chunk's bits,
// and lane l = c * plan_tiles + slot assembles the masks of chunk c of the
// group for that tile slot, chunk = [k0, k1): need bit m for plane k0+m to
// process (some source word of the 3 x 3 tiles around the tile is active at a
// plane within one of it, through the z map, or its own destination word is).
// Items leave a wave chunk-major, so the list runs through z-chunk groups in
// order and the items in flight together lie in few planes.  put: the chunk has planes to
// process; item = its work-list code.
__device__ __forceinline__ void plan_wave(const StepArgs& a, int gw, int lane, bool& put, int& item,
                                          uint64_t& need)
{
    const int R = plan_rows(a.kchunk);
    const int TW = plan_tiles(a.kchunk);
    const int C = plan_group(a.kchunk);
    const int wpg = (a.items_chunk + TW - 1) / TW;  // waves per chunk group
    const int cg = gw / wpg;
    const int t0 = (gw - cg * wpg) * TW;
    const int zc0 = cg * C;
    const int kb = 1 + zc0 * a.kchunk;
    const int klast = min(kb + C * a.kchunk, a.fnz - 1);  // upper halo plane of the last chunk
    bool on = false, dst = false;
    {
        const int t = t0 + lane / R;
        const int kk = kb - 1 + lane % R;
        if (a.use_act && t < a.items_chunk && kk <= klast) {
            const int ty = t / a.tiles_x;
            const int tx = t - ty * a.tiles_x;
            const int i0 = 1 + tx * kTX, j0 = 1 + ty * kTY;
            const int xl = act_tile_x(bc_map(i0 - 1, a.fnx, a.bcx));
            const int xr = act_tile_x(bc_map(min(i0 + kTX, a.fnx - 1), a.fnx, a.bcx));
            const int yl = act_tile_y(bc_map(j0 - 1, a.fny, a.bcy));
            const int yr = act_tile_y(bc_map(min(j0 + kTY, a.fny - 1), a.fny, a.bcy));
            const int rl = yl * a.ntx, rc = ty * a.ntx, rr = yr * a.ntx;
            const unsigned* w = a.act_src + bc_map(kk, a.fnz, a.bcz) * a.ntiles;
            const unsigned e = a.ep_src;
            // bitwise ors: the nine reads go out together
            on = (w[xl + rl] >= e) | (w[tx + rl] >= e) | (w[xr + rl] >= e) | (w[xl + rc] >= e) |
                 (w[tx + rc] >= e) | (w[xr + rc] >= e) | (w[xl + rr] >= e) | (w[tx + rr] >= e) |
                 (w[xr + rr] >= e);
            dst = kk >= kb && kk < klast && a.act_dst[kk * a.ntiles + tx + rc] >= a.ep_dst;
        }
    }
    const uint64_t A = __ballot(on);
    const uint64_t D = __ballot(dst);
    const int c = lane / TW;
    const int slot = lane - c * TW;
    const int zc = zc0 + c;
    const int t = t0 + slot;
    put = false;
    item = 0;
    need = 0ull;
    if (c < C && zc < a.nzchunk && t < a.items_chunk) {
        const int k0 = 1 + zc * a.kchunk;
        const int n = min(k0 + a.kchunk, a.fnz - 1) - k0;
        const uint64_t full = (1ull << n) - 1ull;  // n <= 61
        if (!a.use_act) {
            need = full;
        } else {
            const int sh = slot * R + c * a.kchunk;  // lane of plane k0 - 1 for this tile
            const uint64_t ac = (A >> sh) & ((1ull << (n + 2)) - 1ull);
            need = ((ac | (ac >> 1) | (ac >> 2)) | ((D >> (sh + 1)) & full)) & full;
        }
        put = need != 0ull;
        item = zc * a.items_chunk + t;
    }
}

// List position of this lane's chunk if `put`.  Every thread of the workgroup
// (kPlanWaves waves) calls it; waves take consecutive runs of positions in
// wave order, reserved with one atomic per workgroup.
template <int kPlanWaves>
__device__ __forceinline__ unsigned plan_slot(bool put, unsigned* count, unsigned* s_cnt)
{
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const unsigned long long m = __ballot(put);
    if (lane == 0) s_cnt[w] = (unsigned)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned t = 0u;
        for (int u = 0; u < kPlanWaves; ++u) {
            const unsigned c = s_cnt[u];
            s_cnt[u] = t;
            t += c;
        }
        s_cnt[kPlanWaves] = t ? atomicAdd(count, t) : 0u;
    }
    __syncthreads();
    return s_cnt[kPlanWaves] + s_cnt[w] + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
}

// One workgroup of a step's plan (apt_plan, and the plan half of
// apt_fixplan): plan block pb covers waves 4*pb .. 4*pb+3; block 0 also
// clears the counter set of the step after this one.
__device__ __forceinline__ void plan_block(const StepArgs& a, int pb)
{
    constexpr int kPlanWaves = kBlock / 64;
    __shared__ unsigned s_cnt[kPlanWaves + 1];
    const int g = pb * kBlock + (int)threadIdx.x;
    // the counter set of the step after this one (last used two steps
    // before, whose fix-up has finished) starts from zero
    if (g <= kSpread) a.cnt_next[kLineWords * g] = 0u;  // the list segments' and the work list's
    const int gw = g >> 6;  // wave-uniform
    const int lane = threadIdx.x & 63;
    bool put = false;
    int item = 0;
    uint64_t need = 0ull;
    if (gw < plan_waves(a.kchunk, a.nzchunk, a.items_chunk)) plan_wave(a, gw, lane, put, item, need);
    const unsigned q = plan_slot<kPlanWaves>(put, a.wl_count, s_cnt);
    if (put) {
        a.wl_item[q] = item;
        a.wl_need[q] = need;
    }
}

__host__ __device__ inline int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

}  // namespace

}  // namespace cupf
