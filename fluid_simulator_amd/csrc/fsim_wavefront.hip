// fsim_wavefront.hip — persistent wavefront kernels for the MIC(0) factor
// and the two triangular sweeps (bridsonSolverGrid.cpp:91-163).
//
// Each cell depends only on its three upstream neighbours (-x,-y,-z for the
// factor and the forward sweep, +x,+y,+z for the backward sweep), so the
// serial lexicographic loop of the reference can run on i+j+k planes; every
// cell performs the same operations in the same order as the serial loop, so
// the result is bit-identical to it whatever the schedule (values that are not
// finite: on_water).
//
// Decomposition.  One workgroup owns a tile of WF_TY x 64 (y, z) columns and
// marches along x, one rotated plane (ridx) per step: lane tz of every row
// works on x = p - rot(z) at plane p, so its -z value was produced by lane
// tz - 1 one step earlier (DPP wave shift), its -x value by itself one step
// earlier, and its -y value by the row above at the same step.  A compute wave
// holds WF_R rows, whose -y values pass in registers; between waves they pass
// through LDS rings.  The backward sweep mirrors y, z inside a z-tile, and the
// planes, so that its upstream is also the row above, lane tz - 1 and the
// previous step.
//
// Groups.  Everything outside the arithmetic happens once per group of WF_G =
// 4 steps.  The solver vectors interleave four planes, so a lane loads and
// stores the four steps of one row with one 16-byte access each; a wave hands
// its last row's four values per lane on with one 16-byte LDS write, and one
// readiness test covers the group.  A sweep is a chain of about
// nx + nz + 4 * ny / WF_R dependent steps, and a step's cost is its instruction
// count (a wave issues one per 4.7 cycles, measured; an LDS read returns after
// 50, a branch on a vector comparison takes 35), so what is spent per step
// decides.  One handshake, one tag test and six 4-byte memory accesses per
// step measured 0.30 us a step, 209 and 202 us a sweep at 256^3 (water in 0.6
// of the height) and 98 us at 128^3; groups take 0.07 us a step, 132 and 126
// us at 256^3 and 46 us at 128^3, the same bits.  At 256^3 the tiles' memory
// traffic counts: a compute unit moves 18 KB per group of a 6-row tile (24 in
// the forward sweep of an iteration), and without the result's stores the
// sweep takes 113 us.  Three compute waves of two rows measured best (2 x 4:
// 142 us forward, 2 x 8: 190 us, 1 x 4: 164 us, 4 x 2: 154 us), and at no size
// clearly worse than another number of waves (frames in ms with 2 / 3 / 4 / 5
// waves: 32^3 1.29 / 1.21 / 1.23 / 1.18, 70x52x91 5.9 / 5.6 / 6.0 / 6.2, 96^3
// 9.0 / 8.8 / 8.7 / 8.9, 128^3 13.1 / 12.5 / 12.6 / 12.9, 203x67x131 20.8 /
// 21.3 / 23.1 / 25.3, 256^3 147 / 144 / 149 / 168); storing waves that take the results over LDS, so that the
// in-order memory counter does not hold loads behind stores, did not pay
// (166 us), nor did stores past the caches.
//
// Memory.  Buffer resources: a wave's group offset lives in a scalar register
// and each lane has a constant in-plane offset per row, replaced by an
// out-of-range one (loads read 0, stores drop) while none of the lane's cells
// of the group is in the marched x range, or the lane is off the grid.  A
// group never holds the first and the last cells of a column at once
// (rot_planes), so the values around the range inside a group belong to cells
// without WATER: their factor is 0 and so is every value derived from it
// (on_water).
// Storing such zeros needs no mask.  The march covers the x range that holds
// WATER (xrange), which the first pass over the labels found.
//
// Hand-over inside a workgroup: a ring slot per group and a counter of groups
// published.  LDS executes one wave's accesses in order, so a reader that sees
// the counter sees the slot, and a reader issues counter and slot reads
// together, one group ahead; only if the counter was too low are they read
// again.  The consumers' counters bound the reuse of the slots.
//
// Across workgroups, values at the tile edges travel through boundary buffers
// in HBM as packets of four values per lane, written with device-scope stores
// (see "boundary packets").  The last compute wave stores the +y edge itself;
// three communication waves per workgroup do the rest: two poll the upstream
// tiles' packets and republish them into LDS rings, one takes the +z edge
// values from LDS and stores them.  On gfx9 the memory counter completes in
// order, so a global read whose result is needed "now" would stall the compute
// waves' prefetch stream (kPrefetch groups ahead, each prefetch slot in fixed
// registers).
//
// Side work.  At most a tile per compute unit runs, and the tiles wait most of
// the time: blocks behind the tiles' do the iteration's streaming passes
// (SideWork) beside them.  The forward sweep of an iteration computes r - alpha
// q itself while they store it: a third load a row, 46 instead of 43 us at
// 128^3, 164 instead of 132 at 256^3, where the tiles are bound by their memory
// accesses (a separate pass takes 13 and 35).  The backward sweep with t . t
// takes 44 (44) and 129 (126), with the x update as well 44 and 160.
//
// Every wait is bounded: past kSpinLimit polls, or as soon as any wave in the
// grid has given up, a wave raises the error flag and carries on, so the
// grid always drains.  Workgroups take tiles from a ticket counter in
// row-major (J, K) order, so the tiles a workgroup waits on were taken by
// workgroups already running.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fsim_reduce.hpp"

namespace fsim {

constexpr int kSpinLimit = 1 << 21;
constexpr int kBusyPolls = 64;   // polls before a waiting wave starts to sleep
constexpr int kRing = 8;         // ring slots (groups) between waves, and the unroll of the group loop
constexpr int kPrefetch = 6;     // groups of per-cell inputs loaded ahead (7: no change)
static_assert(kPrefetch >= 1 && kPrefetch <= kRing, "a prefetch slot per unrolled group");
constexpr int kRingZ = 32;   // +z out-ring slots (groups): the z edge runs 16 groups behind its tile
constexpr int kAll = 0x3fffffff;              // counter value "everything": no upstream, or no consumer
constexpr uint32_t kOob = 0x80000000u;        // buffer offset beyond every array: reads 0, drops stores
constexpr uint32_t kEmpty = 0xffffffffu;      // boundary-packet word that has not been sent
constexpr int kRawBufferFlags = 0x00020000;   // buffer resource word 3 (raw 32-bit access, gfx9)
constexpr int kDeviceScope = 16;              // sc1 of a buffer access: past the L1, through the L2
constexpr int kVolatile = (int)0x80000000;    // a buffer load that is neither merged nor moved

template <int KIND>
struct Kind {   // WaveKind: the sweeps (FP32)
    using T = float;
    static constexpr bool FWD = KIND == WAVE_FWD || KIND == WAVE_FWD_UPDATE || KIND == WAVE_FWD_ALONE;
    static constexpr bool MASK = KIND == WAVE_FWD_ALONE || KIND == WAVE_BWD_ALONE;   // on_water
    static constexpr int NP = 1;     // 32-bit words per value
};
template <>
struct Kind<0> {   // MIC(0) factor (FP64)
    using T = double;
    static constexpr bool FWD = true;
    static constexpr int NP = 2;
};

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N-1>) in order
template <int N, int I = 0, class F>
__device__ __forceinline__ void unroll(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unroll<N, I + 1>(f);
    }
}
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ inline bool gave_up(const int* err) { return __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; }

// LDS accesses that keep their order among each other (volatile, explicit LDS pointers)
typedef __attribute__((address_space(3))) volatile u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) volatile uint32_t lds_u32;
typedef __attribute__((address_space(3))) volatile int lds_i32;
typedef __attribute__((address_space(3))) volatile i32x4 lds_i32x4;
__device__ inline int lget(const int* p) { return *(lds_i32*)p; }
__device__ inline i32x4 lget4(const int* p) { return *(lds_i32x4*)p; }
__device__ inline void lput(int* p, int v) { *(lds_i32*)p = v; }
__device__ inline uint32_t lget(const uint32_t* p) { return *(lds_u32*)p; }
__device__ inline u32x4 lget4(const uint32_t* p) { return *(lds_u32x4*)p; }
__device__ inline void lput4(uint32_t* p, u32x4 v) { *(lds_u32x4*)p = v; }

__device__ inline __amdgpu_buffer_rsrc_t rsrc(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, kRawBufferFlags);
}

// lane i receives lane i-1's value, lane 0 receives `first` (DPP wave_shr:1)
__device__ inline uint32_t shr1_bits(uint32_t first, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)v, 0x138, 0xf, 0xf, false);
}

// the four values of a lane's group as 32-bit words: value j, word k at [j * NP + k]
template <class T>
struct Group;
template <>
struct Group<float> {
    u32x4 q[1];
    __device__ float get(int j) const { return __uint_as_float(q[0][j]); }
    __device__ void set(int j, float v) { q[0][j] = __float_as_uint(v); }
    // lane i - 1's value, +0 on lane 0 (a DPP operand of the instruction that uses it)
    __device__ static float shr1(float v) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
    }
};
template <>
struct Group<double> {
    u32x4 q[2];
    __device__ double get(int j) const {
        return __hiloint2double((int)q[j >> 1][2 * (j & 1) + 1], (int)q[j >> 1][2 * (j & 1)]);
    }
    __device__ void set(int j, double v) {
        q[j >> 1][2 * (j & 1)] = (uint32_t)__double2loint(v);
        q[j >> 1][2 * (j & 1) + 1] = (uint32_t)__double2hiint(v);
    }
    __device__ static double shr1(double first, double v) {
        const uint32_t lo = shr1_bits((uint32_t)__double2loint(first), (uint32_t)__double2loint(v));
        const uint32_t hi = shr1_bits((uint32_t)__double2hiint(first), (uint32_t)__double2hiint(v));
        return __hiloint2double((int)hi, (int)lo);
    }
};

// Ticket in [0, TJ*TK), or -1 (with *err raised) if the counter is out of
// step with the launch (only after a failed launch); the caller then exits.
__device__ inline int take_tile(const WaveArgs& A) {
    __shared__ int s_tile;
    if (threadIdx.x == 0) {
        long long t = (long long)(atomicAdd(A.ticket, 1ull) - A.ticket_base);
        if (t < 0 || t >= (long long)A.TJ * A.TK) {
            atomicOr(A.err, 2);
            t = -1;
        }
        s_tile = (int)t;
    }
    __syncthreads();
    return s_tile;
}

// Grid y and z of local row ty, lane tz of tile (J, K).
template <bool FWD>
__device__ inline int y_of(const WaveArgs& A, int J, int ty) { return FWD ? 1 + J * WF_TY + ty : A.ny - 2 - (J * WF_TY + ty); }
template <bool FWD>
__device__ inline int z_of(const WaveArgs& A, int K, int tz) {
    return FWD ? 1 + K * WF_TZ + tz : 1 + (A.TK - 1 - K) * WF_TZ + (WF_TZ - 1 - tz);
}

// The march of a tile's z column K: groups of planes, counted from 0 in the
// order of the march.  All tiles of one K share it.
struct March {
    int xa, xb;   // x range with WATER
    int g0;       // plane group of march group 0 (unwrapped planes: x + rot)
    int ng;       // groups
};
template <bool FWD>
__device__ inline March march_of(const WaveArgs& A, int K, int xa, int xb) {
    const int kz = FWD ? K : A.TK - 1 - K;
    const int cols = min(WF_TZ, A.nz - 2 - kz * WF_TZ);
    const int first = xa / WF_G, last = (xb + cols - 1) / WF_G;
    return March{xa, xb, FWD ? first : last, last - first + 1};
}
// The element (step) of the upstream z tile's march that holds the -z value of
// element e of tile K's march is e + z_shift: the upstream lane 63 is 63 planes
// away from lane 0 (forward: ahead, backward: behind), and the two marches may
// start at different groups.
template <bool FWD>
__device__ inline int z_shift(const March& up, const March& me) {
    return WF_TZ - 1 - (FWD ? 0 : WF_G * (me.g0 - up.g0));
}
// march groups in which lane 0 of tile K is inside the x range, counted from 0
template <bool FWD>
__device__ inline int z_groups(const March& me) {
    return FWD ? me.xb / WF_G - me.g0 + 1 : me.g0 - (me.xa + WF_TZ - 1) / WF_G + 1;
}

// What the waves of a workgroup share.  Counters: a compute wave reads one
// record a group.  in: groups of its -y values published (by the wave above, or
// the receiving wave); zin: groups of the -z edge published; out: groups it may
// have written to its ring (those its reader is done with, plus the ring's
// slots); zout: the same for zo.
struct Counters {
    int in, zin, out, zout;
};
// Factor: the terms that depend on a cell's info word alone, so that a step has no loop or branch
struct FactorTable {
    f64x2 diag[8];   // by the number of non-SOLID neighbours: their sum of scales, and what replaces a small e
    double up[4];    // by the two NB_UP bits of an axis: the sum of the -neighbour's other two A entries
};
struct NoTable {};
template <int KIND>
struct WaveLds {
    static constexpr int NP = Kind<KIND>::NP;
    std::conditional_t<KIND == 0, FactorTable, NoTable> tab;
    // ring 0: the -y edge; ring w + 1: the last row of compute wave w
    alignas(16) uint32_t ring[WF_NW][kRing][NP][WF_TZ][4];
    // -z edge: lane 0's upstream value of every row; the other lanes read zeros from beside it
    alignas(16) uint32_t zi[2][kRing][WF_TY][NP][4];
    alignas(16) uint32_t zo[WF_TY][kRingZ * WF_G * NP];           // +z edge: lane 63's values of every row
    // of compute wave w at [w + 1]; what the first wave hands up and the last one down goes to the
    // outer records.  cnt[w + 2].in is what compute wave w has finished
    alignas(16) Counters cnt[WF_NW + 2];
};

struct Tile {
    int J, K;
    March m;
    bool yup, zup;   // an upstream tile along y / z that holds WATER
    bool ydn, zdn;   // a downstream one
};

// ---- boundary packets -----------------------------------------------------------
// One row of 16-byte packets per group and edge: NL lanes x NP packets, a
// lane's four values.  A word that has not been sent holds kEmpty, a NaN that
// no value takes (may_send); of an FP64 value the high word tells.  The
// receiver puts kEmpty back, so a row is empty again when the kernel ends: a
// tile sends exactly the groups that its downstream tile receives.
template <int NP>
__device__ inline u32x4 may_send(u32x4 v) {
    if constexpr (NP == 1) {
        for (int k = 0; k < 4; k++) v[k] = min(v[k], kEmpty - 1);
    } else {
        v[1] = min(v[1], kEmpty - 1);
        v[3] = min(v[3], kEmpty - 1);
    }
    return v;
}
template <int NP>
__device__ inline bool is_sent(u32x4 v) {
    if constexpr (NP == 1) return max(max(v[0], v[1]), max(v[2], v[3])) != kEmpty;
    else return max(v[1], v[3]) != kEmpty;
}

// ---- receiving wave: upstream tile edge -> LDS ring ---------------------------
// The -y edge carries 64 lanes, the -z edge WF_TY rows; the wave forwards whole
// groups, once all packets of a group are there and its ring slot is free.
template <int KIND, bool YEDGE>
__device__ void recv_wave(const WaveArgs& A, WaveLds<KIND>& S, const Tile& T) {
    constexpr int NP = Kind<KIND>::NP;
    constexpr int B = 4;   // groups polled at once: a poll takes as long as two to three groups
    constexpr int NL = YEDGE ? WF_TZ : WF_TY;
    constexpr uint32_t kRow = NL * NP * 16;   // bytes per group
    if (YEDGE ? !T.yup : !T.zup) return;      // no upstream tile, or one without WATER (its edge is all zeros)
    const int l = threadIdx.x % 64;
    const bool on = l < NL;
    const int li = on ? l : 0;
    const int end = YEDGE ? T.m.ng : z_groups<Kind<KIND>::FWD>(T.m);
    const int64_t up = YEDGE ? (int64_t)(T.J - 1) * A.TK + T.K : (int64_t)T.J * A.TK + T.K - 1;
    const __amdgpu_buffer_rsrc_t buf = rsrc((YEDGE ? A.ybnd : A.zbnd) + up * A.SG * (kRow / 16), (int64_t)A.SG * kRow);
    // the consumer of lane l: wave 0 for the -y edge, the wave holding row l for the -z edge
    const int* used = &S.cnt[(YEDGE ? 0 : li / WF_R) + 2].in;
    auto publish = [&](int g) {
        if (YEDGE) {
            if (l == 0) lput(&S.cnt[1].in, g);
        } else if (l < WF_NW) {
            lput(&S.cnt[l + 1].zin, g);
        }
    };
    int g0 = 0, idle = 0;
    while (g0 < end) {
        u32x4 v[B][NP];
#pragma unroll
        for (int b = 0; b < B; b++) {
            const uint32_t row = (uint32_t)min(g0 + b, end - 1) * kRow;
#pragma unroll
            for (int c = 0; c < NP; c++)
                v[b][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    buf, (uint32_t)(c * NL + li) * 16u, row, kDeviceScope | kVolatile));
        }
        const int limit = lget(used) + kRing;   // groups below it have a free slot
        int n = 0;
        bool stop = false;
#pragma unroll
        for (int b = 0; b < B; b++) {
            bool ok = g0 + b < limit;
#pragma unroll
            for (int c = 0; c < NP; c++) ok = ok && is_sent<NP>(v[b][c]);
            stop = stop || g0 + b >= end || !__all(!on || ok);
            if (!stop) {
                const int slot = (g0 + b) % kRing;
                if (on) {
#pragma unroll
                    for (int c = 0; c < NP; c++)
                        lput4(YEDGE ? &S.ring[0][slot][c][li][0] : &S.zi[0][slot][li][c][0], v[b][c]);
                }
                n++;
                publish(g0 + n);
            }
        }
        g0 += n;
        if (n > 0) {
            idle = 0;
        } else {
            if (++idle > kSpinLimit / 64) {
                if (l == 0) atomicOr(A.err, 1);
                break;
            }
            if ((idle & 15) == 0 && gave_up(A.err)) break;
        }
    }
    publish(kAll);
    // empty the rows again, after the last poll: the memory counter orders a poll behind older stores
    if (on)
        for (int g = 0; g < end; g++)
#pragma unroll
            for (int c = 0; c < NP; c++)
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{kEmpty, kEmpty, kEmpty, kEmpty}, buf,
                                                       (uint32_t)(c * NL + li) * 16u, (uint32_t)g * kRow, 0);
}

// ---- sending wave: this tile's +z edge (LDS) -> packets ---------------------------
// Element e of the downstream march is element e + z_shift of this tile's lane
// 63 (zero outside this march).
template <int KIND>
__device__ void send_wave(const WaveArgs& A, WaveLds<KIND>& S, const Tile& T) {
    constexpr bool FWD = Kind<KIND>::FWD;
    constexpr int NP = Kind<KIND>::NP;
    constexpr int NL = WF_TY;
    constexpr uint32_t kRow = NL * NP * 16;
    constexpr int kMask = kRingZ * WF_G - 1;
    if (!T.zdn) return;   // nobody downstream: counters preset to kAll
    const int l = threadIdx.x % 64;
    const bool on = l < NL;
    const int li = on ? l : 0;
    const int64_t tile = (int64_t)T.J * A.TK + T.K;
    const __amdgpu_buffer_rsrc_t buf = rsrc(A.zbnd + tile * A.SG * (kRow / 16), (int64_t)A.SG * kRow);
    const March dn = march_of<FWD>(A, T.K + 1, T.m.xa, T.m.xb);
    const int end = z_groups<FWD>(dn), shift = z_shift<FWD>(T.m, dn);
    const int* ready = &S.cnt[li / WF_R + 2].in;
    auto release = [&](int g) {   // zo slots below g have been sent
        if (l < WF_NW) lput(&S.cnt[l + 1].zout, g + kRingZ);
    };
    for (int g = 0; g < end; g++) {
        const int e0 = WF_G * g + shift;   // first element of this march that the group needs
        const int need = min((e0 + 2 * WF_G - 1) / WF_G, T.m.ng);
        for (int spins = 0; !__all(!on || lget(ready) >= need);) {
            if (++spins > kSpinLimit || ((spins & 1023) == 0 && gave_up(A.err))) {
                if (l == 0) atomicOr(A.err, 1);
                release(kAll);   // never block the compute waves
                return;
            }
            if (spins > kBusyPolls) __builtin_amdgcn_s_sleep(1);
        }
        if (on) {
            u32x4 v[NP];
#pragma unroll
            for (int k = 0; k < WF_G * NP; k++) {
                const int e = e0 + k / NP;
                const uint32_t u = lget(&S.zo[li][(e & kMask) * NP + k % NP]);
                v[k / 4][k % 4] = e < 0 || e >= WF_G * T.m.ng ? 0u : u;
            }
#pragma unroll
            for (int c = 0; c < NP; c++)
                __builtin_amdgcn_raw_buffer_store_b128(may_send<NP>(v[c]), buf, (uint32_t)(c * NL + li) * 16u,
                                                       (uint32_t)g * kRow, kDeviceScope);
        }
        release(max(0, (e0 + WF_G) / WF_G));   // groups whose elements all lie below the next one needed
        for (int i = 0; i < A.send_delay; i++) __builtin_amdgcn_s_sleep(127);
    }
    release(kAll);
}

// A sweep's value v of a cell whose factor is p (0 off WATER).  Off WATER it is
// 0 by itself while every value is finite.  What is not finite (an input, or
// the infinite factor of a WATER cell between SOLID ones) would pass through
// AIR and SOLID cells to WATER that does not depend on it, which the sweeps
// outside a solve (WAVE_FWD_ALONE, WAVE_BWD_ALONE) keep from it by a select.  In
// a solve it makes s.q and alpha NaN and the solve ends with the pressure of
// before, wherever else it has been; there the select, a comparison and a
// move on the chain of every cell, costs a frame 32^3 1.17 -> 1.26 ms, 128^3
// APIC 12.3 -> 12.9, 256^3 148 -> 151.
template <int KIND>
__device__ inline float on_water(float v, float p) {
    if constexpr (Kind<KIND>::MASK) return p != 0.f ? v : 0.f;
    else return v;
}

// ---- compute waves -------------------------------------------------------------
// Factor (KIND 0, FP64):   e = diag - sum_a (A_a p_a)^2 - tau sum_a A_a (o1 + o2) p_a^2,
//                          guarded by sigma, p = 1/sqrt(e)  (calculatePreconditioner); passes p on
//                          No branch or loop in a step: diag and o1 + o2 come from a table by the info
//                          word, a neighbour that is not WATER carries 0.  450 us at 256^3 and 188 at
//                          128^3 (1055 and 420 with a loop over the neighbours per cell), of which the
//                          square root and the division are the larger part
// forward sweep (KIND 1):  q = (r - sum_{-a fluid} A_a q_a p_a) * p; passes m = A_a q p on
// backward sweep (KIND 2): z = (q - p * sum_{+a fluid} A_a z_a) * p; passes m = A_a z on
// with A_a = -scale, products and sums in the reference's order (x, y, z).
// A sweep's neighbour term A_a * value is the same for the three cells that use
// it, so the cell computes it once (same rounding).  A neighbour that is not
// WATER carries +0 (the fused multiply-add with +0 turns -0 into it), which
// leaves any partial sum unchanged, so the sweeps sum all three.
// LAST: the tile's last wave, whose last row is the +y edge: it stores the packets itself, which
// spares the edge a round trip through LDS and another wave.
template <int KIND, bool LAST>
__device__ __forceinline__ void compute_wave(const WaveArgs& A, const SideWork& W, WaveLds<KIND>& S, const Tile& T) {
#pragma clang fp contract(off)
    using KD = Kind<KIND>;
    using V = typename KD::T;
    constexpr bool FWD = KD::FWD;
    constexpr int NP = KD::NP, R = WF_R;
    constexpr bool UPD = KIND == WAVE_FWD_UPDATE;
    const int w = LAST ? WF_NW - 1 : __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int tz = threadIdx.x % 64;
    const uint32_t cells = (uint32_t)(A.ny * A.nz);   // of one plane
    const uint32_t ngroups = (uint32_t)(A.nxp / WF_G);
    // byte offsets are counted for the float vectors: 16 per (y, z) column and group
    const uint32_t gstride = cells * 16u, total = gstride * ngroups;
    // buffer resources.  sweeps: rA P32, rB in, rC out; factor: rA nbinfo (offsets halved), rC P32
    __amdgpu_buffer_rsrc_t rA, rB, rC, rQ;
    if constexpr (KIND == 0) {
        rA = rsrc(A.nbinfo, (int64_t)total / 2);
        rC = rsrc(A.P32, (int64_t)total);
        rB = rQ = rA;
    } else {
        // ranges one and two words longer than the arrays (never addressed): distinct descriptor
        // words keep the compiler from rebuilding one descriptor from another at every access
        rA = rsrc(A.P32, (int64_t)total + 8);
        rB = rsrc(A.in, (int64_t)total);
        rC = rsrc(A.out, (int64_t)total + 4);
        rQ = UPD ? rsrc(W.q, (int64_t)total + 12) : rA;
        // opaque to the compiler from here on, so that it keeps each descriptor whole in
        // four SGPRs instead of sharing equal words and reassembling them at every access
        asm volatile("" : "+s"(rA), "+s"(rB), "+s"(rC));
        if constexpr (UPD) asm volatile("" : "+s"(rQ));
    }
    const float ms = A.ms;
    const double scale = A.scale;
    const float malpha = UPD ? (float)(-W.red.sc->alpha) : 0.f;
    const int z = z_of<FWD>(A, T.K, tz);
    const int rho = FWD ? tz : WF_TZ - 1 - tz;   // rot(z)
    uint32_t off[R];                             // the lane's byte offset per row, kOob off the grid
    unroll<R>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        const int ty = w * R + r;
        const int y = y_of<FWD>(A, T.J, ty);
        const bool in = T.J * WF_TY + ty < A.ny - 2 && z <= A.nz - 2;
        off[r] = in ? (uint32_t)(y * A.nz + z) * 16u : kOob;
    });
    // the lane has cells of the x range in the march groups first .. first + span
    const int glo = (T.m.xa + rho) / WF_G, ghi = (T.m.xb + rho) / WF_G;
    const int first = FWD ? glo - T.m.g0 : T.m.g0 - ghi;
    const uint32_t span = (uint32_t)(ghi - glo);
    // ORed onto the offsets of group g: 0 inside, kOob outside (opaque, so that it stays a select)
    auto outside = [&](int g) {
        uint32_t o = (uint32_t)(g - first) <= span ? 0u : kOob;
        asm volatile("" : "+v"(o));
        return o;
    };
    auto advance = [&](uint32_t& o) {
        if (FWD) {
            o += gstride;
            if (o >= total) o -= total;
        } else {
            // o - gstride wraps above every offset when o < gstride: the smaller of the two is the
            // wrapped-around group
            const uint32_t below = o - gstride, wrapped = o + (total - gstride);
            o = below < wrapped ? below : wrapped;
        }
        o = __builtin_amdgcn_readfirstlane(o);   // a per-lane copy turns each buffer access into a loop
    };
    uint32_t op = __builtin_amdgcn_readfirstlane((uint32_t)T.m.g0 % ngroups * gstride);   // prefetched group's offset
    // inputs of the next kPrefetch groups, with the offsets they were loaded from: the result of a
    // group goes to the same place of another vector.  factor: nbinfo; sweeps: P32 and the input vector
    f32x4 pq[kRing][R], iq[kRing][R], uq[kRing][R];
    u32x2 nq[kRing][R];
    uint32_t lo[kRing][R], go[kRing];
    auto fetch = [&](auto dc, int g) {
        constexpr int d = decltype(dc)::value;
        const uint32_t out = outside(g);
        go[d] = op;
        unroll<R>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            const uint32_t o = off[r] | out;
            lo[d][r] = o;
            if constexpr (KIND == 0) {
                nq[d][r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rA, o >> 1, op >> 1, 0));
            } else {
                pq[d][r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rA, o, op, 0));
                iq[d][r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rB, o, op, 0));
                if constexpr (UPD) uq[d][r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rQ, o, op, 0));
            }
        });
        advance(op);
    };
    // issue order pinned, and each prologue group issues as many memory operations as the loop's
    // groups do (the stores, here dropped as out of range, then the loads): the wait for slot d then
    // allows the same number of younger operations on entry as at every later group
    constexpr int kStores = (KIND == 0 ? 3 : 1) * R + (LAST ? NP : 0);
    unroll<kPrefetch>([&](auto dc) {
        unroll<kStores>([&](auto kc) {
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{}, rC, kOob + 16u * decltype(kc)::value, 0, 0);
        });
        fetch(dc, decltype(dc)::value);
        __builtin_amdgcn_sched_barrier(0);
    });
    constexpr int kSlot = NP * WF_TZ * 4, kSlotZ = WF_TY * NP * 4;   // words per ring slot
    const uint32_t* const in_ring = &S.ring[w][0][0][tz][0];
    uint32_t* const out_ring = &S.ring[LAST ? 0 : w + 1][0][0][tz][0];   // LAST: not used
    const uint32_t* const z_ring = &S.zi[tz == 0 ? 0 : 1][0][w * R][0][0];
    const int* const my_cnt = &S.cnt[w + 1].in;
    int* const in_below = &S.cnt[w + 2].in;
    int* const out_above = &S.cnt[w].out;
    // ends with the march's groups, or is empty if nobody is downstream: what is sent is received
    const __amdgpu_buffer_rsrc_t ybuf = rsrc(A.ybnd + ((int64_t)T.J * A.TK + T.K) * A.SG * (WF_TZ * NP),
                                             LAST && T.ydn ? (int64_t)T.m.ng * WF_TZ * NP * 16 : 0);
    // upstream values of a group: its ring slots, read once the counters vouch for them
    Group<V> up, zp[R];
    auto read_slots = [&](auto dc) {
        constexpr int d = decltype(dc)::value % kRing;
#pragma unroll
        for (int c = 0; c < NP; c++) up.q[c] = lget4(in_ring + d * kSlot + c * WF_TZ * 4);
        unroll<R>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
#pragma unroll
            for (int c = 0; c < NP; c++) zp[r].q[c] = lget4(z_ring + d * kSlotZ + (r * NP + c) * 4);
        });
    };
    // waits until group g can run: its upstream values are there, and the slots it writes are free
    auto wait_for = [&](i32x4 cnt, int g, auto dc) {
        auto behind = [&]() {
            return __builtin_amdgcn_ballot_w64(min(min(cnt[0], cnt[1]), min(cnt[2], cnt[3])) <= g) != 0;
        };
        if (__builtin_expect(behind(), 0)) {
            int spins = 0;
            do {
                if (spins > kBusyPolls) __builtin_amdgcn_s_sleep(1);
                cnt = lget4(my_cnt);
                read_slots(dc);
                if ((++spins & 1023) == 0 && (spins >= kSpinLimit || gave_up(A.err))) {
                    if (tz == 0) atomicOr(A.err, 1);
                    cnt = i32x4{kAll, kAll, kAll, kAll};   // carry on with whatever is there
                }
            } while (behind());
        }
    };
    V prev[R];
    unroll<R>([&](auto rc) { prev[decltype(rc)::value] = 0; });
    wait_for(i32x4{0, 0, 0, 0}, 0, std::integral_constant<int, 0>{});
    auto group = [&](auto dc, int g, uint32_t* zo) {
        constexpr int d = decltype(dc)::value;
        __builtin_amdgcn_sched_barrier(0);
        // ---- the group's 4 steps of R rows
        Group<V> mine[R];    // what the rows pass on
        f32x4 res[R];        // sweeps: the result; factor: the FP32 copy
        unroll<WF_G>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            constexpr int e = FWD ? j : WF_G - 1 - j;   // the step's plane inside the storage group
            V above = up.get(j);
            unroll<R>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                if constexpr (KIND == 0) {
                    const V vz = Group<V>::shr1(zp[r].get(j), prev[r]);
                    const uint32_t info = (nq[d][r][e >> 1] >> (16 * (e & 1))) & 0xffffu;
                    const double upv[3] = {prev[r], above, vz};
                    double eneg = 0, eneg_tau = 0;
#pragma unroll
                    for (int ax = 0; ax < 3; ax++) {
                        const double ap = -scale * upv[ax];
                        eneg += ap * ap;
                        eneg_tau += ap * S.tab.up[(info >> (NB_UP_SHIFT + 2 * ax)) & 3] * upv[ax];
                    }
                    const f64x2 dg = S.tab.diag[(info >> NB_NONSOLID_SHIFT) & 7];
                    double ee = dg[0] - eneg - eneg_tau * 0.97;
                    ee = ee < 0.25 * dg[0] ? dg[1] : ee;
                    double v = 1.0 / sqrt(ee);
                    v = (info & NB_FLUID) ? v : 0.0;
                    res[r][e] = (float)v;
                    prev[r] = v;
                } else {
                    const float p = pq[d][r][e];
                    float in = iq[d][r][e];
                    if constexpr (UPD) in = __builtin_fmaf(uq[d][r][e], malpha, in);
                    // -z: the packet's value on lane 0 (+0 on the others), lane tz - 1's on the others (+0 on
                    // lane 0): their sum is the one that counts
                    const float vz = zp[r].get(j) + Group<V>::shr1(prev[r]);
                    float acc = prev[r] + above;
                    acc += vz;
                    float outv, v;
                    if (FWD) {
                        outv = on_water<KIND>((in - acc) * p, p);
                        v = outv * p;
                    } else {
                        outv = on_water<KIND>((in - acc * p) * p, p);
                        v = outv;
                    }
                    res[r][e] = outv;
                    prev[r] = __builtin_fmaf(ms, v, 0.f);
                }
                mine[r].set(j, prev[r]);
                above = prev[r];
            });
        });
        // ---- publish first (the next wave waits for it) and ask for the next group's counters; store
        // while they come; then the next group's slots, whose latency the prefetch covers
        int next = g + 1;
        asm volatile("" : "+s"(next));   // stays a scalar beside the lane branch below
#pragma unroll
        for (int c = 0; c < NP; c++) {
            if constexpr (LAST)
                __builtin_amdgcn_raw_buffer_store_b128(may_send<NP>(mine[R - 1].q[c]), ybuf,
                                                       (uint32_t)(c * WF_TZ + tz) * 16u, (uint32_t)g * (WF_TZ * NP * 16),
                                                       kDeviceScope);
            else lput4(out_ring + d * kSlot + c * WF_TZ * 4, mine[R - 1].q[c]);
        }
        if (tz == WF_TZ - 1) {
            unroll<R>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
#pragma unroll
                for (int c = 0; c < NP; c++)
                    lput4(zo + (r * kRingZ + d) * WF_G * NP + c * 4, mine[r].q[c]);
            });
            lput(in_below, next);   // also tells the sending wave that zo is there
            lput(out_above, next + kRing);
        }
        const i32x4 cnt = lget4(my_cnt);
        read_slots(std::integral_constant<int, d + 1>{});
        unroll<R>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, res[r]), rC, lo[d][r], go[d], 0);
            if constexpr (KIND == 0) {
                // FP64: 32 bytes per column and group, beyond 32-bit offsets on the largest grids: a
                // resource per group
                const __amdgpu_buffer_rsrc_t rD =
                    rsrc(reinterpret_cast<char*>(A.P64) + 2 * (int64_t)go[d], 2 * (int64_t)gstride);
                const uint32_t o = lo[d][r] < kOob ? 2 * lo[d][r] : kOob;
                __builtin_amdgcn_raw_buffer_store_b128(mine[r].q[0], rD, o, 0, 0);
                __builtin_amdgcn_raw_buffer_store_b128(mine[r].q[1], rD, o, 16, 0);
            }
        });
        fetch(std::integral_constant<int, (d + kPrefetch) % kRing>{}, g + kPrefetch);
        __builtin_amdgcn_sched_barrier(0);
        wait_for(cnt, next, std::integral_constant<int, d + 1>{});
    };
    // whole blocks of kRing groups: the groups past the march have no cells (their waits are met at
    // once, their packets fall outside ybuf), and without exits inside a block every prefetch slot has
    // the same number of younger memory operations whenever it is waited for
    for (int g0 = 0; g0 < T.m.ng; g0 += kRing) {
        uint32_t* const zo = &S.zo[w * R][(g0 & (kRingZ - 1)) * WF_G * NP];
        unroll<kRing>([&](auto dc) { group(dc, g0 + decltype(dc)::value, zo); });
    }
    // nobody waits for this wave any more (the last group has waited for one more than there is)
    if (tz == 0) {
        lput(in_below, kAll);
        lput(out_above, kAll);
    }
}

template <int KIND>
__global__ void __launch_bounds__(WF_THREADS) k_wave(WaveArgs A, SideWork W) {
    using KD = Kind<KIND>;
    constexpr int NP = KD::NP;
    const unsigned tiles = gridDim.x - W.blocks;
    if (blockIdx.x >= tiles) {
        const Part part{blockIdx.x - tiles, W.blocks};
        if constexpr (KIND == WAVE_FWD_UPDATE) {
            update_r<WF_THREADS>(part, W.n, W.flags, W.q, W.r, W.r_next, W.red);
        } else if constexpr (KIND == WAVE_BWD) {
            dot_self<WF_THREADS>(part, W.n, W.flags, W.t, W.red);
            if (W.x_steps == 2) update_x_chunks<2>(part, W.n, W.flags, W.x, W.red.sc);
        }
        return;
    }
    __shared__ WaveLds<KIND> S;
    const int tile = take_tile(A);
    if (tile < 0) return;
    Tile T;
    T.J = __builtin_amdgcn_readfirstlane(tile / A.TK);
    T.K = __builtin_amdgcn_readfirstlane(tile % A.TK);
    // A tile none of whose (y, z) columns holds WATER has nothing to compute
    // (its cells' values are 0 from before the solve): it leaves at once.  Its
    // downstream tiles take its edge values as the zeros they are, exactly as
    // on a first tile, instead of waiting for packets, and its upstream tiles
    // send it none.
    // The flags come with the solve's masks: found from the columns here, behind
    // six barriers, they cost every launch 2 us (a frame at 32^3 1.27 -> 1.16 ms,
    // 128^3 APIC 13.0 -> 12.6).
    const uint8_t* const water = A.tilew + (KD::FWD ? 0 : A.TJ * A.TK);
    const int at = T.J * A.TK + T.K;
    auto holds = [&](bool there, int i) { return __builtin_amdgcn_readfirstlane(there ? water[i] : 0) != 0; };
    const bool mine = holds(true, at);
    T.yup = holds(T.J > 0, at - A.TK);
    T.zup = holds(T.K > 0, at - 1);
    T.ydn = holds(T.J < A.TJ - 1, at + A.TK);
    T.zdn = holds(T.K < A.TK - 1, at + 1);
    const int xa = __builtin_amdgcn_readfirstlane(A.xrange[0]);
    const int xb = __builtin_amdgcn_readfirstlane(A.xrange[1]);
    if (!mine) return;
    T.m = march_of<KD::FWD>(A, T.K, xa, xb);
    // without an upstream tile (or below / beside one without WATER) the -y / -z rings hold zeros
    for (int i = threadIdx.x; i < kRing * NP * WF_TZ * 4; i += WF_THREADS) (&S.ring[0][0][0][0][0])[i] = 0;
    for (int i = threadIdx.x; i < 2 * kRing * WF_TY * NP * 4; i += WF_THREADS) (&S.zi[0][0][0][0][0])[i] = 0;
    if (threadIdx.x < WF_NW + 2) {
        const int w = (int)threadIdx.x - 1;
        Counters c;
        c.in = w == 0 && !T.yup ? kAll : 0;
        c.zin = T.zup ? 0 : kAll;
        c.out = w == WF_NW - 1 ? kAll : kRing;   // the last row's packets have a row per group
        // zo: leading groups that no packet needs are free at once
        c.zout = kAll;
        if (T.zdn) c.zout = kRingZ + max(0, z_shift<KD::FWD>(T.m, march_of<KD::FWD>(A, T.K + 1, xa, xb)) / WF_G);
        S.cnt[threadIdx.x] = c;
    }
    if constexpr (KIND == 0) {
        if (threadIdx.x < 8) {
            double d = 0;
            for (unsigned k = 0; k < threadIdx.x; k++) d += A.scale;
            S.tab.diag[threadIdx.x] = f64x2{d, d < 1e-6 ? 1.0 : d};
        }
        if (threadIdx.x < 4) S.tab.up[threadIdx.x] = ((threadIdx.x & 1) ? -A.scale : 0.0) + ((threadIdx.x & 2) ? -A.scale : 0.0);
    }
    __syncthreads();
    const int wave = threadIdx.x / 64;
    if (wave < WF_NW - 1) compute_wave<KIND, false>(A, W, S, T);
    else if (wave == WF_NW - 1) compute_wave<KIND, true>(A, W, S, T);
    else if (wave == WF_NW) recv_wave<KIND, true>(A, S, T);
    else if (wave == WF_NW + 1) recv_wave<KIND, false>(A, S, T);
    else send_wave<KIND>(A, S, T);
}

// ---- 2D grids ----------------------------------------------------------------------
// One column of cells along z leaves 63 lanes of a compute wave idle, and the
// chain passes from wave to wave every two rows: 29 us a sweep of 128 x 128.
// Here a wave takes 64 rows, a row per lane, and lane l works on x = step - l:
// its -x value is its own of the step before and its -y value lane l - 1's of
// the step before (DPP wave shift), so a sweep is a chain of nx + ny steps,
// 15 us.  One workgroup does it; a wave's last row goes to the next one over
// LDS.
// A lane moves four steps of its row with one 16-byte access, but the lanes
// reach the ends of their groups at different steps: lane l is l mod 4 elements
// behind its group, and a group of four steps takes its operands from two
// consecutive storage groups, shifted by selects, and puts its results
// together in the same way.  The operations on a cell and their order are those
// of compute_wave: the same bits.
constexpr int k2dAhead = 8;    // groups of steps loaded ahead, and the unroll of their loop
constexpr int k2dLag = 17;     // groups of steps from a wave's first to its last row, + 1
constexpr int k2dPad = 64;     // elements before an edge row's first
__host__ __device__ inline int groups_2d(int ng) { return (ng + k2dLag + k2dAhead - 1) / k2dAhead * k2dAhead; }
__host__ __device__ inline int edge_2d(int ng) { return WF_G * groups_2d(ng) + k2dPad; }
static int waves_2d(int ny) { return (ny - 2 + WF_TZ - 1) / WF_TZ; }
static size_t lds_2d(int ny, int nxp) { return sizeof(float) * (size_t)(waves_2d(ny) - 1) * edge_2d(nxp / WF_G); }
constexpr size_t kLds2d = size_t(40) << 10;   // what the side blocks' reductions leave of 64 KB
static bool fits_2d(const WaveArgs& A) {
    return A.nz == 3 && waves_2d(A.ny) <= WF_THREADS / WF_TZ && lds_2d(A.ny, A.nxp) <= kLds2d;
}

// t[j] = seq[4 + j - c] and back, seq the elements of lo and hi, c = 2 c2 + c1
__device__ inline f32x4 behind(f32x4 lo, f32x4 hi, bool c1, bool c2) {
    const float seq[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    float t[8];
#pragma unroll
    for (int k = 2; k < 8; k++) t[k] = c1 ? seq[k - 1] : seq[k];
    f32x4 out;
#pragma unroll
    for (int j = 0; j < 4; j++) out[j] = c2 ? t[2 + j] : t[4 + j];
    return out;
}
__device__ inline f32x4 ahead(f32x4 lo, f32x4 hi, bool c1, bool c2) {   // seq[j + c]
    const float seq[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    float t[6];
#pragma unroll
    for (int k = 0; k < 6; k++) t[k] = c1 ? seq[k + 1] : seq[k];
    f32x4 out;
#pragma unroll
    for (int j = 0; j < 4; j++) out[j] = c2 ? t[j + 2] : t[j];
    return out;
}

template <int KIND>
__global__ void __launch_bounds__(WF_THREADS) k_wave_2d(WaveArgs A, SideWork W) {
#pragma clang fp contract(off)
    constexpr bool FWD = Kind<KIND>::FWD, UPD = KIND == WAVE_FWD_UPDATE;
    if (blockIdx.x > 0) {
        const Part part{blockIdx.x - 1, W.blocks};
        if constexpr (UPD) {
            update_r<WF_THREADS>(part, W.n, W.flags, W.q, W.r, W.r_next, W.red);
        } else if constexpr (KIND == WAVE_BWD) {
            dot_self<WF_THREADS>(part, W.n, W.flags, W.t, W.red);
            if (W.x_steps == 2) update_x_chunks<2>(part, W.n, W.flags, W.x, W.red.sc);
        }
        return;
    }
    extern __shared__ __align__(16) uint32_t edges[];   // row w: what wave w hands to wave w + 1
    __shared__ int done[WF_THREADS / WF_TZ];            // groups of steps that wave w has finished
    const int xa = __builtin_amdgcn_readfirstlane(A.xrange[0]), xb = __builtin_amdgcn_readfirstlane(A.xrange[1]);
    if (xb < xa) return;   // no WATER
    const int g0 = xa / WF_G, g1 = xb / WF_G, ng = g1 - g0 + 1;
    const int steps = groups_2d(ng), elen = edge_2d(ng);
    const int nwaves = (A.ny - 2 + WF_TZ - 1) / WF_TZ;
    for (int i = threadIdx.x; i < (nwaves - 1) * elen; i += WF_THREADS) edges[i] = 0;
    if (threadIdx.x < WF_THREADS / WF_TZ) done[threadIdx.x] = 0;
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WF_TZ), lane = threadIdx.x % WF_TZ;
    if (w >= nwaves) return;
    const uint32_t gstride = (uint32_t)A.ny * 3u * 16u, total = gstride * (uint32_t)(A.nxp / WF_G);
    const __amdgpu_buffer_rsrc_t rP = rsrc(A.P32, (int64_t)total), rI = rsrc(A.in, (int64_t)total),
                                 rO = rsrc(A.out, (int64_t)total), rQ = rsrc(UPD ? W.q : A.in, (int64_t)total);
    const float ms = A.ms;
    const float malpha = UPD ? (float)(-W.red.sc->alpha) : 0.f;
    const int row = WF_TZ * w + lane, q = lane / WF_G;
    const bool in_grid = row < A.ny - 2, c1 = (lane & 1) != 0, c2 = (lane & 2) != 0;
    const uint32_t column = (uint32_t)((FWD ? 1 + row : A.ny - 2 - row) * 3 + 1) * 16u;
    // byte offset of the lane's k-th group in the order of the march, beyond the arrays if it has none
    auto at = [&](int k) {
        return in_grid && (unsigned)k < (unsigned)ng ? (uint32_t)(FWD ? g0 + k : g1 - k) * gstride + column : kOob;
    };
    auto marched = [](f32x4 v) { return FWD ? v : f32x4{v[3], v[2], v[1], v[0]}; };
    f32x4 pv[k2dAhead], iv[k2dAhead], uv[k2dAhead];
    auto fetch = [&](auto dc, int g) {
        constexpr int d = decltype(dc)::value;
        const uint32_t o = at(g - q);
        pv[d] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rP, o, 0, 0));
        iv[d] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rI, o, 0, 0));
        if constexpr (UPD) uv[d] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rQ, o, 0, 0));
    };
    unroll<k2dAhead>([&](auto dc) { fetch(dc, decltype(dc)::value); });
    // the row above the wave's first: elements 4 g .. 4 g + 3 once wave w - 1 has done g + k2dLag groups
    const uint32_t* const above = edges + (w - 1) * elen + k2dPad;
    uint32_t* const below = edges + w * elen + k2dPad;
    u32x4 edge = {0, 0, 0, 0};
    auto wait_edge = [&](int g) {
        if (w == 0) return;
        const int need = min(g + k2dLag, steps);
        int spins = 0;
        for (;;) {
            const int have = lget(&done[w - 1]);
            edge = lget4(above + WF_G * min(g, steps - 1));
            if (__builtin_amdgcn_readfirstlane(have) >= need) return;
            if ((++spins & 1023) == 0 && (spins >= kSpinLimit || gave_up(A.err))) {
                if (lane == 0) atomicOr(A.err, 1);
                return;   // carry on with whatever is there
            }
        }
    };
    wait_edge(0);
    const f32x4 none = {0.f, 0.f, 0.f, 0.f};
    f32x4 plo = none, ilo = none, rlo = none;   // the group of steps before: operands and results
    float m = 0.f;                              // what the lane passed on at the step before
    for (int g8 = 0; g8 < steps; g8 += k2dAhead) {
        unroll<k2dAhead>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            const int g = g8 + d;
            const f32x4 phi = marched(pv[d]);
            f32x4 ihi = marched(iv[d]);
            if constexpr (UPD) {
                const f32x4 u = marched(uv[d]);
#pragma unroll
                for (int j = 0; j < 4; j++) ihi[j] = __builtin_fmaf(u[j], malpha, ihi[j]);
            }
            fetch(dc, g + k2dAhead);
            const f32x4 p = behind(plo, phi, c1, c2), in = behind(ilo, ihi, c1, c2);
            plo = phi;
            ilo = ihi;
            f32x4 res;
            float pass[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // +-y: lane l - 1's value of the step before, the upstream wave's on lane 0
                const float up = __builtin_bit_cast(
                    float, __builtin_amdgcn_update_dpp((int)edge[j], __builtin_bit_cast(int, m), 0x138, 0xf, 0xf, false));
                const float acc = m + up;
                float outv, v;
                if (FWD) {
                    outv = on_water<KIND>((in[j] - acc) * p[j], p[j]);
                    v = outv * p[j];
                } else {
                    outv = on_water<KIND>((in[j] - acc * p[j]) * p[j], p[j]);
                    v = outv;
                }
                m = __builtin_fmaf(ms, v, 0.f);
                res[j] = outv;
                pass[j] = m;
            }
            if (w + 1 < nwaves && lane == WF_TZ - 1) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *(lds_u32*)(below + WF_G * (g - 15) + j - 3) = __builtin_bit_cast(uint32_t, pass[j]);
                lput(&done[w], g + 1);
            }
            const f32x4 whole = marched(ahead(rlo, res, c1, c2));
            rlo = res;
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, whole), rO, at(g - q - 1), 0, 0);
            wait_edge(g + 1);
        });
    }
}

int wave_launch(fsim_ctx* ctx, WaveKind kind, const float* in, float* out, double scale, const SideWork* side) {
    WaveArgs A = ctx->wave;
    A.in = in;
    A.out = out;
    A.scale = scale;
    A.ms = -(float)scale;
    if (kind != WAVE_FACTOR && fits_2d(A)) {
        const SideWork W = side ? *side : SideWork{};
        const dim3 grid(1 + W.blocks), block(WF_THREADS);
        const size_t lds = lds_2d(A.ny, A.nxp);
        if (kind == WAVE_FWD) hipLaunchKernelGGL(k_wave_2d<WAVE_FWD>, grid, block, lds, ctx->stream, A, W);
        else if (kind == WAVE_BWD) hipLaunchKernelGGL(k_wave_2d<WAVE_BWD>, grid, block, lds, ctx->stream, A, W);
        else if (kind == WAVE_FWD_ALONE) hipLaunchKernelGGL(k_wave_2d<WAVE_FWD_ALONE>, grid, block, lds, ctx->stream, A, W);
        else if (kind == WAVE_BWD_ALONE) hipLaunchKernelGGL(k_wave_2d<WAVE_BWD_ALONE>, grid, block, lds, ctx->stream, A, W);
        else hipLaunchKernelGGL(k_wave_2d<WAVE_FWD_UPDATE>, grid, block, lds, ctx->stream, A, W);
        FSIM_HIP(ctx, hipGetLastError());
        return FSIM_OK;
    }
    const unsigned ntiles = (unsigned)(A.TJ * A.TK);
    const int counter = kind == WAVE_FACTOR ? 0 : kind == WAVE_BWD || kind == WAVE_BWD_ALONE ? 2 : 1;
    A.ticket = ctx->wave_ticket + counter;
    A.ticket_base = ctx->wave_ticket_base[counter];
    ctx->wave_ticket_base[counter] += ntiles;
    A.send_delay = ctx->wave_send_delay;
    // the blocks beside the tiles come last: the tiles, which wait for each other, start first
    const SideWork W = side ? *side : SideWork{};
    const dim3 grid(ntiles + W.blocks), block(WF_THREADS);
    switch (kind) {
    case WAVE_FACTOR: hipLaunchKernelGGL(k_wave<WAVE_FACTOR>, grid, block, 0, ctx->stream, A, W); break;
    case WAVE_FWD: hipLaunchKernelGGL(k_wave<WAVE_FWD>, grid, block, 0, ctx->stream, A, W); break;
    case WAVE_BWD: hipLaunchKernelGGL(k_wave<WAVE_BWD>, grid, block, 0, ctx->stream, A, W); break;
    case WAVE_FWD_ALONE: hipLaunchKernelGGL(k_wave<WAVE_FWD_ALONE>, grid, block, 0, ctx->stream, A, W); break;
    case WAVE_BWD_ALONE: hipLaunchKernelGGL(k_wave<WAVE_BWD_ALONE>, grid, block, 0, ctx->stream, A, W); break;
    case WAVE_FWD_UPDATE: hipLaunchKernelGGL(k_wave<WAVE_FWD_UPDATE>, grid, block, 0, ctx->stream, A, W); break;
    }
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

}  // namespace fsim
