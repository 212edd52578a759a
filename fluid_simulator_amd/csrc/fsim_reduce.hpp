// Block reductions and streaming passes over solver vectors, for the solver's
// own kernels and for the blocks that the triangular sweeps run beside their
// tiles (SideWork).
#pragma once
#include "fsim_internal.hpp"

namespace fsim {

// ---- block reductions (FP64, fixed order) ------------------------------------
__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_down(v, d, 64);
    return v;
}
__device__ inline double wave_max(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmax(v, __shfl_down(v, d, 64));
    return v;
}
// ---- in-kernel finish of a reduction -------------------------------------------------
// Each block reduces its values to one partial (plus an aux value: max or sum)
// and stores it with device-scope stores; once they are acknowledged the block
// takes a ticket from a device-scope counter.  The block with the last ticket
// sums all partials in a fixed order (thread t: partials t, t + kBlock, ...,
// then a pairwise tree), applies the reduction's scalar update and resets the
// counter.  The sum's order does not depend on which block is last, so the
// result is deterministic, and no separate finalize launch is needed.
constexpr int AUX_NONE = 0, AUX_MAX = 1, AUX_SUM = 2;
enum FinOp {
    FIN_NONE = -1, FIN_BB = 0, FIN_SIGMA0 = 1, FIN_ALPHA = 2, FIN_RES = 3, FIN_BETA = 4, FIN_TRUE = 5, FIN_FBETA = 6,
    FIN_ALPHA_ZR = 7
};

struct Reduce {
    double* partials;   // 2 x gridDim.x
    unsigned* count;    // zero between launches
    SolveScalars* sc;
    int op;             // FinOp
    SolveScalars* host = nullptr;   // pinned host copy written by the finishing block, or null
    unsigned seq = 0;               // what the host waits for in it (host->seq)
    const int* wave_err = nullptr;  // the wavefront kernels' error flag, copied along
};

__device__ inline void apply_fin(int op, double s, double m, SolveScalars* sc) {
    switch (op) {
    case FIN_BB: sc->bb = s; sc->nfluid = m; break;
    case FIN_SIGMA0: sc->zr = s; break;
    case FIN_ALPHA:      // sigma is the last z.r (initial, restart or beta step)
    case FIN_ALPHA_ZR: { // sigma = m, z.r summed beside s.q
        sc->sigma = op == FIN_ALPHA ? sc->zr : m;
        sc->sq = s;
        const double alpha = sc->sigma / s;
        sc->alpha_prev = sc->alpha;
        sc->alpha = alpha;
        if (alpha != alpha) sc->nan_flag |= 1;
        break;
    }
    case FIN_RES: sc->rr = s; sc->rmax = m; break;
    case FIN_BETA: {
        if (sc->sigma != sc->sigma) sc->nan_flag |= 2;   // the reference tests the old sigma (:285-286)
        sc->zr = s;
        sc->beta = s / sc->sigma;
        break;
    }
    case FIN_TRUE: sc->tr_ss = s; sc->tr_max = m; break;
    case FIN_FBETA: {   // s = z'.r', m = z'.q.  Flexible PCG: beta = z'.(r' - r) / z.r = -alpha z'.q / z.r
        if (sc->sigma != sc->sigma) sc->nan_flag |= 2;
        sc->zr = s;
        sc->beta = -sc->alpha * m / sc->sigma;
        break;
    }
    default: break;
    }
}

__device__ inline void put_dev(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline double get_dev(const double* p) {
    return __builtin_bit_cast(double, __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT));
}

// The blocks that share a streaming pass or a reduction: all of the grid, or
// the ones that a kernel runs beside its tiles.
struct Part {
    unsigned id, n;
};
__device__ inline Part whole_grid() { return Part{blockIdx.x, gridDim.x}; }

template <int AUX, int NT = kBlock>
__device__ void block_finish(double sum, double aux, const Reduce& R, const Part part) {
    constexpr int kTree = NT <= 256 ? 256 : NT <= 512 ? 512 : 1024;   // the pairwise tree's width
    static_assert(NT <= 1024 && kTree % 64 == 0, "threads of a block");
    __shared__ double lds_s[kTree], lds_m[kTree];
    __shared__ int last;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    sum = wave_sum(sum);
    if (AUX == AUX_MAX) aux = wave_max(aux);
    if (AUX == AUX_SUM) aux = wave_sum(aux);
    if (lane == 0) {
        lds_s[wave] = sum;
        lds_m[wave] = aux;
    }
    __syncthreads();
    const unsigned nparts = part.n;
    if (threadIdx.x == 0) {
        double s = 0, m = 0;
        for (int w = 0; w < NT / 64; w++) {
            s += lds_s[w];
            m = AUX == AUX_SUM ? m + lds_m[w] : fmax(m, lds_m[w]);
        }
        put_dev(&R.partials[part.id], s);
        if (AUX != AUX_NONE) put_dev(&R.partials[nparts + part.id], m);
        __builtin_amdgcn_s_waitcnt(0);   // the partials are acknowledged before the ticket
        last = __hip_atomic_fetch_add(R.count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nparts - 1;
    }
    __syncthreads();
    if (!last) return;
    // all loads first (at most kMaxParts / NT per thread), then the sums in order
    constexpr int kPer = (kMaxParts + NT - 1) / NT;
    double vs[kPer], vm[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const unsigned i = threadIdx.x + k * NT;
        vs[k] = i < nparts ? get_dev(&R.partials[i]) : 0.0;
        vm[k] = AUX != AUX_NONE && i < nparts ? get_dev(&R.partials[nparts + i]) : 0.0;
    }
    double s = 0, m = 0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        s += vs[k];
        m = AUX == AUX_SUM ? m + vm[k] : fmax(m, vm[k]);
    }
    lds_s[threadIdx.x] = s;
    lds_m[threadIdx.x] = m;
    if ((int)threadIdx.x + NT < kTree) lds_s[threadIdx.x + NT] = lds_m[threadIdx.x + NT] = 0.0;   // (kTree <= 2 NT)
    __syncthreads();
    for (int off = kTree / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            lds_s[threadIdx.x] += lds_s[threadIdx.x + off];
            lds_m[threadIdx.x] = AUX == AUX_SUM ? lds_m[threadIdx.x] + lds_m[threadIdx.x + off]
                                                : fmax(lds_m[threadIdx.x], lds_m[threadIdx.x + off]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        apply_fin(R.op, lds_s[0], lds_m[0], R.sc);
        __hip_atomic_store(R.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (R.host) {
            // the words the host tests after the reduction straight into pinned host memory with
            // system-scope stores, the word with seq, which the host polls, when the others have been
            // acknowledged
            auto put_host = [](void* dst, uint64_t v) {
                __hip_atomic_store(reinterpret_cast<uint64_t*>(dst), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            };
            double* const to = R.op == FIN_BB ? &R.host->bb : R.op == FIN_TRUE ? &R.host->tr_ss : &R.host->rr;
            double* const to2 = R.op == FIN_BB ? &R.host->nfluid : R.op == FIN_TRUE ? &R.host->tr_max : &R.host->rmax;
            put_host(to, __builtin_bit_cast(uint64_t, lds_s[0]));
            put_host(to2, __builtin_bit_cast(uint64_t, lds_m[0]));
            if (R.wave_err)
                put_host(&R.host->wave_err,
                         (uint64_t)(uint32_t)__hip_atomic_load(R.wave_err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            __builtin_amdgcn_s_waitcnt(0);
            static_assert(offsetof(SolveScalars, seq) == offsetof(SolveScalars, nan_flag) + 4, "one 8-byte word");
            put_host(&R.host->nan_flag, (uint32_t)R.sc->nan_flag | (uint64_t)R.seq << 32);
        }
    }
}
template <int AUX, int NT = kBlock>
__device__ void block_finish(double sum, double aux, const Reduce& R) {
    block_finish<AUX, NT>(sum, aux, R, whole_grid());
}

constexpr int kChunk = 256;   // values of a solver vector per chunk flag (the streaming kernels)

// Streaming kernels without per-cell masks: the solver vectors r, q and z
// are exactly zero off WATER (zeroed at the start of a solve, written with
// zeros there), so the extra terms are exact zeros.  The vectors are cut
// into chunks of 256 values (16 bytes per lane); a chunk without WATER is
// skipped.  Its flag is one 32-bit word (built with nbinfo for every solve),
// so a wave reads it with a scalar load; a wave takes kUnits chunks per trip
// (grid stride) and issues all their loads before using any, so several
// memory round trips are in flight.
constexpr int kUnits = 4;
template <int NV, class Load, class Use>
__device__ inline void for_flagged_chunks(const Part part, int64_t n, const uint32_t* __restrict__ flags, Load&& load, Use&& use) {
    const int lane = threadIdx.x & 63;
    const int nchunks = (int)((n + kChunk - 1) / kChunk);
    const int nwaves = (int)(part.n * (blockDim.x / 64));
    const int w0 = __builtin_amdgcn_readfirstlane((int)(part.id * (blockDim.x / 64) + (threadIdx.x >> 6)));
    for (int u0 = w0; u0 < nchunks; u0 += kUnits * nwaves) {
        uint32_t f[kUnits];
#pragma unroll
        for (int k = 0; k < kUnits; k++) {
            const int u = u0 + k * nwaves;
            f[k] = u < nchunks ? flags[u] : 0u;
        }
        // loads without branches (a skipped lane reads cell 0 and uses nothing), so that all
        // kUnits x NV loads are issued before the first wait
        float4 v[kUnits][NV];
        bool on[kUnits];
        int64_t at[kUnits];
#pragma unroll
        for (int k = 0; k < kUnits; k++) {
            const int64_t i = (int64_t)(u0 + k * nwaves) * kChunk + 4 * lane;
            on[k] = f[k] != 0u && i < n;
            at[k] = on[k] ? i : 0;
            load(at[k], v[k]);
        }
#pragma unroll
        for (int k = 0; k < kUnits; k++)
            if (on[k]) use(at[k], v[k]);
    }
}

// x += alpha s (FP64) for WATER cells, of the last direction step (STEPS 1) or
// of the last two in their order (STEPS 2: s_prev and the alpha before).  A NaN
// alpha leaves x as it is: the reference breaks before multAdd
// (bridsonSolverGrid.cpp:270-272) and applies the last pressure.
struct UpdateX {
    const uint16_t* nbinfo;
    const float *s_prev, *s;
    double* x;
};
template <int STEPS>
__device__ inline void update_x_chunks(const Part part, int64_t n, const uint32_t* __restrict__ flags, const UpdateX& A,
                                       const SolveScalars* __restrict__ sc) {
    const int lane = threadIdx.x & 63;
    const int nchunks = (int)((n + kChunk - 1) / kChunk);
    const int nwaves = (int)(part.n * (blockDim.x / 64));
    const double alpha_prev = sc->alpha_prev, alpha = sc->alpha;
    const bool last = !(sc->nan_flag & 1);
    // kUnits chunks a trip, all loads first, as for_flagged_chunks
    for (int u0 = __builtin_amdgcn_readfirstlane((int)(part.id * (blockDim.x / 64) + (threadIdx.x >> 6))); u0 < nchunks;
         u0 += kUnits * nwaves) {
        u16x4 nb[kUnits];
        f64x4 v[kUnits];
        f32x4 a[kUnits], b[kUnits];
        bool on[kUnits];
        int64_t at[kUnits];
#pragma unroll
        for (int k = 0; k < kUnits; k++) {
            const int u = u0 + k * nwaves;
            const int64_t i = (int64_t)u * kChunk + 4 * lane;
            on[k] = (u < nchunks ? flags[u] : 0u) != 0u && i < n;
            at[k] = on[k] ? i : 0;
        }
#pragma unroll
        for (int k = 0; k < kUnits; k++) {
            nb[k] = *reinterpret_cast<const u16x4*>(A.nbinfo + at[k]);
            v[k] = *reinterpret_cast<const f64x4*>(A.x + at[k]);
            if constexpr (STEPS == 2) a[k] = *reinterpret_cast<const f32x4*>(A.s_prev + at[k]);
            b[k] = *reinterpret_cast<const f32x4*>(A.s + at[k]);
        }
#pragma unroll
        for (int k = 0; k < kUnits; k++) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (!(nb[k][c] & NB_FLUID)) continue;
                if constexpr (STEPS == 2) v[k][c] += (double)a[k][c] * alpha_prev;
                if (last) v[k][c] += (double)b[k][c] * alpha;
            }
            if (on[k]) *reinterpret_cast<f64x4*>(A.x + at[k]) = v[k];
        }
    }
}

// r_next = r - alpha q, with ||r_next||^2 and max|r_next|.  The forward sweep
// computes the same r_next for itself: one fused multiply-add in both.
template <int NT>
__device__ inline void update_r(const Part part, int64_t n, const uint32_t* __restrict__ flags, const float* q,
                                const float* r, float* r_next, const Reduce& red) {
    double ss = 0.0, mx = 0.0;
    const float malpha = (float)(-red.sc->alpha);
    auto cell = [&](float qv, float& rv) {
        rv = __builtin_fmaf(qv, malpha, rv);
        ss += (double)rv * (double)rv;
        mx = fmax(mx, fabs((double)rv));
    };
    for_flagged_chunks<2>(
        part, n, flags,
        [&](int64_t i, float4(&v)[2]) {
            v[0] = *reinterpret_cast<const float4*>(q + i);
            v[1] = *reinterpret_cast<const float4*>(r + i);
        },
        [&](int64_t i, float4(&v)[2]) {
            cell(v[0].x, v[1].x);
            cell(v[0].y, v[1].y);
            cell(v[0].z, v[1].z);
            cell(v[0].w, v[1].w);
            *reinterpret_cast<float4*>(r_next + i) = v[1];
        });
    block_finish<AUX_MAX, NT>(ss, mx, red, part);
}

// a . b over this thread's part of the flagged chunks (FP64 products of the FP32 values)
__device__ inline double dot_part(const Part part, int64_t n, const uint32_t* __restrict__ flags, const float* __restrict__ a,
                                  const float* __restrict__ b) {
    double d = 0.0;
    for_flagged_chunks<2>(
        part, n, flags,
        [&](int64_t i, float4(&v)[2]) {
            v[0] = *reinterpret_cast<const float4*>(a + i);
            v[1] = *reinterpret_cast<const float4*>(b + i);
        },
        [&](int64_t, float4(&v)[2]) {
            d += (double)v[0].x * (double)v[1].x;
            d += (double)v[0].y * (double)v[1].y;
            d += (double)v[0].z * (double)v[1].z;
            d += (double)v[0].w * (double)v[1].w;
        });
    return d;
}

// t . t (FP64 products of the FP32 values)
template <int NT>
__device__ inline void dot_self(const Part part, int64_t n, const uint32_t* __restrict__ flags, const float* t,
                                const Reduce& red) {
    double d = 0.0;
    for_flagged_chunks<1>(
        part, n, flags, [&](int64_t i, float4(&v)[1]) { v[0] = *reinterpret_cast<const float4*>(t + i); },
        [&](int64_t, float4(&v)[1]) {
            d += (double)v[0].x * (double)v[0].x;
            d += (double)v[0].y * (double)v[0].y;
            d += (double)v[0].z * (double)v[0].z;
            d += (double)v[0].w * (double)v[0].w;
        });
    block_finish<AUX_NONE, NT>(d, 0.0, red, part);
}

// What the blocks behind a sweep's tiles do.  Beside the forward sweep of an
// iteration: r_next and its norms.  Beside the backward sweep: t . t of the
// forward sweep's result t, and x += alpha s of the last x_steps (0 or 2)
// direction steps.
struct SideWork {
    unsigned blocks = 0;   // 0: none
    int64_t n = 0;
    const uint32_t* flags = nullptr;
    const float *q = nullptr, *r = nullptr;   // forward
    float* r_next = nullptr;
    const float* t = nullptr;                 // backward
    UpdateX x{};
    int x_steps = 0;
    Reduce red{};
};

}  // namespace fsim
