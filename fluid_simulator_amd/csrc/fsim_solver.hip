// fsim_solver.hip — Bridson pressure projection on gfx950.
//
// BridsonSolverGrid::solveIncompressibility (bridsonSolverGrid.cpp:244-293)
// over dense vectors with a WATER mask:
//   * b = -(1/dx) div(v2) [+ density term] evaluated in FP64, stored FP32;
//   * A is matrix-free: diag = scale * #non-SOLID neighbours, off-diagonal
//     -scale towards each WATER neighbour (calculateAMatrix, :40-77);
//   * MIC(0) factor (calculatePreconditioner, :91-124) in FP64 with the
//     reference's expression order, level-scheduled on i+j+k planes: every
//     cell depends only on its -x/-y/-z neighbours, so any topological order
//     gives the serial loop's values;
//   * MIC(0) apply (:126-163): forward/backward triangular sweeps in FP32,
//     level-scheduled the same way;
//   * PCG with FP32 vectors, FP64 pressure, FP64 dot products (deterministic
//     block partials summed in a fixed order) and FP64 reliable updates: when
//     the recursive residual meets the tolerance, the true residual b - A x is
//     recomputed in FP64; the solve stops only if that meets the tolerance,
//     otherwise r is replaced by it and the iteration continues.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <thread>
#include <type_traits>

#include "fsim_march.hpp"
#include "fsim_reduce.hpp"

namespace fsim {

// ---- RHS and neighbour masks (calculateRHS :79-89, calculateAMatrix :40-77) ------
struct RhsArgs {
    SolveArgs S;
    const uint8_t* label;
    const float* u2;
    const float* v2;
    const float* w2;
    const float* density;
    uint16_t* info_flat;   // masks and b in flat order (k_rotate moves them to the solver's layout)
    float* b_flat;
    uint8_t* colw;   // set to 1 for the (y, z) column of each WATER cell (cleared before)
    uint8_t* xw;     // the same for the x rows
    double inv_dx;
    double avg_p, pk;
    int pressure_enabled;
    Reduce red;   // FIN_BB: ||b||^2 and the WATER cell count
};

__device__ inline bool is_fluid(const SolveArgs& S, const uint8_t* label, int x, int y, int z) {
    return x > 0 && y > 0 && z > 0 && x < S.nx - 1 && y < S.ny - 1 && z < S.nz - 1 && label[sidx(S, x, y, z)] == FSIM_WATER;
}

// Neighbour mask of interior cell (x, y, z), 0 unless it is WATER.
__device__ inline uint16_t neighbour_mask(const SolveArgs& S, const uint8_t* label, int x, int y, int z) {
    if (!is_fluid(S, label, x, y, z)) return 0;
    const int64_t st[3] = {(int64_t)S.ny * S.nz, S.nz, 1};
    const int64_t i = sidx(S, x, y, z);
    uint16_t info = NB_FLUID;
    int nonsolid = 0;
    const int p[3] = {x, y, z};
    for (int a = 0; a < 3; a++) {
        int qp[3] = {p[0], p[1], p[2]}, qm[3] = {p[0], p[1], p[2]};
        qp[a] += 1;
        qm[a] -= 1;
        uint8_t lp = label[i + st[a]], lm = label[i - st[a]];
        if (lp != FSIM_SOLID) nonsolid++;
        if (lm != FSIM_SOLID) nonsolid++;
        if (is_fluid(S, label, qp[0], qp[1], qp[2])) info |= (uint16_t)(NB_PX << a);
        if (is_fluid(S, label, qm[0], qm[1], qm[2])) info |= (uint16_t)(NB_MX << a);
    }
    info |= (uint16_t)(nonsolid << NB_NONSOLID_SHIFT);
    // for each -a neighbour that is WATER: are its +(a+1)%3 and
    // +(a+2)%3 neighbours WATER (the MIC(0) "other" off-diagonals)
    for (int a = 0; a < 3; a++) {
        if (!(info & (NB_MX << a))) continue;
        for (int k = 0; k < 2; k++) {
            const int b = (a + 1 + k) % 3;
            int q[3] = {p[0], p[1], p[2]};
            q[a] -= 1;
            q[b] += 1;
            if (is_fluid(S, label, q[0], q[1], q[2])) info |= (uint16_t)(1u << (NB_UP_SHIFT + 2 * a + k));
        }
    }
    return info;
}

__global__ void __launch_bounds__(kBlock) k_nbinfo_rhs(RhsArgs A, int with_rhs) {
#pragma clang fp contract(off)
    const SolveArgs& S = A.S;
    double bsq = 0.0, nfl = 0.0;
    const int nrows = S.nx * S.ny;
    // lanes along z, as many grid rows (x, y) per block iteration as fit.  With one row at a time the blocks
    // of a 2D grid waited for memory 85 times over (us: 128 x 128 88 -> 5, 32^3 16 -> 10, 128^3 42 -> 35)
    int wide = 4;
    while (wide < S.nz && wide < kBlock) wide *= 2;
    const int per = kBlock / wide;
    for (int row = blockIdx.x * per + threadIdx.x / wide; row < nrows; row += gridDim.x * per)
    for (int z = threadIdx.x & (wide - 1); z < S.nz; z += wide) {
        const int x = row / S.ny, y = row - x * S.ny;
        const int64_t i = (int64_t)row * S.nz + z;
        const uint16_t info = neighbour_mask(S, A.label, x, y, z);
        float bv = 0.f;
        if (info) {
            nfl += 1.0;
            A.colw[y * S.nz + z] = 1;
            A.xw[x] = 1;
            if (with_rhs) {
                double dv = (double)A.u2[i] + (double)A.v2[i] + (double)A.w2[i] - (double)A.u2[i - (int64_t)S.ny * S.nz] -
                            (double)A.v2[i - S.nz] - (double)A.w2[i - 1];
                double bd = -A.inv_dx * dv +
                            (A.pressure_enabled ? ((double)A.density[i] - A.avg_p) * A.pk : 0.0);
                bsq += bd * bd;
                bv = (float)bd;
            }
        }
        A.info_flat[i] = info;
        if (with_rhs) A.b_flat[i] = bv;
    }
    if (with_rhs) block_finish<AUX_SUM>(bsq, nfl, A.red);
}

// Masks and b from flat order into the solver's layout, with the chunk flags.
// A block item: W planes of one row y and one z-tile.  The cells of a rotated
// plane lie in 64 different x rows, so the block reads flat rows (lanes along
// z), puts them into LDS by plane, and writes each column's groups of four
// planes with 8- and 16-byte stores; every interior column's value moves once.
// The right-hand-side kernel used to scatter 2- and 4-byte values over 64
// planes itself: 0.57 ms at 256^3, 0.27 ms for the two kernels.
template <int W>
__global__ void __launch_bounds__(kBlock) k_rotate(SolveArgs S, const uint16_t* __restrict__ info_flat,
                                                   const float* __restrict__ b_flat, uint16_t* __restrict__ nbinfo,
                                                   float* __restrict__ b, uint32_t* __restrict__ flags,
                                                   const uint8_t* __restrict__ colw, const uint8_t* __restrict__ xw,
                                                   int* __restrict__ xrange, uint8_t* __restrict__ tilew) {
    __shared__ uint16_t info_lds[W][WF_TZ];
    __shared__ float b_lds[W][WF_TZ];
    constexpr int nwaves = kBlock / 64, kRows = (W + WF_TZ - 1 + nwaves - 1) / nwaves;   // rows per wave
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ntile = (S.nz - 2 + WF_TZ - 1) / WF_TZ;
    const int k = blockIdx.x;
    const int z0 = 1 + k % ntile * WF_TZ, y = 1 + k / ntile % (S.ny - 2), p0 = k / (ntile * (S.ny - 2)) * W;
    const int np = min(W, S.nxp - p0), cols = min(WF_TZ, S.nz - 1 - z0);
    const int z = z0 + lane;
    // row t (x = t mod nxp) holds the cells of planes t + lane; loads in batches of 8 rows
    for (int k0 = 0; k0 < kRows; k0 += 8) {
        uint16_t n[8];
        float v[8];
        int slot[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int t = p0 - (cols - 1) + (k0 + j) * nwaves + wave;
            const int p = t + lane;
            const int x = t >= 0 ? (t < S.nxp ? t : 0) : (t % S.nxp + S.nxp) % S.nxp;
            const bool on = k0 + j < kRows && lane < cols && p >= p0 && p < p0 + np;
            const bool cell = on && x < S.nx;
            const int64_t i = cell ? sidx(S, x, y, z) : 0;
            slot[j] = on ? (p - p0) * WF_TZ + lane : -1;
            n[j] = cell ? info_flat[i] : (uint16_t)0;
            v[j] = cell && b_flat ? b_flat[i] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (slot[j] >= 0) {
                (&info_lds[0][0])[slot[j]] = n[j];
                (&b_lds[0][0])[slot[j]] = v[j];
            }
    }
    // which wavefront tiles hold WATER: a wave per tile and direction (fewer than this kernel's blocks)
    const int tk = (S.nz - 2 + WF_TZ - 1) / WF_TZ, tiles = (S.ny - 2 + WF_TY - 1) / WF_TY * tk;
    if (k < 2 * tiles && wave == 1) {
        const bool fwd = k < tiles;
        const int J = (fwd ? k : k - tiles) / tk, K = (fwd ? k : k - tiles) % tk;
        const int z = 1 + (fwd ? K : tk - 1 - K) * WF_TZ + lane;
        bool any = false;
#pragma unroll
        for (int ty = 0; ty < WF_TY; ty++) {
            const int row = J * WF_TY + ty;
            if (row < S.ny - 2 && z <= S.nz - 2) any = any || colw[(fwd ? 1 + row : S.ny - 2 - row) * S.nz + z] != 0;
        }
        const bool water = __any(any);
        if (lane == 0) tilew[k] = water ? 1 : 0;
    }
    if (k == 0 && wave == 0) {   // the x range with WATER, for the wavefront kernels
        int xlo = S.nx, xhi = -1;
        for (int x = lane; x < S.nx; x += 64)
            if (xw[x]) {
                xlo = min(xlo, x);
                xhi = x;
            }
        for (int d = 32; d >= 1; d >>= 1) {
            xlo = min(xlo, __shfl_down(xlo, d, 64));
            xhi = max(xhi, __shfl_down(xhi, d, 64));
        }
        if (lane == 0) {
            xrange[0] = xlo;
            xrange[1] = xhi;
        }
    }
    __syncthreads();
    if (lane >= cols) return;
    for (int g = wave; g < np / WF_G; g += nwaves) {
        const int64_t i = pidx(p0 + g * WF_G, y, z, S.ny, S.nz);
        u16x4 n;
        f32x4 v;
#pragma unroll
        for (int c = 0; c < WF_G; c++) {
            n[c] = info_lds[g * WF_G + c][lane];
            v[c] = b_lds[g * WF_G + c][lane];
        }
        *reinterpret_cast<u16x4*>(nbinfo + i) = n;
        if (b_flat) *reinterpret_cast<f32x4*>(b + i) = v;
        if ((n[0] | n[1] | n[2] | n[3]) & NB_FLUID) flags[i / kChunk] = 1u;
    }
}

// ---- MIC(0) factor, one i+j+k plane per launch (FP64) -----------------------------
struct PlaneArgs {
    SolveArgs S;
    const uint16_t* nbinfo;
    int level;
};

__device__ inline bool plane_cell(const PlaneArgs& A, int64_t t, int& x, int& y, int& z) {
    const SolveArgs& S = A.S;
    const int ny_in = S.ny - 2;
    x = 1 + (int)(t / ny_in);
    y = 1 + (int)(t % ny_in);
    z = A.level - x - y;
    return x < S.nx - 1 && z >= 1 && z < S.nz - 1;
}

__global__ void __launch_bounds__(kBlock) k_mic_factor_plane(PlaneArgs A, double* __restrict__ P64, float* __restrict__ P32) {
#pragma clang fp contract(off)
    const SolveArgs& S = A.S;
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int x, y, z;
    if (!plane_cell(A, t, x, y, z)) return;
    int64_t i = rsidx(S, x, y, z);
    uint16_t info = A.nbinfo[i];
    if (!(info & NB_FLUID)) return;
    const double tau = 0.97, sigma = 0.25, scale = S.scale;
    double eneg = 0, eneg_tau = 0;
    for (int a = 0; a < 3; a++) {
        if (!(info & (NB_MX << a))) continue;
        int64_t j = rnb_minus(S, x, y, z, a);
        double pj = P64[j];
        double ap = -scale * pj;   // xWater of the -neighbour times its precon
        double o1 = (info & (1u << (NB_UP_SHIFT + 2 * a))) ? -scale : 0.0;
        double o2 = (info & (1u << (NB_UP_SHIFT + 2 * a + 1))) ? -scale : 0.0;
        eneg += ap * ap;
        eneg_tau += ap * (o1 + o2) * pj;
    }
    int cnt = (info >> NB_NONSOLID_SHIFT) & 7;
    double diag = 0;
    for (int k = 0; k < cnt; k++) diag += scale;
    double e = diag - eneg - eneg_tau * tau;
    if (e < sigma * diag) e = diag < 1e-6 ? 1.0 : diag;
    double p = 1.0 / sqrt(e);
    P64[i] = p;
    P32[i] = (float)p;
}

// ---- MIC(0) apply: forward and backward sweeps, one plane per launch (FP32) -------
// Contraction is off in both sweep implementations so that they round alike.
__global__ void __launch_bounds__(kBlock) k_fwd_plane(PlaneArgs A, const float* __restrict__ r, float* __restrict__ q,
                                                      const float* __restrict__ P) {
#pragma clang fp contract(off)
    const SolveArgs& S = A.S;
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int x, y, z;
    if (!plane_cell(A, t, x, y, z)) return;
    int64_t i = rsidx(S, x, y, z);
    uint16_t info = A.nbinfo[i];
    if (!(info & NB_FLUID)) return;
    const float ms = -S.scale_f;
    float qneg = 0.f;
#pragma unroll
    for (int a = 0; a < 3; a++)
        if (info & (NB_MX << a)) {
            const int64_t j = rnb_minus(S, x, y, z, a);
            qneg += ms * (q[j] * P[j]);
        }
    q[i] = (r[i] - qneg) * P[i];
}

__global__ void __launch_bounds__(kBlock) k_bwd_plane(PlaneArgs A, const float* __restrict__ q, float* __restrict__ z,
                                                      const float* __restrict__ P) {
#pragma clang fp contract(off)
    const SolveArgs& S = A.S;
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int x, y, zc;
    if (!plane_cell(A, t, x, y, zc)) return;
    int64_t i = rsidx(S, x, y, zc);
    uint16_t info = A.nbinfo[i];
    if (!(info & NB_FLUID)) return;
    const float ms = -S.scale_f;
    float tneg = 0.f;
#pragma unroll
    for (int a = 0; a < 3; a++)
        if (info & (NB_PX << a)) tneg += ms * z[rnb_plus(S, x, y, zc, a)];
    z[i] = (q[i] - tneg * P[i]) * P[i];
}

// ---- SpMV (applyAMatrix :165-198) with the s.q dot ---------------------------------
constexpr int SPMV_PLAIN = 0, SPMV_COPY = 1, SPMV_XPAY = 2;

// z.r beside the product, in blocks of its own, for alpha = z.r / s'.q
struct SpmvDot {
    unsigned blocks = 0;   // the grid's last ones; 0: none
    int64_t n = 0;
    const uint32_t* flags = nullptr;
    const float* r = nullptr;
};

// SPMV_PLAIN: q = A s.  SPMV_COPY: s' = z, q = A s'.  SPMV_XPAY: s' = s * beta + z
// (multSelfAndAdd :229-242), q = A s'.  The new search direction s' goes to a
// second buffer and is recomputed for the neighbours from z and the old s, so
// no block reads a value another block has already replaced.  A lane owns the
// four cells of one column of a plane group and stores them whole, zero off
// WATER (q and s are zeroed before a solve, so the columns without WATER that
// it leaves out hold zeros as well).  Bound by memory: at 256^3 65 us against
// 53 that its 18 bytes per cell take at the rate of a large copy; 74 where
// every lane gathered its neighbours (10 loads of 16 bytes and 8 of 4 per
// lane, of which 6 and 0 are left), 17 against 31 at 128^3.
template <int MODE>
__global__ void __launch_bounds__(64 * kMarchWaves) k_spmv(SolveArgs S, MarchPlan m, const uint16_t* __restrict__ nbinfo,
                                                           const float* __restrict__ z, const float* __restrict__ s,
                                                           float* __restrict__ s_new, float* __restrict__ q, Reduce red,
                                                           SpmvDot dot) {
    if (MODE != SPMV_PLAIN && blockIdx.x >= gridDim.x - dot.blocks) {
        const double zr = dot_part(Part{blockIdx.x - (gridDim.x - dot.blocks), dot.blocks}, dot.n, dot.flags, z, dot.r);
        block_finish<AUX_SUM, 64 * kMarchWaves>(0.0, zr, red);
        return;
    }
    double d = 0.0;
    const float ms = -S.scale_f;
    const float beta = MODE == SPMV_XPAY ? (float)red.sc->beta : 0.f;
    struct Raw {
        f32x4 s, z;
    };
    march(
        m, gridDim.x - dot.blocks, S.ny, S.nz, S.nxp, nbinfo,
        [&](int64_t j) {
            Raw v;
            if constexpr (MODE != SPMV_COPY) v.s = *reinterpret_cast<const f32x4*>(s + j);
            if constexpr (MODE != SPMV_PLAIN) v.z = *reinterpret_cast<const f32x4*>(z + j);
            return v;
        },
        [&](const Raw& v) {
            if constexpr (MODE == SPMV_PLAIN) return v.s;
            else if constexpr (MODE == SPMV_COPY) return v.z;
            else return v.s * beta + v.z;
        },
        [&](int64_t j, const MarchCells& n) {
            f32x4 out, snew;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                // the sums with the reference's term order, by mask
                const uint32_t f = n.info[c];
                const int cnt = (f >> NB_NONSOLID_SHIFT) & 7;
                const float si = n.own[c];
                float val = (S.scale_f * (float)cnt) * si;
                val = (f & NB_PX) ? val + ms * n.xp[c] : val;
                val = (f & NB_PY) ? val + ms * n.yp[c] : val;
                val = (f & NB_PZ) ? val + ms * n.zp[c] : val;
                val = (f & NB_MX) ? val + ms * n.xm[c] : val;
                val = (f & NB_MY) ? val + ms * n.ym[c] : val;
                val = (f & NB_MZ) ? val + ms * n.zm[c] : val;
                const bool fl = (f & NB_FLUID) != 0;
                out[c] = fl ? val : 0.f;
                snew[c] = fl ? si : 0.f;
                d += (double)snew[c] * (double)out[c];
            }
            *reinterpret_cast<f32x4*>(q + j) = out;
            if (MODE != SPMV_PLAIN) *reinterpret_cast<f32x4*>(s_new + j) = snew;
        });
    if constexpr (MODE == SPMV_PLAIN) block_finish<AUX_NONE, 64 * kMarchWaves>(d, 0.0, red);
    else block_finish<AUX_SUM, 64 * kMarchWaves>(d, 0.0, red);
}

// Large blocks: every block takes a ticket from one counter at its end, and
// the tickets are handed out one after the other.  256 blocks of 1024 threads
// against 1024 of 256: dot 21 us (27) at 256^3 and 9.7 (13.7) at 128^3, r
// update beside the x update 52 (53) and 13.6 (16.5); 128 and 512 blocks are
// slower at 256^3 (24.5 / 20.9 and 65 / 58).
constexpr int kStream = 1024;   // threads per block
constexpr unsigned kStreamBlocks = 256;
static_assert(kStreamBlocks <= kMaxParts, "stream grid within the reduction");
static unsigned stream_blocks(int64_t n) {
    const unsigned need = (unsigned)((n / kChunk + kUnits * (kStream / 64) - 1) / (kUnits * (kStream / 64)));
    return std::max(1u, std::min<unsigned>(need, kStreamBlocks));
}

template <int STEPS>
__global__ void __launch_bounds__(kBlock) k_update_x(int64_t n, const uint32_t* __restrict__ flags, UpdateX A,
                                                     const SolveScalars* __restrict__ sc) {
    update_x_chunks<STEPS>(whole_grid(), n, flags, A, sc);
}

// r_next = r - alpha q (r_next may be r); with X also the x update of the last
// two steps, behind the block's part of the reduction.
template <int NT, bool X>
__global__ void __launch_bounds__(NT) k_update_r(int64_t n, const uint32_t* __restrict__ flags, const float* q,
                                                 const float* r, float* r_next, UpdateX ux, Reduce red) {
    update_r<NT>(whole_grid(), n, flags, q, r, r_next, red);
    if constexpr (X) update_x_chunks<2>(whole_grid(), n, flags, ux, red.sc);
}

template <int NT>
__global__ void __launch_bounds__(NT) k_dot_self(int64_t n, const uint32_t* __restrict__ flags, const float* t, Reduce red) {
    dot_self<NT>(whole_grid(), n, flags, t, red);
}

// a . b (FP64 products of the FP32 values)
__global__ void __launch_bounds__(kStream) k_dot(int64_t n, const uint32_t* __restrict__ flags,
                                                const float* __restrict__ a, const float* __restrict__ b, Reduce red) {
    block_finish<AUX_NONE, kStream>(dot_part(whole_grid(), n, flags, a, b), 0.0, red);
}

// z . r and z . q: z is read once, and one launch and its tickets are saved
// (128^3: 2 x 7.5 -> 9.3 us, 256^3: 2 x 18.5 -> 27.5)
__global__ void __launch_bounds__(kStream) k_dot_zr_zq(int64_t n, const uint32_t* __restrict__ flags,
                                                      const float* __restrict__ z, const float* __restrict__ r,
                                                      const float* __restrict__ q, Reduce red) {
    double zr = 0.0, zq = 0.0;
    for_flagged_chunks<3>(
        whole_grid(), n, flags,
        [&](int64_t i, float4(&v)[3]) {
            v[0] = *reinterpret_cast<const float4*>(z + i);
            v[1] = *reinterpret_cast<const float4*>(r + i);
            v[2] = *reinterpret_cast<const float4*>(q + i);
        },
        [&](int64_t, float4(&v)[3]) {
            zr += (double)v[0].x * (double)v[1].x;
            zr += (double)v[0].y * (double)v[1].y;
            zr += (double)v[0].z * (double)v[1].z;
            zr += (double)v[0].w * (double)v[1].w;
            zq += (double)v[0].x * (double)v[2].x;
            zq += (double)v[0].y * (double)v[2].y;
            zq += (double)v[0].z * (double)v[2].z;
            zq += (double)v[0].w * (double)v[2].w;
        });
    block_finish<AUX_SUM, kStream>(zr, zq, red);
}

// FP64 true residual t = b - A x; optionally r = (float)t (0 off WATER, as r is).
// A lane owns the four cells of a column of a plane group and reads whole
// columns (ColumnNeighbours): 32 bytes of x where a gather cell by cell takes
// 8 bytes from every 32.  At most kResidualBlocks blocks, each of which takes a
// ticket of the reduction.  us a launch, 64^3 / 128^3 / 192^3 / 256^3: cell by
// cell with 2048 blocks 12.7 / 36 / 54 / 113, columns with 2048 11.8 / 35 / 44 /
// 77, 1024 12.1 / 24 / 35 / 71, 512 12 / 22 / 41 / 90.  256^3 needs 14 bytes a
// cell, 48 us at the rate of a large copy.
__global__ void __launch_bounds__(kBlock) k_true_residual(SolveArgs S, const uint16_t* __restrict__ nbinfo,
                                                          const float* __restrict__ b, const double* __restrict__ x,
                                                          float* __restrict__ r, int replace, Reduce red) {
#pragma clang fp contract(off)
    double ss = 0.0, mx = 0.0;
    const RowItems it = row_items(S.ny, S.nz, S.nxp);
    for (int k = it.first; k < it.end; k += it.step) {
        int g, y, zc;
        if (!item_column(it, k, S.ny, S.nz, g, y, zc)) continue;
        const ColumnNeighbours n = column_neighbours(S.ny, S.nz, S.nxp / WF_G, g, y, zc);
        const u16x4 info = *reinterpret_cast<const u16x4*>(nbinfo + n.own);
        if (((info[0] | info[1] | info[2] | info[3]) & NB_FLUID) == 0) continue;
        // all loads first, then the reference's terms in order, each kept by its flag
        const f64x4 own = *reinterpret_cast<const f64x4*>(x + n.own), yp = *reinterpret_cast<const f64x4*>(x + n.yp),
                    ym = *reinterpret_cast<const f64x4*>(x + n.ym), zp = *reinterpret_cast<const f64x4*>(x + n.zp),
                    zm = *reinterpret_cast<const f64x4*>(x + n.zm);
        const double xp3 = x[n.xp3], xm0 = x[n.xm0], zp3 = x[n.zp3], zm0 = x[n.zm0];
        const f32x4 bv = *reinterpret_cast<const f32x4*>(b + n.own);
        f32x4 out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint16_t f = info[c];
            if (!(f & NB_FLUID)) continue;
            const int cnt = (f >> NB_NONSOLID_SHIFT) & 7;
            double diag = 0;
            for (int j = 0; j < cnt; j++) diag += S.scale;
            double val = diag * own[c];
            val = (f & NB_PX) ? val + -S.scale * (c < 3 ? own[(c + 1) & 3] : xp3) : val;
            val = (f & NB_PY) ? val + -S.scale * yp[c] : val;
            val = (f & NB_PZ) ? val + -S.scale * (c < 3 ? zp[(c + 1) & 3] : zp3) : val;
            val = (f & NB_MX) ? val + -S.scale * (c > 0 ? own[(c + 3) & 3] : xm0) : val;
            val = (f & NB_MY) ? val + -S.scale * ym[c] : val;
            val = (f & NB_MZ) ? val + -S.scale * (c > 0 ? zm[(c + 3) & 3] : zm0) : val;
            const double t = (double)bv[c] - val;
            ss += t * t;
            mx = fmax(mx, fabs(t));
            out[c] = (float)t;
        }
        if (replace) *reinterpret_cast<f32x4*>(r + n.own) = out;
    }
    block_finish<AUX_MAX>(ss, mx, red);
}

// applyPressureToVelocities (:295-327), FP64 pressure
__global__ void __launch_bounds__(kBlock) k_apply_pressure(SolveArgs S, const uint16_t* __restrict__ nbinfo,
                                                           const uint8_t* __restrict__ label, const double* __restrict__ x,
                                                           float* __restrict__ u2, float* __restrict__ v2,
                                                           float* __restrict__ w2, double sc) {
#pragma clang fp contract(off)
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.nc) return;
    const int cz = (int)(i % S.nz), cy = (int)((i / S.nz) % S.ny), cx = (int)(i / ((int64_t)S.nz * S.ny));
    // only interior cells are WATER (their six neighbours exist); the test keeps
    // the accesses below in range whatever the mask holds
    if (cx < 1 || cy < 1 || cz < 1 || cx > S.nx - 2 || cy > S.ny - 2 || cz > S.nz - 2) return;
    const int64_t ri = rsidx(S, cx, cy, cz);
    if (!(nbinfo[ri] & NB_FLUID)) return;
    const int64_t st[3] = {(int64_t)S.ny * S.nz, S.nz, 1};
    float* f[3] = {u2, v2, w2};
    const double pi = x[ri];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        uint8_t lp = label[i + st[a]];
        if (lp == FSIM_AIR) f[a][i] = (float)((double)f[a][i] + sc * pi);
        else if (lp == FSIM_WATER) f[a][i] = (float)((double)f[a][i] + sc * (pi - x[rnb_plus(S, cx, cy, cz, a)]));
        if (label[i - st[a]] == FSIM_AIR) f[a][i - st[a]] = (float)((double)f[a][i - st[a]] - sc * pi);
    }
}

// Start of a solve: r = b, x = 0 and the other vectors 0 (n: a multiple of 4).
constexpr int kZeroed = 6;
struct SolveStart {
    int64_t n;
    const float* b;
    float* r;
    double* x;
    float* zero[kZeroed];   // null: none
};
__global__ void __launch_bounds__(kBlock) k_solve_start(SolveStart A) {
    const f32x4 none = {0.f, 0.f, 0.f, 0.f};
    const int64_t step = (int64_t)gridDim.x * kBlock * 4;
    for (int64_t i = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4; i < A.n; i += step) {
        *reinterpret_cast<f32x4*>(A.r + i) = *reinterpret_cast<const f32x4*>(A.b + i);
        *reinterpret_cast<f64x4*>(A.x + i) = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < kZeroed; k++)
            if (A.zero[k]) *reinterpret_cast<f32x4*>(A.zero[k] + i) = none;
    }
}

// ---- host driver --------------------------------------------------------------------
static SolveArgs solve_args(const fsim_ctx* ctx, double dt) {
    SolveArgs S;
    S.nx = ctx->g.nx;
    S.ny = ctx->g.ny;
    S.nz = ctx->g.nz;
    S.nc = ctx->g.nc;
    S.nxp = ctx->g.nxp;
    S.ncr = ctx->g.ncr;
    S.scale = dt / (ctx->prm.fluid_density * ctx->g.cd * ctx->g.cd);
    S.scale_f = (float)S.scale;
    return S;
}

// No boundary packet is on its way (the wavefront kernels leave the rows so): every word empty
static int clear_packets(fsim_ctx* ctx) {
    FSIM_TRY(fill_i32(ctx, reinterpret_cast<int32_t*>(ctx->ybnd), -1, 4 * ctx->wave_packets[0]));
    return fill_i32(ctx, reinterpret_cast<int32_t*>(ctx->zbnd), -1, 4 * ctx->wave_packets[1]);
}

// A wavefront kernel whose boundary poll ran out of spins sets wave_err; its
// results are then invalid and the call fails.
static int wave_failed(fsim_ctx* ctx, int err) {
    if (err) {
        FSIM_HIP(ctx, hipMemsetAsync(ctx->wave_err, 0, sizeof(int), ctx->stream));
        FSIM_TRY(clear_packets(ctx));   // what the launch sent and nobody received
        return set_err(ctx, FSIM_ERR_TIMEOUT, "wavefront sweep boundary wait timed out");
    }
    return FSIM_OK;
}

static int check_wave_err(fsim_ctx* ctx) {
    if (ctx->sweep_mode != 0) return FSIM_OK;
    int err = 0;
    FSIM_HIP(ctx, hipMemcpyAsync(&err, ctx->wave_err, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return wave_failed(ctx, err);
}

// Reduction grids: at most kMaxParts blocks (grid-stride; 8 blocks of 4 waves
// per CU keep HBM busy), a multiple of 8 for the XCD-aware row split, and
// the last block sums the partials in one pass.
static unsigned red_blocks(int64_t n) { return std::min<unsigned>((nblocks(n) + 7) / 8 * 8, kMaxParts); }
// blocks of the true residual: one per item up to kResidualBlocks (its comment)
constexpr unsigned kResidualBlocks = 1024;
static_assert(kResidualBlocks % 8 == 0 && kResidualBlocks <= kMaxParts, "true residual's grid within the reduction");
static unsigned residual_blocks(const SolveArgs& S) {
    const unsigned items = (unsigned)row_item_count(S.ny, S.nz, S.nxp);
    return std::max(8u, std::min<unsigned>((items + 7) / 8 * 8, kResidualBlocks));
}

static Reduce reduce_to(fsim_ctx* ctx, int op) { return Reduce{ctx->partials, ctx->red_count, ctx->scal, op}; }
// the same, with the finished scalars also written to the pinned host copy (wait_scalars)
static Reduce reduce_to_host(fsim_ctx* ctx, int op) {
    return Reduce{ctx->partials, ctx->red_count, ctx->scal, op, ctx->scal_host, ++ctx->scal_seq};
}

// Waits until the finishing block of the last reduce_to_host reduction has
// written its scalars: polls the pinned word, since an event after the kernel
// is one more packet that the kernels behind it wait for (5 us an iteration),
// and a copy another, with the stream's synchronisation behind it (20 to 40 us).
// After kScalarPolls, some 20 us, it gives up the processor between polls:
// with more contexts than cores the others' threads would wait for it.
// A queue that takes longer than the polls is waited for as a whole, which
// also reports a failed kernel.
constexpr int kScalarPolls = 256;
static int wait_scalars(fsim_ctx* ctx) {
    const volatile unsigned* seq = &ctx->scal_host->seq;
    const auto t0 = std::chrono::steady_clock::now();
    for (int polls = 0; *seq != ctx->scal_seq; polls++) {
        if (polls >= kScalarPolls) std::this_thread::yield();
        if (std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(100)) continue;
        FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (*seq != ctx->scal_seq) return set_err(ctx, FSIM_ERR_HIP, "the solver's scalars did not arrive");
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return FSIM_OK;
}

// colw: one byte per (y, z) column; behind it, each from a multiple of 4 bytes,
// the two words of xrange, a byte per x row, the chunk flags and the tiles' flags, cleared with it
static int64_t colw_columns(int ny, int nz) { return ((int64_t)ny * nz + 3) / 4 * 4; }
static int64_t colw_bytes(const SolveArgs& S) {
    const int64_t tiles = (int64_t)((S.ny - 2 + WF_TY - 1) / WF_TY) * ((S.nz - 2 + WF_TZ - 1) / WF_TZ);
    return colw_columns(S.ny, S.nz) + 8 + (S.nx + 3) / 4 * 4 + 4 * (S.ncr / kChunk + 1) + 2 * tiles;
}
static int* xrange_of(uint8_t* colw, int ny, int nz) { return reinterpret_cast<int*>(colw + colw_columns(ny, nz)); }

static int build_nbinfo(fsim_ctx* ctx, const SolveArgs& S, bool with_rhs) {
    FSIM_PROF(ctx, KID_RHS);
    RhsArgs A{};
    A.S = S;
    A.label = ctx->label;
    A.u2 = ctx->u2;
    A.v2 = ctx->v2;
    A.w2 = ctx->w2;
    A.density = ctx->density;
    // the search directions are free between solves
    A.info_flat = reinterpret_cast<uint16_t*>(ctx->s);
    A.b_flat = ctx->s2;
    A.colw = ctx->colw;
    A.xw = reinterpret_cast<uint8_t*>(xrange_of(ctx->colw, S.ny, S.nz) + 2);
    A.inv_dx = 1.0 / ctx->g.cd;
    A.avg_p = ctx->prm.average_pressure;
    A.pk = ctx->prm.pressure_k;
    A.pressure_enabled = ctx->prm.pressure_enabled;
    A.red = with_rhs ? reduce_to_host(ctx, FIN_BB) : reduce_to(ctx, FIN_BB);
    FSIM_TRY(fill_u8(ctx, ctx->colw, 0, colw_bytes(S)));   // and xrange and the chunk flags behind it
    hipLaunchKernelGGL(k_nbinfo_rhs, dim3(red_blocks(S.nc)), dim3(kBlock), 0, ctx->stream, A, with_rhs ? 1 : 0);
    // wide windows leave fewer lanes idle, narrow ones give small grids more and shorter blocks (this stage in us
    // with windows of 16 / 64: 32^3 22 / 25, 64^3 34.5 / 36, 96^3 53 / 53, 128^3 60 / 56, 192^3 130 / 115, 256^3
    // 267 / 235): wide ones from two blocks a compute unit on (wide windows make 376 blocks at 96^3, 756 at 128^3)
    auto items = [&](int w) {
        return (unsigned)((S.nxp + w - 1) / w * (S.ny - 2) * ((S.nz - 2 + WF_TZ - 1) / WF_TZ));
    };
    const float* b_flat = with_rhs ? A.b_flat : nullptr;
    int* xrange = xrange_of(ctx->colw, S.ny, S.nz);
    if (items(64) >= 2 * 256)
        hipLaunchKernelGGL(k_rotate<64>, dim3(items(64)), dim3(kBlock), 0, ctx->stream, S, A.info_flat, b_flat, ctx->nbinfo,
                           ctx->b, ctx->chunk_flags, A.colw, A.xw, xrange,
                           const_cast<uint8_t*>(ctx->wave.tilew));
    else
        hipLaunchKernelGGL(k_rotate<16>, dim3(items(16)), dim3(kBlock), 0, ctx->stream, S, A.info_flat, b_flat, ctx->nbinfo,
                           ctx->b, ctx->chunk_flags, A.colw, A.xw, xrange,
                           const_cast<uint8_t*>(ctx->wave.tilew));
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

static int nplane_threads(const SolveArgs& S) { return (S.nx - 2) * (S.ny - 2); }

static int mic_factor(fsim_ctx* ctx, const SolveArgs& S) {
    FSIM_PROF(ctx, KID_MIC_FACTOR);
    FSIM_TRY(fill_f64(ctx, ctx->P64, 0.0, S.ncr));
    FSIM_TRY(fill_f32(ctx, ctx->P32, 0.0f, S.ncr));
    if (ctx->sweep_mode == 0) return wave_launch(ctx, WAVE_FACTOR, nullptr, nullptr, S.scale, nullptr);
    PlaneArgs A{S, ctx->nbinfo, 0};
    const int nt = nplane_threads(S);
    const int lmax = (S.nx - 2) + (S.ny - 2) + (S.nz - 2);
    for (int L = 3; L <= lmax; L++) {
        A.level = L;
        hipLaunchKernelGGL(k_mic_factor_plane, dim3(nblocks(nt)), dim3(kBlock), 0, ctx->stream, A, ctx->P64, ctx->P32);
    }
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

// Blocks of WF_THREADS threads beside a sweep's tiles, on the compute units
// that the tiles leave free.  At 256^3, where they have 300 MB to move, a solve
// takes 66.8 ms with 128 blocks, 63.9 with 256 and 62.6 with 512.  Frames of
// 32^3 to 203x67x131 do not tell 256 from 512 (128^3 12.2 to 12.6 ms with
// either).
constexpr unsigned kSideBlocks = 512;
static_assert(kSideBlocks <= kMaxParts, "side blocks within the reduction");
static unsigned side_blocks(int64_t n) {
    const unsigned need = (unsigned)((n / kChunk + kUnits * (WF_THREADS / 64) - 1) / (kUnits * (WF_THREADS / 64)));
    return std::max(1u, std::min<unsigned>(need, kSideBlocks));
}

// t = L^-1 r and z = L^-T t, M = L L^T.
// fwd: r -= alpha q on the way (side work of the forward sweep, the new r goes
// to fwd->r_next); bwd: t . t and x (side work of the backward sweep).  Null:
// none.  alone: outside a solve.  One launch per plane does the side work in
// launches of their own, with the same blocks and so the same bits.
static int mic_apply(fsim_ctx* ctx, const SolveArgs& S, const float* r, float* t, float* z, const SideWork* fwd = nullptr,
                     const SideWork* bwd = nullptr, bool alone = false) {
    if (ctx->sweep_mode == 0) {
        {
            FSIM_PROF(ctx, KID_SWEEP_FWD);
            FSIM_TRY(wave_launch(ctx, fwd ? WAVE_FWD_UPDATE : alone ? WAVE_FWD_ALONE : WAVE_FWD, r, t, S.scale, fwd));
        }
        FSIM_PROF(ctx, KID_SWEEP_BWD);
        return wave_launch(ctx, alone ? WAVE_BWD_ALONE : WAVE_BWD, t, z, S.scale, bwd);
    }
    if (fwd) {
        hipLaunchKernelGGL((k_update_r<WF_THREADS, false>), dim3(fwd->blocks), dim3(WF_THREADS), 0, ctx->stream, fwd->n,
                           fwd->flags, fwd->q, fwd->r, fwd->r_next, UpdateX{}, fwd->red);
        r = fwd->r_next;
    }
    PlaneArgs A{S, ctx->nbinfo, 0};
    const int nt = nplane_threads(S);
    const int lmax = (S.nx - 2) + (S.ny - 2) + (S.nz - 2);
    for (int L = 3; L <= lmax; L++) {
        A.level = L;
        hipLaunchKernelGGL(k_fwd_plane, dim3(nblocks(nt)), dim3(kBlock), 0, ctx->stream, A, r, t, ctx->P32);
    }
    if (bwd) {
        hipLaunchKernelGGL(k_dot_self<WF_THREADS>, dim3(bwd->blocks), dim3(WF_THREADS), 0, ctx->stream, bwd->n, bwd->flags,
                           bwd->t, bwd->red);
        if (bwd->x_steps == 2)
            hipLaunchKernelGGL(k_update_x<2>, dim3(bwd->blocks), dim3(kBlock), 0, ctx->stream, bwd->n, bwd->flags, bwd->x,
                               ctx->scal);
    }
    for (int L = lmax; L >= 3; L--) {
        A.level = L;
        hipLaunchKernelGGL(k_bwd_plane, dim3(nblocks(nt)), dim3(kBlock), 0, ctx->stream, A, t, z, ctx->P32);
    }
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

static int true_residual(fsim_ctx* ctx, const SolveArgs& S, float* r, bool replace) {
    FSIM_PROF(ctx, KID_TRUE_RES);
    Reduce red = reduce_to_host(ctx, FIN_TRUE);
    red.wave_err = ctx->wave_err;
    hipLaunchKernelGGL(k_true_residual, dim3(residual_blocks(S)), dim3(kBlock), 0, ctx->stream, S, ctx->nbinfo, ctx->b, ctx->x,
                       r, replace ? 1 : 0, red);
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

static int dot_with(fsim_ctx* ctx, const float* a, const float* b, int op) {
    FSIM_PROF(ctx, KID_DOT);
    const int64_t n = ctx->g.ncr;
    hipLaunchKernelGGL(k_dot, dim3(stream_blocks(n)), dim3(kStream), 0, ctx->stream, n, ctx->chunk_flags, a, b,
                       reduce_to(ctx, op));
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

// Blocks beside the product's for z.r, of two trips a wave up to their limit: each takes a ticket of the reduction, and
// fewer end after the product.  us a launch of both with 1 / 2 / 4 / 8 trips: 64^3 11.6 / 10.9 / 11.1 / 14.4, 96^3 16.2 /
// 15.2 / 15.5 / 19.5, 128^3 19.1 / 19.5 / 19.4 / 21.2; with a limit of 64 / 128 / 256 / 384 / 512 blocks: 256^3 143 / 91
// / 71 / 75 / 73.  The product alone takes 10.3, 14.2, 17.9 and 63, a launch of its own for z.r 6 to 18.
static unsigned dot_blocks(int64_t n) {
    const unsigned per = 2 * kUnits * kMarchWaves;
    const unsigned need = (unsigned)((n / kChunk + per - 1) / per);
    return std::max(1u, std::min<unsigned>(need, kBesideMarch));
}

// New search direction s (z, or z + beta s) into the second buffer, q = A s,
// s.q -> alpha.
static int direction_step(fsim_ctx* ctx, const SolveArgs& S, bool copy, const float* r) {
    {
        FSIM_PROF(ctx, KID_SPMV);
        const MarchPlan m = march_of(S.ny, S.nz, S.nxp);
        SpmvDot dot;
        if (r) dot = SpmvDot{dot_blocks(S.ncr), S.ncr, ctx->chunk_flags, r};
        const dim3 grid(march_blocks(m) + dot.blocks), block(64 * kMarchWaves);
        const Reduce red = reduce_to(ctx, r ? FIN_ALPHA_ZR : FIN_ALPHA);
        if (copy)
            hipLaunchKernelGGL(k_spmv<SPMV_COPY>, grid, block, 0, ctx->stream, S, m, ctx->nbinfo, ctx->z, ctx->s, ctx->s2,
                               ctx->q, red, dot);
        else
            hipLaunchKernelGGL(k_spmv<SPMV_XPAY>, grid, block, 0, ctx->stream, S, m, ctx->nbinfo, ctx->z, ctx->s, ctx->s2,
                               ctx->q, red, dot);
    }
    FSIM_HIP(ctx, hipGetLastError());
    std::swap(ctx->s, ctx->s2);
    return FSIM_OK;
}

// x takes two direction steps at a time: it is read and written half as often
// (both s buffers still hold their step).  What is left when the loop ends is
// one step.
static UpdateX update_x_args(fsim_ctx* ctx) { return UpdateX{ctx->nbinfo, ctx->s2, ctx->s, ctx->x}; }
static int update_x_last(fsim_ctx* ctx) {
    FSIM_PROF(ctx, KID_UPDATE);
    const int64_t n = ctx->g.ncr;
    hipLaunchKernelGGL(k_update_x<1>, dim3(std::max(1u, std::min(nblocks(n / 4), kMaxParts))), dim3(kBlock), 0, ctx->stream, n,
                       ctx->chunk_flags, update_x_args(ctx), ctx->scal);
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

static bool stop_met(const fsim_ctx* ctx, double ss, double mx, double bnorm) {
    if (ctx->prm.stop_rule == FSIM_STOP_REL_L2) return std::sqrt(ss) <= ctx->prm.residual_tolerance * bnorm;
    return mx < ctx->prm.residual_tolerance;
}

// One iteration's update and preconditioner application, after the direction
// step: r -= alpha q with its norms (which the host waits for), z = M^-1 r,
// beta, and x if two steps are due.
//
// MIC(0): the r update and its norms run beside the forward sweep, which
// computes the new r for itself, and t.t and the x update beside the backward
// sweep: the sweeps are chains of waits that leave most of the chip idle.
// z'.r' = r'^T L^-T L^-1 r' = t.t with t = L^-1 r', the forward sweep's result,
// which is there before the backward sweep starts: beta = t.t / z.r, which the
// product takes rounded to FP32 (6e-8; t.t is off by the FP32 rounding inside
// the sweeps, mean error against 64 bits with random and smooth r' 24^3 3.4e-9 /
// 5.5e-9, 64^3 9e-10 / 2.1e-9, 128^3 2.6e-10 / 1.4e-9, 2D 128^2 3.9e-9 / 5.3e-9).
// alpha, which x takes in FP64, has z.r itself, of the z that is used: with
// t.t there 4 steps of the 128^3 dam break took 333 iterations instead of 330,
// 256^3 588 instead of 586.  r has two buffers, since the tiles read the old
// one.
// An iteration, against launches of their own for the r update, the dot
// product and the x update (the last on a second stream at 256^3): 32^3 62 ->
// 49 us, 2D 128^2 100 -> 86, 128^3 132 -> 115, 256^3 395 -> 386.
static int update_mic(fsim_ctx* ctx, const SolveArgs& S, float** r, float** r_next, bool x_due) {
    SideWork fwd, bwd;
    fwd.blocks = bwd.blocks = side_blocks(S.ncr);
    fwd.n = bwd.n = S.ncr;
    fwd.flags = bwd.flags = ctx->chunk_flags;
    fwd.q = ctx->q;
    fwd.r = *r;
    fwd.r_next = *r_next;
    fwd.red = reduce_to_host(ctx, FIN_RES);
    bwd.t = ctx->t;
    bwd.x = update_x_args(ctx);
    bwd.x_steps = x_due ? 2 : 0;
    bwd.red = reduce_to(ctx, FIN_BETA);
    FSIM_TRY(mic_apply(ctx, S, *r, ctx->t, ctx->z, &fwd, &bwd));
    std::swap(*r, *r_next);
    return FSIM_OK;
}
// The learned multigrid V-cycle (fsim_mg.hip), whose coarsest level the network
// solves, is not a fixed symmetric map: flexible PCG, beta = z'.(r' - r) / z.r
// = -alpha z'.q / z.r, since r' - r = -alpha q.
static int update_flexible(fsim_ctx* ctx, const SolveArgs& S, bool x_due) {
    {
        FSIM_PROF(ctx, KID_UPDATE);
        const dim3 grid(stream_blocks(S.ncr)), block(kStream);
        const Reduce red = reduce_to_host(ctx, FIN_RES);
        if (x_due)
            hipLaunchKernelGGL((k_update_r<kStream, true>), grid, block, 0, ctx->stream, S.ncr, ctx->chunk_flags, ctx->q, ctx->r,
                               ctx->r, update_x_args(ctx), red);
        else
            hipLaunchKernelGGL((k_update_r<kStream, false>), grid, block, 0, ctx->stream, S.ncr, ctx->chunk_flags, ctx->q,
                               ctx->r, ctx->r, UpdateX{}, red);
        FSIM_HIP(ctx, hipGetLastError());
    }
    FSIM_TRY(mg_apply(ctx, ctx->r, ctx->z, S.scale));
    FSIM_PROF(ctx, KID_DOT);
    hipLaunchKernelGGL(k_dot_zr_zq, dim3(stream_blocks(S.ncr)), dim3(kStream), 0, ctx->stream, S.ncr, ctx->chunk_flags, ctx->z,
                       ctx->r, ctx->q, reduce_to(ctx, FIN_FBETA));
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}
// z = M^-1 r and sigma, at the start and after a restart
static int precondition(fsim_ctx* ctx, const SolveArgs& S, const float* r, bool flexible) {
    if (flexible) {
        FSIM_TRY(mg_apply(ctx, ctx->r, ctx->z, S.scale));
        return dot_with(ctx, ctx->z, ctx->r, FIN_SIGMA0);
    }
    return mic_apply(ctx, S, r, ctx->t, ctx->z);   // sigma comes with the matrix product
}

struct PcgResult {
    int iterations = 0;
    bool converged = false;   // stopped on the FP64 true residual
    bool nan = false;         // stopped on a NaN alpha or sigma
};

// PCG from x = 0, r = b.  Reliable updates (restarted mixed-precision PCG):
// when the FP32 recursive residual meets the tolerance, or has dropped by
// kDelta (FSIM_OPT_RELIABLE_DROP) since the last FP64 true residual, the true residual b - A x is
// recomputed in FP64.  The solve stops if it meets the tolerance; otherwise r
// takes its value and the search direction restarts from z = M^-1 r.  (Keeping
// the direction instead, with beta from the replaced residual, was measured:
// 185 iterations against 145 at the 256^3 double dam break, 1e-6.)
//
// One host round trip per iteration: the r update's finishing block writes the
// scalars for the host, and the preconditioner application and beta run while
// the host waits for them.  If the solve stops or restarts, those results are
// discarded.
static int pcg_run(fsim_ctx* ctx, const SolveArgs& S, double bnorm, bool flexible, int max_it, PcgResult* res) {
    const int64_t n = S.ncr;
    fsim_step_stats& st = ctx->stats;
    float *r = ctx->r, *r_next = ctx->r_next;   // flexible: r stays where the V-cycle's graph reads it
    {
        // t and r_next as well: the sweeps leave out the tiles without WATER, and the cells there are summed
        const SolveStart A{n, ctx->b, r, ctx->x,
                           {ctx->q, ctx->z, ctx->s, ctx->s2, flexible ? nullptr : ctx->t, flexible ? nullptr : r_next}};
        hipLaunchKernelGGL(k_solve_start, dim3(std::min(nblocks(n / 4), kMaxParts)), dim3(kBlock), 0, ctx->stream, A);
        FSIM_HIP(ctx, hipGetLastError());
    }
    FSIM_TRY(precondition(ctx, S, r, flexible));
    const int max_reliable = 64;
    const double kDelta = ctx->reliable_drop > 0 ? std::pow(10.0, -ctx->reliable_drop) : 0.0;
    double last_true = bnorm;
    bool copy = true;
    int it = 0;
    int behind = 0;   // direction steps that x does not hold yet (0 or 1 between iterations)
    res->converged = false;
    res->nan = false;
    for (; it < max_it; it++) {
        FSIM_TRY(direction_step(ctx, S, copy, flexible ? nullptr : r));
        const bool two = ++behind == 2;
        if (two) behind = 0;
        if (flexible) FSIM_TRY(update_flexible(ctx, S, two));
        else FSIM_TRY(update_mic(ctx, S, &r, &r_next, two));
        FSIM_TRY(wait_scalars(ctx));
        const SolveScalars h = *ctx->scal_host;
        // the previous iteration's old-sigma test, then this iteration's alpha test
        if (h.nan_flag & 2) {
            it--;
            res->nan = true;
            break;
        }
        if (h.nan_flag & 1) {
            res->nan = true;
            break;
        }
        bool restart = false;
        if (stop_met(ctx, h.rr, h.rmax, bnorm) || std::sqrt(h.rr) < kDelta * last_true) {
            if (behind) FSIM_TRY(update_x_last(ctx));
            behind = 0;
            const bool replace = st.reliable_updates < max_reliable;
            FSIM_TRY(true_residual(ctx, S, r, replace));
            FSIM_TRY(wait_scalars(ctx));
            if (stop_met(ctx, ctx->scal_host->tr_ss, ctx->scal_host->tr_max, bnorm)) {
                res->converged = true;
                break;
            }
            if (!replace) {
                if (stop_met(ctx, h.rr, h.rmax, bnorm)) break;
            } else {
                st.reliable_updates++;
                last_true = std::sqrt(ctx->scal_host->tr_ss);
                restart = true;
            }
        }
        if (restart) FSIM_TRY(precondition(ctx, S, r, flexible));
        copy = restart;
    }
    if (behind) FSIM_TRY(update_x_last(ctx));
    res->iterations = it;
    return FSIM_OK;
}

// ---- BasicMacGrid::solveIncompressibility, basicMacGrid.cpp:5-102 -------------
// The reference's release (parallel) branch: each iteration one pass over the
// cells with x + y + z odd, then one over the even ones.  A WATER cell with s
// non-SOLID neighbours computes d = (-u - v - w + u(-x) + v(-y) + w(-z)
// [+ (avgPNum - averagePressure) pressureK]) * 1.98 / s and moves its six
// faces by +-d where the cell across is not SOLID.  Cells of one colour share
// no face, so one thread per cell of the colour needs no atomics and the
// result does not depend on the schedule.  The faces are FP64 during the
// sweeps (the reference's Face::v2 type): over many iterations of an
// over-relaxed sweep, FP32 rounding would grow far beyond the oracle's.
struct SorArgs {
    int nx, ny, nz, kz;
    const uint8_t* label;
    const float* density;
    double* f[3];
    double pk, avg_p;
    int pressure_enabled;
};

template <int ODD>
__global__ void __launch_bounds__(kBlock) k_sor_pass(SorArgs A) {
#pragma clang fp contract(off)
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t rows = (int64_t)(A.nx - 2) * (A.ny - 2);
    if (t >= rows * A.kz) return;
    const int k = (int)(t % A.kz);
    const int64_t r = t / A.kz;
    const int y = 1 + (int)(r % (A.ny - 2));
    const int x = 1 + (int)(r / (A.ny - 2));
    const int z = (ODD ? 1 + ((x + y) & 1) : 2 - ((x + y) & 1)) + 2 * k;
    if (z > A.nz - 2) return;
    const int64_t sx = (int64_t)A.ny * A.nz, sy = A.nz;
    const int64_t i = ((int64_t)x * A.ny + y) * A.nz + z;
    if (A.label[i] != FSIM_WATER) return;
    const int s1 = A.label[i + 1] != FSIM_SOLID, s2 = A.label[i - 1] != FSIM_SOLID;
    const int s3 = A.label[i + sy] != FSIM_SOLID, s4 = A.label[i - sy] != FSIM_SOLID;
    const int s5 = A.label[i + sx] != FSIM_SOLID, s6 = A.label[i - sx] != FSIM_SOLID;
    const int sum = s1 + s2 + s3 + s4 + s5 + s6;
    if (sum == 0) return;
    double* const u = A.f[0];
    double* const v = A.f[1];
    double* const w = A.f[2];
    double d = -u[i] - v[i] - w[i] + u[i - sx] + v[i - sy] + w[i - 1] +
               (A.pressure_enabled ? ((double)A.density[i] - A.avg_p) * A.pk : 0.0);
    d = d * 1.98 / sum;   // overRelaxation, basicMacGrid.cpp:13
    if (s1) w[i] += d;
    if (s2) w[i - 1] -= d;
    if (s3) v[i] += d;
    if (s4) v[i - sy] -= d;
    if (s5) u[i] += d;
    if (s6) u[i - sx] -= d;
}

__global__ void __launch_bounds__(kBlock) k_f32_to_f64(int64_t n, const float* __restrict__ a, double* __restrict__ b) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (double)a[i];
}
__global__ void __launch_bounds__(kBlock) k_f64_to_f32(int64_t n, const double* __restrict__ a, float* __restrict__ b) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

static int stage_basic_sor(fsim_ctx* ctx, const SolveArgs& S) {
    fsim_step_stats& st = ctx->stats;
    const int64_t nc = S.nc;
    if (!ctx->sor64) {
        if (hipMalloc(reinterpret_cast<void**>(&ctx->sor64), sizeof(double) * 3 * (size_t)nc) != hipSuccess) {
            ctx->sor64 = nullptr;
            return set_err(ctx, FSIM_ERR_OOM, "SOR face buffer allocation failed");
        }
    }
    FSIM_HIP(ctx, hipMemsetAsync(ctx->scal, 0, sizeof(SolveScalars), ctx->stream));
    FSIM_TRY(fill_f64(ctx, ctx->x, 0.0, S.ncr));   // no pressure field
    FSIM_TRY(build_nbinfo(ctx, S, true));
    FSIM_TRY(wait_scalars(ctx));
    const double b0 = std::sqrt(ctx->scal_host->bb);
    st.b_norm_l2 = b0;
    st.num_fluid_cells = (int64_t)ctx->scal_host->nfluid;
    SorArgs A{};
    A.nx = S.nx;
    A.ny = S.ny;
    A.nz = S.nz;
    A.kz = (S.nz - 1) / 2;   // z values of one colour in a row: at most this many
    A.label = ctx->label;
    A.density = ctx->density;
    float* f32[3] = {ctx->u2, ctx->v2, ctx->w2};
    for (int a = 0; a < 3; a++) A.f[a] = ctx->sor64 + (size_t)a * nc;
    A.pk = ctx->prm.pressure_k;
    A.avg_p = ctx->prm.average_pressure;
    A.pressure_enabled = ctx->prm.pressure_enabled;
    const int iters = ctx->prm.max_iterations;
    {
        FSIM_PROF(ctx, KID_SOR);
        for (int a = 0; a < 3; a++)
            hipLaunchKernelGGL(k_f32_to_f64, dim3(nblocks(nc)), dim3(kBlock), 0, ctx->stream, nc, f32[a], A.f[a]);
        const int64_t work = (int64_t)(S.nx - 2) * (S.ny - 2) * A.kz;
        for (int n = 0; n < iters; n++) {
            hipLaunchKernelGGL(k_sor_pass<1>, dim3(nblocks(work)), dim3(kBlock), 0, ctx->stream, A);
            hipLaunchKernelGGL(k_sor_pass<0>, dim3(nblocks(work)), dim3(kBlock), 0, ctx->stream, A);
        }
        for (int a = 0; a < 3; a++)
            hipLaunchKernelGGL(k_f64_to_f32, dim3(nblocks(nc)), dim3(kBlock), 0, ctx->stream, nc, A.f[a], f32[a]);
        FSIM_HIP(ctx, hipGetLastError());
    }
    // the right-hand side left on the projected faces (FSIM_FIELD_RHS reads it)
    FSIM_HIP(ctx, hipMemsetAsync(ctx->scal, 0, sizeof(SolveScalars), ctx->stream));
    FSIM_TRY(build_nbinfo(ctx, S, true));
    FSIM_TRY(wait_scalars(ctx));
    st.residual_rel_l2 = b0 > 0 ? std::sqrt(ctx->scal_host->bb) / b0 : 0.0;
    st.residual_abs_inf = 0.0;
    st.pcg_iterations = iters;   // BasicMacGrid returns its iteration count (basicMacGrid.cpp:10)
    return FSIM_OK;
}

int stage_solve(fsim_ctx* ctx, double dt) {
    const SolveArgs S = solve_args(ctx, dt);
    const int64_t nc = S.nc;
    const unsigned nb = nblocks(nc);
    ctx->last_dt = dt;
    fsim_step_stats& st = ctx->stats;
    st.early_exit = 0;
    st.fallback = 0;
    st.reliable_updates = 0;
    st.pcg_iterations = 0;
    st.learned_iterations = 0;
    st.learned_stop = 0;
    st.solve_nan = 0;
    st.learned_budget = 0;
    if (ctx->prm.precond == FSIM_SOLVER_BASIC_SOR) return stage_basic_sor(ctx, S);
    const bool learned = ctx->prm.precond == FSIM_PRECOND_LEARNED;
    if (learned && ctx->mg_coarse == FSIM_MG_COARSE_NETWORK && !learned_ready(ctx))
        return set_err(ctx, FSIM_ERR_INVALID, "learned preconditioner selected but it has no parameters "
                                              "(fsim_learned_init or fsim_learned_set_params)");
    FSIM_HIP(ctx, hipMemsetAsync(ctx->scal, 0, sizeof(SolveScalars), ctx->stream));
    FSIM_TRY(build_nbinfo(ctx, S, true));
    FSIM_TRY(wait_scalars(ctx));
    const double bb = ctx->scal_host->bb;
    const double bnorm = std::sqrt(bb);
    st.b_norm_l2 = bnorm;
    st.num_fluid_cells = (int64_t)ctx->scal_host->nfluid;
    if (bb < 1e-7) {   // early exit without pressure (bridsonSolverGrid.cpp:254-258)
        st.early_exit = 1;
        FSIM_TRY(fill_f64(ctx, ctx->x, 0.0, S.ncr));
        FSIM_TRY(true_residual(ctx, S, ctx->r, false));
        FSIM_TRY(wait_scalars(ctx));
        st.residual_abs_inf = ctx->scal_host->tr_max;
        st.residual_rel_l2 = 1.0;
        return FSIM_OK;
    }
    const int max_it = ctx->prm.max_iterations;
    PcgResult res;
    bool use_mic = !learned;
    if (learned && !ctx->mg_harvesting &&
        (ctx->last_mic_iterations <= 0 || (ctx->learned_refresh > 0 && ctx->learned_since_mic >= ctx->learned_refresh))) {
        // no MIC(0) count to budget against yet (or it is old): this solve is
        // MIC(0)-PCG, which measures it
        use_mic = true;
        st.learned_stop = 3;
    } else if (learned) {
        // flexible PCG with the network; MIC(0)-PCG from scratch when it does not
        // reach the tolerance within twice the last MIC(0) iteration count
        const int budget = ctx->mg_harvesting ? max_it : std::min(max_it, 2 * ctx->last_mic_iterations);
        st.learned_budget = budget;
        if (!ctx->mg_harvesting) ctx->learned_since_mic++;
        FSIM_TRY(mg_setup(ctx));
        FSIM_TRY(pcg_run(ctx, S, bnorm, true, budget, &res));
        st.learned_iterations = res.iterations;
        st.learned_stop = res.converged ? 0 : res.nan ? 2 : 1;
        if (!res.converged) {
            st.fallback = 1;
            use_mic = true;
            FSIM_HIP(ctx, hipMemsetAsync(ctx->scal, 0, sizeof(SolveScalars), ctx->stream));
        }
    }
    if (use_mic) {
        FSIM_TRY(mic_factor(ctx, S));
        FSIM_TRY(pcg_run(ctx, S, bnorm, false, max_it, &res));
        if (res.converged) {
            ctx->last_mic_iterations = res.iterations;
            ctx->learned_since_mic = 0;
        }
    }
    st.pcg_iterations = res.iterations;
    const double sc = dt / (ctx->prm.fluid_density * ctx->g.cd);
    {
        FSIM_PROF(ctx, KID_PRESSURE);
        hipLaunchKernelGGL(k_apply_pressure, dim3(nb), dim3(kBlock), 0, ctx->stream, S, ctx->nbinfo, ctx->label, ctx->x,
                           ctx->u2, ctx->v2, ctx->w2, sc);
    }
    FSIM_HIP(ctx, hipGetLastError());
    FSIM_TRY(true_residual(ctx, S, ctx->r, false));
    FSIM_TRY(wait_scalars(ctx));
    st.residual_abs_inf = ctx->scal_host->tr_max;
    st.residual_rel_l2 = bnorm > 0 ? std::sqrt(ctx->scal_host->tr_ss) / bnorm : 0.0;
    // a NaN alpha or sigma ended the solve: like the reference, the last
    // finite pressure has been applied and the step goes on
    st.solve_nan = res.nan ? 1 : 0;
    return ctx->sweep_mode == 0 ? wave_failed(ctx, (int)ctx->scal_host->wave_err) : FSIM_OK;
}

int wave_init(fsim_ctx* ctx) {
    WaveArgs& A = ctx->wave;
    A.nx = ctx->g.nx;
    A.ny = ctx->g.ny;
    A.nz = ctx->g.nz;
    A.nxp = ctx->g.nxp;
    A.TJ = (A.ny - 2 + WF_TY - 1) / WF_TY;
    A.TK = (A.nz - 2 + WF_TZ - 1) / WF_TZ;
    // packet rows: one per plane group that a tile's march can reach (planes x + rot(z)); two words per
    // value (the factor's FP64), the sweeps use one
    A.SG = (A.nx - 2 + WF_TZ - 1) / WF_G + 1;
    ctx->wave_packets[0] = 2 * (int64_t)A.TJ * A.TK * A.SG * WF_TZ;
    ctx->wave_packets[1] = 2 * (int64_t)A.TJ * A.TK * A.SG * WF_TY;
    if (ctx->g.nc > kWaveMaxCells) ctx->sweep_mode = 1;
    if (hipMalloc(&ctx->ybnd, sizeof(uint4) * ctx->wave_packets[0]) != hipSuccess ||
        hipMalloc(&ctx->zbnd, sizeof(uint4) * ctx->wave_packets[1]) != hipSuccess ||
        hipMalloc(&ctx->wave_ticket, sizeof(unsigned long long) * 3) != hipSuccess ||
        hipMalloc(&ctx->wave_err, sizeof(int)) != hipSuccess ||
        hipMalloc(&ctx->colw, (size_t)colw_bytes(solve_args(ctx, 1.0))) != hipSuccess)
        return set_err(ctx, FSIM_ERR_OOM, "wavefront buffer allocation failed");
    FSIM_TRY(fill_u8(ctx, ctx->colw, 0, colw_bytes(solve_args(ctx, 1.0))));
    ctx->chunk_flags = reinterpret_cast<uint32_t*>(xrange_of(ctx->colw, A.ny, A.nz) + 2 + (A.nx + 3) / 4);
    FSIM_TRY(clear_packets(ctx));
    FSIM_HIP(ctx, hipMemsetAsync(ctx->wave_ticket, 0, sizeof(unsigned long long) * 3, ctx->stream));
    FSIM_HIP(ctx, hipMemsetAsync(ctx->wave_err, 0, sizeof(int), ctx->stream));
    A.nbinfo = ctx->nbinfo;
    A.P64 = ctx->P64;
    A.P32 = ctx->P32;
    A.ybnd = ctx->ybnd;
    A.zbnd = ctx->zbnd;
    A.err = ctx->wave_err;
    A.tilew = reinterpret_cast<const uint8_t*>(ctx->chunk_flags + ctx->g.ncr / kChunk + 1);
    A.xrange = xrange_of(ctx->colw, A.ny, A.nz);
    return FSIM_OK;
}

int solver_apply(fsim_ctx* ctx, int op, double dt, const double* in, double* out) {
    const SolveArgs S = solve_args(ctx, dt);
    const int64_t n = S.ncr;
    FSIM_TRY(build_nbinfo(ctx, S, false));
    // host vectors are in flat order, device solver vectors in the rotated one
    auto each = [&](auto&& f) { for_rotated(S.nx, S.ny, S.nz, S.nxp, f); };
    // a host buffer without a first pass over its pages
    auto result = [&](auto* src) {
        using T = std::remove_cv_t<std::remove_pointer_t<decltype(src)>>;
        const std::unique_ptr<T[]> h(new (std::nothrow) T[(size_t)n]);
        if (!h) return set_err(ctx, FSIM_ERR_OOM, "host buffer allocation failed");
        FSIM_TRY(read_back(ctx, h.get(), src, sizeof(T) * (size_t)n));
        each([&](int64_t i, int64_t r) { out[i] = h[r]; });
        return (int)FSIM_OK;
    };
    if (op == FSIM_OP_FACTOR_MIC0) {
        FSIM_TRY(mic_factor(ctx, S));
        FSIM_TRY(check_wave_err(ctx));
        return result(ctx->P64);
    }
    std::vector<float> hin(n);   // padding values 0
    each([&](int64_t i, int64_t r) { hin[r] = (float)in[i]; });
    FSIM_HIP(ctx, hipMemcpyAsync(ctx->r, hin.data(), sizeof(float) * n, hipMemcpyHostToDevice, ctx->stream));
    if (op == FSIM_OP_APPLY_A) {
        FSIM_TRY(fill_f32(ctx, ctx->q, 0.0f, n));   // the SpMV skips columns without WATER
        const MarchPlan m = march_of(S.ny, S.nz, S.nxp);
        hipLaunchKernelGGL(k_spmv<SPMV_PLAIN>, dim3(march_blocks(m)), dim3(64 * kMarchWaves), 0, ctx->stream, S, m,
                           ctx->nbinfo, nullptr, ctx->r, nullptr, ctx->q, reduce_to(ctx, FIN_NONE), SpmvDot{});
        FSIM_HIP(ctx, hipGetLastError());
        return result(ctx->q);
    }
    if (op == FSIM_OP_APPLY_MIC0) {
        FSIM_TRY(mic_factor(ctx, S));
        FSIM_TRY(fill_f32(ctx, ctx->t, 0.0f, n));
        FSIM_TRY(fill_f32(ctx, ctx->z, 0.0f, n));
        FSIM_TRY(mic_apply(ctx, S, ctx->r, ctx->t, ctx->z, nullptr, nullptr, true));
        FSIM_TRY(check_wave_err(ctx));
        return result(ctx->z);
    }
    if (op == FSIM_OP_APPLY_MG) {
        if (ctx->mg_coarse == FSIM_MG_COARSE_NETWORK && !learned_ready(ctx))
            return set_err(ctx, FSIM_ERR_INVALID, "the multigrid's coarse network has no parameters");
        FSIM_TRY(mg_setup(ctx));
        FSIM_TRY(fill_f32(ctx, ctx->z, 0.0f, n));
        FSIM_TRY(mg_apply(ctx, ctx->r, ctx->z, S.scale));
        return result(ctx->z);
    }
    return set_err(ctx, FSIM_ERR_INVALID, "unknown solver op");
}

}  // namespace fsim
