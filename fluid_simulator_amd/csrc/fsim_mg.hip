// fsim_mg.hip — the learned multigrid preconditioner of flexible PCG (no
// counterpart in the reference; MIC(0)-PCG stays the fallback and the
// solve its results are measured against).
//
// z = M(r) is one V-cycle on a hierarchy of aggregation levels whose
// coarsest level is solved by the learned network:
//   * level 0 is the solve's own operator A = s L0 (s = dt / (rho dx^2),
//     L0 the 7-point matrix of calculateAMatrix, bridsonSolverGrid.cpp:40-77:
//     diagonal = non-SOLID neighbours, -1 towards WATER neighbours), read
//     from nbinfo in the solver's rotated layout;
//   * level l+1 aggregates 2x2x2 cells of level l: P is piecewise constant,
//     R = P^T, and L_{l+1} = P^T L_l P (Galerkin).  Aggregates of a 7-point
//     operator couple only face neighbours, so each level stores four FP32
//     arrays: diagonal and the couplings to the +x, +y, +z neighbour;
//   * smoothing: red-black Gauss-Seidel over the parity of x + y + z (one
//     colour has no coupling inside itself, so a half-sweep is a parallel
//     pass with no races), two sweeps before and two after the coarse
//     correction, which is added with the over-correction factor 1.6 that
//     piecewise-constant aggregation needs;
//   * the coarsest level (the first whose largest side is <= 16 cells) is
//     solved by the network from (b / max|b|, the level's operator
//     normalised by 4^-level), followed by a few red-black sweeps; for
//     comparisons it can instead be left out (smoothing only) or solved
//     accurately (600 sweeps), which also harvests training samples.
// The V-cycle is not a symmetric linear map (the network is not linear, and
// pre- and post-smoothing visit the colours in the same order), hence
// flexible PCG.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>
#include <vector>

#include "fsim_internal.hpp"

namespace fsim {

constexpr float kMgOverCorrect = 1.6f;
constexpr int kMgPreSweeps = 2, kMgPostSweeps = 2;
constexpr int kMgExactSweeps = 600;

// ---- layout helpers -------------------------------------------------------------
struct MgGrid {
    int nx, ny, nz;
    const float *diag, *ox, *oy, *oz;
    float *b, *x;
};
__device__ inline int64_t lin(int nx, int ny, int nz, int x, int y, int z) { return ((int64_t)x * ny + y) * nz + z; }
__device__ inline void unlin(int64_t i, int ny, int nz, int& x, int& y, int& z) {
    z = (int)(i % nz);
    y = (int)((i / nz) % ny);
    x = (int)(i / ((int64_t)nz * ny));
}

struct Mg0 {               // level 0: the solve's operator in the rotated layout
    int nx, ny, nz, nxp;
    const uint16_t* nbinfo;
    const float* b;        // r of the PCG iteration
    float* x;              // z
    float binv;            // 1 / s: level 0 solves L0 x = r / s
};
__device__ inline int nb_nonsolid(uint16_t nb) { return (nb >> NB_NONSOLID_SHIFT) & 7; }

// ---- coarsening ---------------------------------------------------------------------
// Level 1 from level 0: an aggregate's diagonal sums its fluid children's
// non-SOLID counts less twice each WATER-WATER coupling inside it; its +a
// coupling counts the couplings of its upper children to the next aggregate.
__global__ void __launch_bounds__(kBlock) k_mg_coarsen0(Mg0 F, int cx, int cy, int cz, float* __restrict__ diag,
                                                         float* __restrict__ ox, float* __restrict__ oy,
                                                         float* __restrict__ oz) {
    const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= (int64_t)cx * cy * cz) return;
    int X, Y, Z;
    unlin(I, cy, cz, X, Y, Z);
    float d = 0.f, c[3] = {0.f, 0.f, 0.f};
    for (int k = 0; k < 8; k++) {
        const int a = k >> 2, b = (k >> 1) & 1, e = k & 1;
        const int x = 2 * X + a, y = 2 * Y + b, z = 2 * Z + e;
        if (x >= F.nx || y >= F.ny || z >= F.nz) continue;
        const uint16_t nb = F.nbinfo[ridx(x, y, z, F.nxp, F.ny, F.nz)];
        if (!(nb & NB_FLUID)) continue;
        d += (float)nb_nonsolid(nb);
        const bool up[3] = {(nb & NB_PX) != 0, (nb & NB_PY) != 0, (nb & NB_PZ) != 0};
        const int loc[3] = {a, b, e};
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            if (!up[ax]) continue;
            if (loc[ax] == 0) d -= 2.f;   // the +ax neighbour is a sibling
            else c[ax] += 1.f;            // it belongs to the next aggregate
        }
    }
    diag[I] = d;
    ox[I] = c[0];
    oy[I] = c[1];
    oz[I] = c[2];
}

// Level l+1 from level l (coefficient arrays)
__global__ void __launch_bounds__(kBlock) k_mg_coarsen(MgGrid F, int cx, int cy, int cz, float* __restrict__ diag,
                                                        float* __restrict__ ox, float* __restrict__ oy,
                                                        float* __restrict__ oz) {
    const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= (int64_t)cx * cy * cz) return;
    int X, Y, Z;
    unlin(I, cy, cz, X, Y, Z);
    float d = 0.f, c[3] = {0.f, 0.f, 0.f};
    for (int k = 0; k < 8; k++) {
        const int a = k >> 2, b = (k >> 1) & 1, e = k & 1;
        const int x = 2 * X + a, y = 2 * Y + b, z = 2 * Z + e;
        if (x >= F.nx || y >= F.ny || z >= F.nz) continue;
        const int64_t i = lin(F.nx, F.ny, F.nz, x, y, z);
        const float di = F.diag[i];
        if (di == 0.f) continue;
        d += di;
        const float o[3] = {F.ox[i], F.oy[i], F.oz[i]};
        const int loc[3] = {a, b, e};
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            if (loc[ax] == 0) d -= 2.f * o[ax];
            else c[ax] += o[ax];
        }
    }
    diag[I] = d;
    ox[I] = c[0];
    oy[I] = c[1];
    oz[I] = c[2];
}

// ---- smoothing: one red-black half-sweep --------------------------------------------
// Launch shape of the coarse levels' per-cell kernels: a block is kMgBy rows
// (y) x kMgBz columns (z) of one plane x, the grid (z chunks, y chunks,
// planes), so no thread divides its index.
constexpr int kMgBz = 64, kMgBy = 4;
struct MgLaunch {
    dim3 grid, block;
};
static MgLaunch mg_launch(int nx, int ny, int nz) {
    int bz = kMgBz;
    while (bz > 16 && bz / 2 >= nz) bz /= 2;   // small coarse levels: narrower z, more rows per block
    const int by = kMgBz * kMgBy / bz;
    return MgLaunch{dim3((unsigned)((nz + bz - 1) / bz), (unsigned)((ny + by - 1) / by), (unsigned)nx),
                    dim3((unsigned)bz, (unsigned)by)};
}

// Level 0: a lane owns the four cells of a column of a plane group
// (ColumnNeighbours).  x + z = p + 1 (mod 2) on plane p, since (z - 1) mod 64
// has the parity of z - 1 and the wrap adds nxp, a multiple of 4: the cells of
// one colour in row y are the elements c with (c + 1 + y) mod 2 equal to it,
// two of a lane's four.  A wave has one row, so the choice is uniform.
struct Column4 {
    f32x4 own, yp, ym, zp, zm;
    float xe, ze;   // the neighbours of the colour's outer element from the next or previous group
};
// odd: elements 1 and 3 (whose outer neighbours are ahead), else 0 and 2 (behind)
__device__ inline Column4 load_column(const float* x, const ColumnNeighbours& n, bool odd) {
    Column4 v;
    v.own = *reinterpret_cast<const f32x4*>(x + n.own);
    v.yp = *reinterpret_cast<const f32x4*>(x + n.yp);
    v.ym = *reinterpret_cast<const f32x4*>(x + n.ym);
    v.zp = *reinterpret_cast<const f32x4*>(x + n.zp);
    v.zm = *reinterpret_cast<const f32x4*>(x + n.zm);
    v.xe = x[odd ? n.xp3 : n.xm0];
    v.ze = x[odd ? n.zp3 : n.zm0];
    return v;
}
// the neighbours of element c in the order -x, +x, -y, +y, -z, +z
template <int C>
__device__ inline void column_terms(const Column4& v, float (&t)[6]) {
    t[0] = C > 0 ? v.own[(C + 3) & 3] : v.xe;
    t[1] = C < 3 ? v.own[(C + 1) & 3] : v.xe;
    t[2] = v.ym[C];
    t[3] = v.yp[C];
    t[4] = C > 0 ? v.zm[(C + 3) & 3] : v.ze;
    t[5] = C < 3 ? v.zp[(C + 1) & 3] : v.ze;
}
constexpr uint16_t kMgNb[6] = {NB_MX, NB_PX, NB_MY, NB_PY, NB_MZ, NB_PZ};

// FIRST: the first half-sweep from x = 0 (no neighbour terms; the other colour
// is set to 0).
template <int PAR, bool FIRST>
__global__ void __launch_bounds__(kBlock) k_mg_rbgs0(Mg0 A) {
    const RowItems it = row_items(A.ny, A.nz, A.nxp);
    for (int k = it.first; k < it.end; k += it.step) {
        int g, y, z;
        if (!item_column(it, k, A.ny, A.nz, g, y, z)) continue;
        const ColumnNeighbours n = column_neighbours(A.ny, A.nz, A.nxp / WF_G, g, y, z);
        const u16x4 nb = *reinterpret_cast<const u16x4*>(A.nbinfo + n.own);
        if (((nb[0] | nb[1] | nb[2] | nb[3]) & NB_FLUID) == 0) continue;
        const f32x4 b = *reinterpret_cast<const f32x4*>(A.b + n.own);
        const bool odd = ((PAR + 1 + y) & 1) != 0;
        if constexpr (FIRST) {
            f32x4 out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; c++)
                if ((c & 1) == (int)odd && (nb[c] & NB_FLUID)) out[c] = b[c] * A.binv / (float)nb_nonsolid(nb[c]);
            *reinterpret_cast<f32x4*>(A.x + n.own) = out;
        } else {
            const Column4 v = load_column(A.x, n, odd);
            f32x4 out = v.own;
            auto cell = [&](auto cc) {
                constexpr int c = decltype(cc)::value;
                if (!(nb[c] & NB_FLUID)) return;
                float t[6];
                column_terms<c>(v, t);
                float s = b[c] * A.binv;
#pragma unroll
                for (int j = 0; j < 6; j++) s = (nb[c] & kMgNb[j]) ? s + t[j] : s;
                out[c] = s / (float)nb_nonsolid(nb[c]);
            };
            if (odd) {
                cell(std::integral_constant<int, 1>{});
                cell(std::integral_constant<int, 3>{});
            } else {
                cell(std::integral_constant<int, 0>{});
                cell(std::integral_constant<int, 2>{});
            }
            *reinterpret_cast<f32x4*>(A.x + n.own) = out;
        }
    }
}

// The couplings and neighbour values of cell i in the order +x, -x, +y, -y, +z,
// -z, all 12 loads issued together (a branch per coupling would wait for each
// load in turn: a half-sweep 3.7 us at 64^3 and 7.8 at 128^3, so 3.1 and 5.0).
// A coupling beyond the level's edge is 0, its x the cell's own.
struct LevelTerms {
    float o[6], x[6];
};
__device__ inline LevelTerms level_terms(const MgGrid& G, int x, int y, int z, int64_t i) {
    const int64_t sx = (int64_t)G.ny * G.nz, sy = G.nz;
    const int64_t mx = x > 0 ? i - sx : i, my = y > 0 ? i - sy : i, mz = z > 0 ? i - 1 : i;
    LevelTerms t;
    t.o[0] = G.ox[i];
    t.o[1] = G.ox[mx];
    t.o[2] = G.oy[i];
    t.o[3] = G.oy[my];
    t.o[4] = G.oz[i];
    t.o[5] = G.oz[mz];
    t.x[0] = G.x[x + 1 < G.nx ? i + sx : i];
    t.x[1] = G.x[mx];
    t.x[2] = G.x[y + 1 < G.ny ? i + sy : i];
    t.x[3] = G.x[my];
    t.x[4] = G.x[z + 1 < G.nz ? i + 1 : i];
    t.x[5] = G.x[mz];
    if (x == 0) t.o[1] = 0.f;
    if (y == 0) t.o[3] = 0.f;
    if (z == 0) t.o[5] = 0.f;
    return t;
}

template <int PAR, bool FIRST>
__global__ void __launch_bounds__(kMgBz * kMgBy) k_mg_rbgs(MgGrid G) {
    const int z = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int x = blockIdx.z;
    if (z >= G.nz || y >= G.ny) return;
    const bool mine = ((x + y + z) & 1) == PAR;
    if (!FIRST && !mine) return;
    const int64_t i = lin(G.nx, G.ny, G.nz, x, y, z);
    const float d = G.diag[i];
    if (d == 0.f) return;
    if (!mine) {
        G.x[i] = 0.f;   // FIRST only
        return;
    }
    float s = G.b[i];
    if (!FIRST) {
        const LevelTerms t = level_terms(G, x, y, z, i);
#pragma unroll
        for (int j = 0; j < 6; j++) s = t.o[j] != 0.f ? s + t.o[j] * t.x[j] : s;
    }
    G.x[i] = s / d;
}

// ---- residual + restriction -----------------------------------------------------------
// b_{l+1}[I] = sum over the fluid children i of (b_i - (L x)_i).
// Level 0: the children of a coarse cell lie in different rotated planes (x +
// ((z - 1) mod 64) differs between them), so a thread per coarse cell
// gathering them would read every value from another plane.  Instead a block
// computes the residual of a 64 (x) x 2 (y) x 64 (z) fine box by columns of
// plane groups, each wave contiguous memory, puts it into LDS, and sums every
// coarse cell's 8 children there in a fixed order.
// The residual follows the last pre-smoothing half-sweep, which solved the
// cells of colour 0 exactly: their residual is the rounding of that division,
// which evaluating it in FP32 would not resolve.  It is taken as 0, for every
// width of the grid, and only the cells of colour 1 are computed.
constexpr int kRtC = 32;   // coarse cells per block along x and along z (a 64 x 2 x 64 fine box)
__global__ void __launch_bounds__(256) k_mg_resid_restrict0(Mg0 A, MgGrid C) {
    // fine box [yy][x - fx0][z - fz0]; a row of 64 words: the lanes of a wave store into a different
    // bank each
    __shared__ float F[2][2 * kRtC][2 * kRtC];
    const int X0 = blockIdx.x * kRtC, Y = blockIdx.y, Z0 = blockIdx.z * kRtC;
    const int fx0 = 2 * X0, fz0 = 2 * Z0;
    for (int k = threadIdx.x; k < 2 * 2 * kRtC * 2 * kRtC; k += blockDim.x) (&F[0][0][0])[k] = 0.f;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwaves = blockDim.x >> 6;
    const int z = fz0 + lane;
    const int rz = rot_of(z);
    const int ng = A.nxp / WF_G;
    // the cells x in [fx0, fx0 + 64) of column z are on the planes fx0 + rz .. fx0 + rz + 63
    constexpr int kGroups = (2 * kRtC + 63) / WF_G + 1;
    for (int k = wave; k < 2 * kGroups; k += nwaves) {
        const int yy = k / kGroups, gu = fx0 / WF_G + k % kGroups;   // unwrapped group
        const int y = 2 * Y + yy;
        const int x0 = WF_G * gu - rz;                               // x of element 0
        if (y < 1 || y > A.ny - 2 || z < 1 || z > A.nz - 2 || x0 + 3 < fx0 || x0 >= fx0 + 2 * kRtC) continue;
        const ColumnNeighbours n = column_neighbours(A.ny, A.nz, ng, gu % ng, y, z);
        const u16x4 nb = *reinterpret_cast<const u16x4*>(A.nbinfo + n.own);
        if (((nb[0] | nb[1] | nb[2] | nb[3]) & NB_FLUID) == 0) continue;
        const bool odd = (y & 1) != 0;   // colour 1: (c + 1 + y) odd
        const Column4 v = load_column(A.x, n, odd);
        const f32x4 b = *reinterpret_cast<const f32x4*>(A.b + n.own);
        auto cell = [&](auto cc) {
            constexpr int c = decltype(cc)::value;
            const int x = x0 + c;
            if (!(nb[c] & NB_FLUID) || x < fx0 || x >= fx0 + 2 * kRtC || x >= A.nx) return;
            float t[6];
            column_terms<c>(v, t);
            float ax = (float)nb_nonsolid(nb[c]) * v.own[c];
#pragma unroll
            for (int j = 0; j < 6; j++) ax = (nb[c] & kMgNb[j]) ? ax - t[j] : ax;
            F[yy][x - fx0][lane] = b[c] * A.binv - ax;
        };
        if (odd) {
            cell(std::integral_constant<int, 1>{});
            cell(std::integral_constant<int, 3>{});
        } else {
            cell(std::integral_constant<int, 0>{});
            cell(std::integral_constant<int, 2>{});
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kRtC * kRtC; k += blockDim.x) {
        const int xl = k / kRtC, zl = k % kRtC;
        const int X = X0 + xl, Z = Z0 + zl;
        if (X >= C.nx || Z >= C.nz) continue;
        const int64_t I = lin(C.nx, C.ny, C.nz, X, Y, Z);
        float sum = 0.f;
        if (C.diag[I] != 0.f) {
#pragma unroll
            for (int c = 0; c < 8; c++) sum += F[(c >> 1) & 1][2 * xl + (c >> 2)][2 * zl + (c & 1)];
        }
        C.b[I] = sum;
    }
}

// Levels >= 1: a thread per child, the eight of a coarse cell in consecutive
// lanes, whose residuals the first sums in order.  A thread that took all
// eight waited for 56 pairs of loads one after the other: 17.6 us from 64^3, so
// 4.9; 21 us a level at 256^3, so 13.
__global__ void __launch_bounds__(kBlock) k_mg_restrict(MgGrid F, MgGrid C) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = (int64_t)C.nx * C.ny * C.nz;
    const int64_t I = min(t >> 3, n - 1);   // every lane takes part in the exchange
    const int k = (int)(t & 7);
    int X, Y, Z;
    unlin(I, C.ny, C.nz, X, Y, Z);
    const int x = 2 * X + (k >> 2), y = 2 * Y + ((k >> 1) & 1), z = 2 * Z + (k & 1);
    bool on = x < F.nx && y < F.ny && z < F.nz;
    float res = 0.f;
    if (on) {
        const int64_t i = lin(F.nx, F.ny, F.nz, x, y, z);
        const float d = F.diag[i], own = F.x[i], b = F.b[i];
        const LevelTerms v = level_terms(F, x, y, z, i);
        on = d != 0.f;
        float ax = d * own;
#pragma unroll
        for (int j = 0; j < 6; j++) ax = v.o[j] != 0.f ? ax - v.o[j] * v.x[j] : ax;
        res = b - ax;
    }
    float sum = 0.f;
    const uint64_t take = __ballot(on);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int from = (lane & ~7) + c;
        const float r = __shfl(res, from, 64);
        if ((take >> from) & 1) sum += r;
    }
    if (k == 0 && (t >> 3) < n) C.b[I] = C.diag[I] == 0.f ? 0.f : sum;
}

// ---- prolongation: x_i += 1.6 x_{l+1}[parent(i)] on the level's unknowns ----------------
__global__ void __launch_bounds__(kBlock) k_mg_prolong0(Mg0 A, MgGrid C) {
    const RowItems it = row_items(A.ny, A.nz, A.nxp);
    for (int k = it.first; k < it.end; k += it.step) {
        int g, y, z;
        if (!item_column(it, k, A.ny, A.nz, g, y, z)) continue;
        const int64_t i = pidx(g * WF_G, y, z, A.ny, A.nz);
        const u16x4 nb = *reinterpret_cast<const u16x4*>(A.nbinfo + i);
        if (((nb[0] | nb[1] | nb[2] | nb[3]) & NB_FLUID) == 0) continue;
        f32x4 x = *reinterpret_cast<const f32x4*>(A.x + i);
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (nb[c] & NB_FLUID)
                x[c] += kMgOverCorrect *
                        C.x[lin(C.nx, C.ny, C.nz, unrot_x(g * WF_G + c, z, A.nxp) >> 1, y >> 1, z >> 1)];
        *reinterpret_cast<f32x4*>(A.x + i) = x;
    }
}

__global__ void __launch_bounds__(kMgBz * kMgBy) k_mg_prolong(MgGrid F, MgGrid C) {
    const int z = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int x = blockIdx.z;
    if (z >= F.nz || y >= F.ny) return;
    const int64_t i = lin(F.nx, F.ny, F.nz, x, y, z);
    if (F.diag[i] == 0.f) return;
    F.x[i] += kMgOverCorrect * C.x[lin(C.nx, C.ny, C.nz, x >> 1, y >> 1, z >> 1)];
}

// ---- host side ------------------------------------------------------------------------------
struct MgLevelBuf {
    int nx = 0, ny = 0, nz = 0;
    int64_t nc = 0;
    float *diag = nullptr, *ox = nullptr, *oy = nullptr, *oz = nullptr, *b = nullptr, *x = nullptr;
};
struct MgState {
    int nlev = 0;   // levels 0 .. nlev-1; nlev-1 is the coarse (network) level
    MgLevelBuf lv[kMgMaxLevels];
    std::vector<void*> allocs;
    // harvest: up to cap coarse (b, x) pairs of the running solve
    int harvest_cap = 0, harvest_n = 0;
    float *hb = nullptr, *hx = nullptr;
    // the V-cycle captured as a HIP graph, with what its kernel arguments were made from
    hipGraphExec_t exec = nullptr;
    struct Key {
        const float* r;
        float* z;
        double scale;
        int mode, nu, conv, net_gen;
        bool operator==(const Key& o) const {
            return r == o.r && z == o.z && scale == o.scale && mode == o.mode && nu == o.nu && conv == o.conv &&
                   net_gen == o.net_gen;
        }
    } key{};
};

static MgGrid grid_of(const MgLevelBuf& L) { return MgGrid{L.nx, L.ny, L.nz, L.diag, L.ox, L.oy, L.oz, L.b, L.x}; }

static void drop_graph(MgState* M) {
    if (M->exec) (void)hipGraphExecDestroy(M->exec);
    M->exec = nullptr;
}

void mg_free(fsim_ctx* ctx) {
    MgState* M = ctx->mg;
    if (!M) return;
    drop_graph(M);
    for (void* p : M->allocs) (void)hipFree(p);
    delete M;
    ctx->mg = nullptr;
}

int mg_levels_for(int nx, int ny, int nz) {
    int l = 0;
    while (std::max({nx, ny, nz}) > kMgCoarseMaxSide && l < kMgMaxLevels - 1) {
        nx = (nx + 1) / 2;
        ny = (ny + 1) / 2;
        nz = (nz + 1) / 2;
        l++;
    }
    return l + 1;
}

static int mg_alloc(fsim_ctx* ctx) {
    if (ctx->mg) return FSIM_OK;
    if (ctx->g.two_d) return set_err(ctx, FSIM_ERR_INVALID, "the multigrid preconditioner is built for 3D grids only");
    MgState* M = new MgState();
    ctx->mg = M;
    M->nlev = mg_levels_for(ctx->g.nx, ctx->g.ny, ctx->g.nz);
    M->lv[0].nx = ctx->g.nx;
    M->lv[0].ny = ctx->g.ny;
    M->lv[0].nz = ctx->g.nz;
    M->lv[0].nc = ctx->g.nc;
    for (int l = 1; l < M->nlev; l++) {
        MgLevelBuf& L = M->lv[l];
        L.nx = (M->lv[l - 1].nx + 1) / 2;
        L.ny = (M->lv[l - 1].ny + 1) / 2;
        L.nz = (M->lv[l - 1].nz + 1) / 2;
        L.nc = (int64_t)L.nx * L.ny * L.nz;
        float** arrs[6] = {&L.diag, &L.ox, &L.oy, &L.oz, &L.b, &L.x};
        for (float** a : arrs) {
            if (hipMalloc(reinterpret_cast<void**>(a), sizeof(float) * (size_t)L.nc) != hipSuccess)
                return set_err(ctx, FSIM_ERR_OOM, "multigrid level allocation failed");
            M->allocs.push_back(*a);
            FSIM_TRY(fill_f32(ctx, *a, 0.0f, L.nc));   // x must be 0 where a level has no unknown
        }
    }
    return FSIM_OK;
}

static Mg0 mg0(fsim_ctx* ctx, const float* r, float* z, double scale) {
    Mg0 A;
    A.nx = ctx->g.nx;
    A.ny = ctx->g.ny;
    A.nz = ctx->g.nz;
    A.nxp = ctx->g.nxp;
    A.nbinfo = ctx->nbinfo;
    A.b = r;
    A.x = z;
    A.binv = (float)(1.0 / scale);
    return A;
}

// Builds the coarse operators of the current labels (once per solve, after nbinfo).
int mg_setup(fsim_ctx* ctx) {
    FSIM_TRY(mg_alloc(ctx));
    MgState* M = ctx->mg;
    if (ctx->mg_coarse == FSIM_MG_COARSE_NETWORK) {   // the network's buffers exist before any capture
        const MgLevelBuf& L = M->lv[M->nlev - 1];
        if (M->nlev > 1) FSIM_TRY(learned_prepare(ctx, L.nx, L.ny, L.nz));
        else FSIM_TRY(learned_prepare(ctx, ctx->g.nx, ctx->g.ny, ctx->g.nz));
    }
    FSIM_PROF(ctx, KID_MG);
    if (M->nlev > 1) {
        MgLevelBuf& C = M->lv[1];
        hipLaunchKernelGGL(k_mg_coarsen0, dim3(nblocks(C.nc)), dim3(kBlock), 0, ctx->stream, mg0(ctx, nullptr, nullptr, 1.0),
                           C.nx, C.ny, C.nz, C.diag, C.ox, C.oy, C.oz);
        for (int l = 2; l < M->nlev; l++) {
            MgLevelBuf& L = M->lv[l];
            hipLaunchKernelGGL(k_mg_coarsen, dim3(nblocks(L.nc)), dim3(kBlock), 0, ctx->stream, grid_of(M->lv[l - 1]), L.nx,
                               L.ny, L.nz, L.diag, L.ox, L.oy, L.oz);
        }
    }
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

// blocks of the level-0 column kernels: one per item
static dim3 mg0_blocks(const Mg0& A) {
    return dim3((unsigned)(row_item_count(A.ny, A.nz, A.nxp) + 7) / 8 * 8);
}

static void smooth0(fsim_ctx* ctx, const Mg0& A, int sweeps, bool first) {
    const dim3 g = mg0_blocks(A), b(kBlock);
    for (int k = 0; k < sweeps; k++) {
        if (first && k == 0) hipLaunchKernelGGL((k_mg_rbgs0<1, true>), g, b, 0, ctx->stream, A);
        else hipLaunchKernelGGL((k_mg_rbgs0<1, false>), g, b, 0, ctx->stream, A);
        hipLaunchKernelGGL((k_mg_rbgs0<0, false>), g, b, 0, ctx->stream, A);
    }
}
static void smooth(fsim_ctx* ctx, const MgLevelBuf& L, int sweeps, bool first) {
    const MgGrid G = grid_of(L);
    const MgLaunch S = mg_launch(L.nx, L.ny, L.nz);
    const dim3 g = S.grid, b = S.block;
    for (int k = 0; k < sweeps; k++) {
        if (first && k == 0) hipLaunchKernelGGL((k_mg_rbgs<1, true>), g, b, 0, ctx->stream, G);
        else hipLaunchKernelGGL((k_mg_rbgs<1, false>), g, b, 0, ctx->stream, G);
        hipLaunchKernelGGL((k_mg_rbgs<0, false>), g, b, 0, ctx->stream, G);
    }
}

// Solves the coarsest level (lv[c], or level 0 itself when the grid is small).
static int coarse_solve(fsim_ctx* ctx, const Mg0& A, int c) {
    MgState* M = ctx->mg;
    const int mode = ctx->mg_coarse;
    const int nu = ctx->learned_smoothing;
    const double norm = std::ldexp(1.0, -2 * c);   // 4^-c: the level's operator on the network's scale
    if (mode == FSIM_MG_COARSE_NETWORK) {
        if (c == 0) {
            FSIM_TRY(learned_apply_level0(ctx, A.b, A.x, A.binv));
            smooth0(ctx, A, nu, false);
        } else {
            const MgLevelBuf& L = M->lv[c];
            FSIM_TRY(learned_apply_level(ctx, L.nx, L.ny, L.nz, L.b, L.diag, L.ox, L.oy, L.oz, norm, L.x));
            smooth(ctx, L, nu, false);
        }
        return FSIM_OK;
    }
    const int sweeps = mode == FSIM_MG_COARSE_ACCURATE ? kMgExactSweeps : std::max(nu, 1);
    if (c == 0) smooth0(ctx, A, sweeps, true);
    else smooth(ctx, M->lv[c], sweeps, true);
    if (mode == FSIM_MG_COARSE_ACCURATE && c > 0 && M->harvest_n < M->harvest_cap) {
        const MgLevelBuf& L = M->lv[c];
        const size_t bytes = sizeof(float) * (size_t)L.nc;
        FSIM_HIP(ctx, hipMemcpyAsync(M->hb + (size_t)M->harvest_n * L.nc, L.b, bytes, hipMemcpyDeviceToDevice, ctx->stream));
        FSIM_HIP(ctx, hipMemcpyAsync(M->hx + (size_t)M->harvest_n * L.nc, L.x, bytes, hipMemcpyDeviceToDevice, ctx->stream));
        M->harvest_n++;
    }
    return FSIM_OK;
}

// z = V-cycle(r) / s: level-0 vectors in the solver's rotated layout.
static int vcycle(fsim_ctx* ctx, const float* r, float* z, double scale) {
    MgState* M = ctx->mg;
    const Mg0 A = mg0(ctx, r, z, scale);
    const int c = M->nlev - 1;
    if (c == 0) {   // the grid itself is the coarse level
        FSIM_TRY(coarse_solve(ctx, A, 0));
        FSIM_HIP(ctx, hipGetLastError());
        return FSIM_OK;
    }
    // down: level 0, then 1 .. c-1
    smooth0(ctx, A, kMgPreSweeps, true);
    {
        const MgLevelBuf& L1 = M->lv[1];
        const dim3 g((unsigned)((L1.nx + kRtC - 1) / kRtC), (unsigned)L1.ny, (unsigned)((L1.nz + kRtC - 1) / kRtC));
        hipLaunchKernelGGL(k_mg_resid_restrict0, g, dim3(256), 0, ctx->stream, A, grid_of(L1));
    }
    for (int l = 1; l < c; l++) {
        smooth(ctx, M->lv[l], kMgPreSweeps, true);
        hipLaunchKernelGGL(k_mg_restrict, dim3(nblocks(8 * M->lv[l + 1].nc)), dim3(kBlock), 0, ctx->stream,
                           grid_of(M->lv[l]), grid_of(M->lv[l + 1]));
    }
    FSIM_TRY(coarse_solve(ctx, A, c));
    // up
    for (int l = c - 1; l >= 1; l--) {
        const MgLaunch P = mg_launch(M->lv[l].nx, M->lv[l].ny, M->lv[l].nz);
        hipLaunchKernelGGL(k_mg_prolong, P.grid, P.block, 0, ctx->stream, grid_of(M->lv[l]), grid_of(M->lv[l + 1]));
        smooth(ctx, M->lv[l], kMgPostSweeps, false);
    }
    hipLaunchKernelGGL(k_mg_prolong0, mg0_blocks(A), dim3(kBlock), 0, ctx->stream, A, grid_of(M->lv[1]));
    smooth0(ctx, A, kMgPostSweeps, false);
    FSIM_HIP(ctx, hipGetLastError());
    return FSIM_OK;
}

// The V-cycle is some 50 launches, most of them small: enqueued one by one they
// keep the GPU waiting on the host.  With FSIM_OPT_MG_GRAPH (default) it is
// captured once into a HIP graph and replayed; the kernels' arguments depend
// only on Key (the buffers are the context's, allocated before the capture),
// so a new capture is made only when Key changes.  The V-cycle records no
// memset node (the network clears its max|b| with a fill kernel).  Profiling
// (per-kernel events) and harvesting (host-side sample counts) run it
// directly.
int mg_apply(fsim_ctx* ctx, const float* r, float* z, double scale) {
    MgState* M = ctx->mg;
    FSIM_PROF(ctx, KID_MG);
    if (!ctx->mg_graph || ctx->prof_on || ctx->mg_harvesting) return vcycle(ctx, r, z, scale);
    const MgState::Key key{r, z, scale, ctx->mg_coarse, ctx->learned_smoothing, ctx->learned_conv_lds, ctx->learned_gen};
    if (!M->exec || !(key == M->key)) {
        drop_graph(M);
        FSIM_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        const int rc = vcycle(ctx, r, z, scale);
        hipGraph_t g = nullptr;
        const hipError_t ec = hipStreamEndCapture(ctx->stream, &g);
        if (rc != FSIM_OK || ec != hipSuccess || !g) {
            if (g) (void)hipGraphDestroy(g);
            return rc != FSIM_OK ? rc : set_err(ctx, FSIM_ERR_HIP, std::string("V-cycle capture: ") + hipGetErrorString(ec));
        }
        const hipError_t ei = hipGraphInstantiate(&M->exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ei != hipSuccess) {
            M->exec = nullptr;
            return set_err(ctx, FSIM_ERR_HIP, std::string("V-cycle graph: ") + hipGetErrorString(ei));
        }
        M->key = key;
    }
    FSIM_HIP(ctx, hipGraphLaunch(M->exec, ctx->stream));
    return FSIM_OK;
}

int mg_info(fsim_ctx* ctx, int* levels, int* dims) {
    const int n = mg_levels_for(ctx->g.nx, ctx->g.ny, ctx->g.nz);
    int d[3] = {ctx->g.nx, ctx->g.ny, ctx->g.nz};
    for (int l = 1; l < n; l++)
        for (int a = 0; a < 3; a++) d[a] = (d[a] + 1) / 2;
    if (levels) *levels = n;
    if (dims)
        for (int a = 0; a < 3; a++) dims[a] = d[a];
    return FSIM_OK;
}

// Harvest buffers for the next solve: cap coarse (b, x) pairs.
int mg_harvest_begin(fsim_ctx* ctx, int cap) {
    FSIM_TRY(mg_alloc(ctx));
    MgState* M = ctx->mg;
    if (M->nlev < 2) return set_err(ctx, FSIM_ERR_INVALID, "the grid has no coarse multigrid level to harvest");
    const int64_t nc = M->lv[M->nlev - 1].nc;
    if (cap > M->harvest_cap) {
        float *hb = nullptr, *hx = nullptr;
        if (hipMalloc(reinterpret_cast<void**>(&hb), sizeof(float) * (size_t)cap * nc) != hipSuccess ||
            hipMalloc(reinterpret_cast<void**>(&hx), sizeof(float) * (size_t)cap * nc) != hipSuccess) {
            if (hb) (void)hipFree(hb);
            return set_err(ctx, FSIM_ERR_OOM, "harvest buffer allocation failed");
        }
        FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (M->hb) (void)hipFree(M->hb);
        if (M->hx) (void)hipFree(M->hx);
        M->hb = hb;
        M->hx = hx;
        M->harvest_cap = cap;
    }
    M->harvest_n = 0;
    return FSIM_OK;
}

// Copies the harvested pairs and the coarse operator (normalised by 4^-level) to the host.
int mg_harvest_end(fsim_ctx* ctx, int cap, float* b, float* op, float* x, int* n_out) {
    MgState* M = ctx->mg;
    const int c = M->nlev - 1;
    const MgLevelBuf& L = M->lv[c];
    const int n = std::min(M->harvest_n, cap);
    FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const size_t nc = (size_t)L.nc;
    if (n > 0) {
        FSIM_HIP(ctx, hipMemcpy(b, M->hb, sizeof(float) * nc * n, hipMemcpyDeviceToHost));
        FSIM_HIP(ctx, hipMemcpy(x, M->hx, sizeof(float) * nc * n, hipMemcpyDeviceToHost));
    }
    std::vector<float> tmp(nc);
    const float* src[4] = {L.diag, L.ox, L.oy, L.oz};
    const float norm = std::ldexp(1.0f, -2 * c);
    for (int k = 0; k < 4; k++) {
        FSIM_HIP(ctx, hipMemcpy(tmp.data(), src[k], sizeof(float) * nc, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < nc; i++) op[k * nc + i] = tmp[i] * norm;
    }
    // the samples' x solve L x = b; on the network's scale (L / 4^c) x / 4^c solves it
    for (size_t i = 0; i < nc * (size_t)n; i++) x[i] /= norm;
    M->harvest_n = 0;
    *n_out = n;
    return FSIM_OK;
}

}  // namespace fsim
