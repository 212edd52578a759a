// fsim_internal.hpp — device state and launch interfaces of libfsim_hip.so.
//
// Device layout (one context, one GPU):
//   * grid fields are dense arrays over all Nc = Nx*Ny*Nz cells in the
//     reference's flat order idx = (x*Ny + y)*Nz + z (z fastest);
//   * face velocities are FP32 SoA: u,v,w (P2G result after boundary
//     conditions, the reference's Face::v) and u2,v2,w2 (Face::v2);
//   * labels are uint8 fsim_cell_type; nbinfo (uint16) caches, per WATER cell,
//     which of the 6 neighbours are WATER and how many are not SOLID;
//   * pressure-solve vectors are dense FP32 (b, r, z, s, q) with FP64
//     pressure x and FP64 MIC(0) diagonal; entries outside WATER cells are 0;
//     they and nbinfo use the rotated layout of ridx() below;
//   * particles are FP32 SoA (pos, vel, APIC C) plus the int32 particle id
//     (its index in the reference's particle vector), kept sorted by cell
//     after every BIN stage.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/fsim.h"

namespace fsim {

constexpr int kMaxObstacles = 64;
constexpr int kBlock = 256;
constexpr unsigned kMaxParts = 2048;   // reduction grids have at most this many blocks

// nbinfo bit layout
constexpr uint16_t NB_FLUID = 1u << 0;      // the cell itself is an interior WATER cell
constexpr uint16_t NB_MX = 1u << 1;         // -x neighbour is WATER (fluid)
constexpr uint16_t NB_MY = 1u << 2;
constexpr uint16_t NB_MZ = 1u << 3;
constexpr uint16_t NB_PX = 1u << 4;         // +x neighbour is WATER (fluid)
constexpr uint16_t NB_PY = 1u << 5;
constexpr uint16_t NB_PZ = 1u << 6;
constexpr int NB_NONSOLID_SHIFT = 7;        // bits 7..9: number of non-SOLID neighbours
// bits 10..15: for each axis a, whether the -a neighbour's +((a+1)%3) and
// +((a+2)%3) neighbours are WATER (the MIC(0) factor's "other" terms)
constexpr int NB_UP_SHIFT = 10;

// Persistent wavefront kernels (MIC(0) factor and triangular sweeps): a tile
// of WF_TY x WF_TZ (y, z) columns per workgroup, WF_NW compute waves of WF_R
// rows each plus three communication waves.
constexpr int WF_R = 2;
constexpr int WF_NW = 3;
constexpr int WF_TY = WF_R * WF_NW;
constexpr int WF_TZ = 64;
constexpr int WF_G = 4;                           // planes per storage group (and steps per handshake)
constexpr int WF_THREADS = (WF_NW + 3) * WF_TZ;   // compute waves, 2 receiving and a sending edge wave
// the wavefront kernels address cells with 32-bit byte offsets into arrays of
// 4-byte words, whose padded length is at most twice the cells (nx = 4 is
// stored as 8 planes); larger grids use the plane-by-plane kernels
constexpr int64_t kWaveMaxCells = ((int64_t(1) << 31) - 1) / 8;

// Solver-vector layout ("rotated, in groups of four planes").  Cell (x, y, z)
// of the pressure solve belongs to plane p = (x + ((z - 1) mod 64)) mod nxp,
// so that the 64 cells of a z-tile [1 + 64k, 64 + 64k] that one wavefront
// step visits (x = c - ((z - 1) mod 64)) share one plane.  Four consecutive
// planes are stored interleaved, the plane fastest: a lane that owns a (y, z)
// column moves the values of four steps with one 16-byte access, and a wave
// 1 KB of contiguous memory (a vector-memory instruction costs a compute unit
// about 16 cycles whether its lanes move 4 or 16 bytes).  The map is a
// bijection of every (y, z) column onto nxp planes, nxp = nx + 1 rounded up to
// whole groups: the planes beyond nx hold no cell (zeros), and no group holds
// both the first and the last interior cells of a column.
__host__ __device__ inline int rot_planes(int nx) { return (nx + WF_G) / WF_G * WF_G; }
__host__ __device__ inline int rot_of(int z) { return (z - 1) & (WF_TZ - 1); }
__host__ __device__ inline int rot_plane(int x, int z, int nxp) {
    const int p = x + rot_of(z);
    return p < nxp ? p : p % nxp;
}
// x of plane p's cell in column z: nx .. nxp - 1 on a padding plane
__host__ __device__ inline int unrot_x(int p, int z, int nxp) {
    const int x = p - rot_of(z);
    return x >= 0 ? x : (x % nxp + nxp) % nxp;
}
// storage index of plane p, row y, column z
__host__ __device__ inline int64_t pidx(int p, int y, int z, int ny, int nz) {
    return ((((int64_t)(p / WF_G) * ny + y) * nz + z) * WF_G) + (p & (WF_G - 1));
}
__host__ __device__ inline int64_t ridx(int x, int y, int z, int nxp, int ny, int nz) {
    return pidx(rot_plane(x, z, nxp), y, z, ny, nz);
}

// f(flat index, index in the rotated layout) of every cell, in flat order, on the host.  The planes' places come from a
// table: the index arithmetic of ridx for every cell made reading a small field 15 % slower than with one plane a row.
template <class F>
inline void for_rotated(int nx, int ny, int nz, int nxp, F&& f) {
    std::vector<int64_t> place((size_t)nx + WF_TZ - 1);   // of plane p, unwrapped
    for (size_t p = 0; p < place.size(); p++) place[p] = pidx((int)(p % nxp), 0, 0, ny, nz);
    int64_t i = 0;
    for (int x = 0; x < nx; x++)
        for (int y = 0; y < ny; y++)
            for (int z = 0; z < nz; z++, i++) f(i, place[x + rot_of(z)] + ((int64_t)y * nz + z) * WF_G);
}

// Dimensions and scale of a pressure solve; stencil neighbours in the rotated layout.
struct SolveArgs {
    int nx, ny, nz;
    int nxp;            // planes of the rotated layout
    int64_t nc;         // cells (flat fields)
    int64_t ncr;        // values of a solver vector: nxp * ny * nz
    float scale_f;      // dt / (rho dx^2)
    double scale;
};

// flat index of the grid fields (labels, velocities, density)
__device__ inline int64_t sidx(const SolveArgs& S, int x, int y, int z) { return ((int64_t)x * S.ny + y) * S.nz + z; }
// index of the solver vectors, nbinfo and the factor (rotated layout)
__device__ inline int64_t rsidx(const SolveArgs& S, int x, int y, int z) { return ridx(x, y, z, S.nxp, S.ny, S.nz); }
// Indices around the four cells that one lane owns: planes 4g .. 4g + 3 of
// column (y, z).  +-y are the same planes of the next rows; the +-x
// neighbours of three of the four are the lane's own, the fourth's are element
// 0 of the next group and element 3 of the previous one; +-z move one column
// and one plane: elements 1, 2, 3 of group gp and 0 of the group after it (+z),
// element 3 of the group before gm and 0, 1, 2 of gm (-z), with gp = gm = g
// except across a z-tile edge, where the plane moves 63 = 4 * 16 - 1 back or
// ahead.  All are in range for an interior column.
struct ColumnNeighbours {
    int64_t own, yp, ym, zp, zm;      // 16-byte accesses
    int64_t xp3, xm0, zp3, zm0;       // single values: +x and +z of element 3, -x and -z of element 0
};
__device__ inline ColumnNeighbours column_neighbours(int ny, int nz, int ng, int g, int y, int z) {
    const int64_t gs = (int64_t)ny * nz * WF_G;
    const int64_t col = ((int64_t)y * nz + z) * WF_G;
    const int rz = rot_of(z);
    const int far = ng > 16 ? 16 : 16 % ng;
    const int gp = rz == WF_TZ - 1 ? (g >= far ? g - far : g - far + ng) : g;
    const int gm = rz == 0 ? (g + far >= ng ? g + far - ng : g + far) : g;
    ColumnNeighbours n;
    n.own = g * gs + col;
    n.yp = n.own + (int64_t)nz * WF_G;
    n.ym = n.own - (int64_t)nz * WF_G;
    n.zp = gp * gs + col + WF_G;
    n.zm = gm * gs + col - WF_G;
    n.xp3 = (g + 1 == ng ? 0 : g + 1) * gs + col;
    n.xm0 = (g == 0 ? ng - 1 : g - 1) * gs + col + 3;
    n.zp3 = (gp + 1 == ng ? 0 : gp + 1) * gs + col + WF_G;
    n.zm0 = (gm == 0 ? ng - 1 : gm - 1) * gs + col - WF_G + 3;
    return n;
}
// Work split of the stencil kernels over the columns: a block of kRowWaves
// waves takes kRowWaves consecutive interior rows of one plane group and one
// z-tile at a time (wave: row, lane l: column z0 + l, whose rotation is l).
// Workgroups are dispatched round-robin over the 8 XCDs (blockIdx mod 8), so
// the block items are cut into 8 contiguous ranges, one per XCD: the +-x/+-y
// neighbours a block reads were loaded by blocks of the same XCD (its L2).
constexpr int kRowWaves = 4;
struct RowItems {
    int ntile, nrow;
    int end;           // end of this XCD's item range (items fit in 32 bits: at most a 64th of the values)
    int first, step;   // this block's first item and stride
};
__host__ __device__ inline int row_item_count(int ny, int nz, int nxp) {
    return nxp / WF_G * ((ny - 2 + kRowWaves - 1) / kRowWaves) * ((nz - 2 + WF_TZ - 1) / WF_TZ);
}
__device__ inline RowItems row_items(int ny, int nz, int nxp) {
    RowItems it;
    it.ntile = (nz - 2 + WF_TZ - 1) / WF_TZ;
    it.nrow = (ny - 2 + kRowWaves - 1) / kRowWaves;
    const int total = row_item_count(ny, nz, nxp);
    const int per_xcd = (total + 7) / 8;
    const int begin = (int)(blockIdx.x & 7) * per_xcd;
    it.end = min(total, begin + per_xcd);
    it.first = begin + (int)(blockIdx.x >> 3);
    it.step = (int)(gridDim.x >> 3);
    return it;
}
// plane group, row and column of this thread for item k; false past the grid's rows or columns
__device__ inline bool item_column(const RowItems& it, int k, int ny, int nz, int& g, int& y, int& z) {
    const int c = k % it.ntile;
    const int rest = k / it.ntile;
    y = 1 + rest % it.nrow * kRowWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    g = rest / it.nrow;
    z = 1 + c * WF_TZ + (threadIdx.x & 63);
    return y <= ny - 2 && z <= nz - 2;
}
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

// rotated indices of the +a and -a neighbours of interior cell (x, y, z)
__device__ inline int64_t rnb_plus(const SolveArgs& S, int x, int y, int z, int a) {
    return rsidx(S, x + (a == 0), y + (a == 1), z + (a == 2));
}
__device__ inline int64_t rnb_minus(const SolveArgs& S, int x, int y, int z, int a) {
    return rsidx(S, x - (a == 0), y - (a == 1), z - (a == 2));
}

struct WaveArgs {
    int nx, ny, nz, nxp;
    int TJ, TK;                   // tiles along y and z
    int SG;                       // boundary-packet rows (groups of WF_G steps) per tile
    const uint16_t* nbinfo;
    const float* in;
    float* out;
    float ms;                     // -scale in FP32
    double scale;                 // dt / (rho dx^2)
    double* P64;
    float* P32;
    uint4* ybnd;                  // packets across y tile edges: [tile J*TK+K][group][1 or 2][64]
    uint4* zbnd;                  // packets across z tile edges: [tile J*TK+K][group][1 or 2][WF_TY]
    unsigned long long* ticket;
    unsigned long long ticket_base;
    int* err;
    const uint8_t* tilew;         // [2][TJ * TK]: 1 if the tile holds a WATER cell, forward and backward tiles
    const int* xrange;            // {least x, greatest x} of the WATER cells
    int send_delay;               // test option: s_sleep(127) periods of the sending waves per group
};

struct GridDims {
    int nx, ny, nz;
    int64_t nc;
    int nxp;              // planes of the solver vectors' rotated layout
    int64_t ncr;          // values of a solver vector
    double cd, cdinv;     // cellD.x == cellD.y
    double cdz, cdzinv;   // cellD.z (cd except in 2D)
    double dims[3];
    double pr;
    int two_d;
};

// Device-resident scalars of the pressure solve (one cache line each group).
struct SolveScalars {
    double sigma, alpha, beta, sq;   // PCG scalars
    double alpha_prev;               // alpha of the direction step before
    double rr, rmax, bb;             // recursive residual ||r||^2, max|r|, ||b||^2
    double tr_ss, tr_max;            // true residual ||b-Ax||^2, max|b-Ax|
    double zr;                       // z.r
    double nfluid;                   // number of WATER cells of the solve
    int64_t wave_err;                // host copy: the wavefront kernels' error flag
    int nan_flag;
    unsigned seq;                    // host copy: number of the reduction that wrote it
};

// Kernel groups timed with HIP events when profiling is on.
enum KernelId {
    KID_SPAWN = 0, KID_MOVE, KID_BIN_KEYS, KID_BIN_SCAN, KID_BIN_SCATTER, KID_BIN_SEGSORT, KID_BIN_GATHER,
    KID_P2G, KID_MARK, KID_OBSTACLES, KID_BORDERS, KID_POST_P2G, KID_RHS, KID_MIC_FACTOR, KID_SWEEP_FWD,
    KID_SWEEP_BWD, KID_SPMV, KID_UPDATE, KID_DOT, KID_TRUE_RES, KID_PRESSURE, KID_EXTRAPOLATE, KID_G2P,
    KID_LEARNED, KID_SOR, KID_PUSH_APART, KID_MG, KID_COUNT
};

struct Particles {
    int64_t n = 0, cap = 0;
    float* base = nullptr;   // one allocation, 16 float planes of cap entries
    float* pos[3] = {};
    float* vel[3] = {};
    float* c[9] = {};
    int32_t* pid = nullptr;
};

}  // namespace fsim

namespace fsim {
struct LearnedNet;
struct MgState;
constexpr int kMgMaxLevels = 8;
constexpr int kMgCoarseMaxSide = 16;   // the network's level: the first whose largest side is <= this
}

struct fsim_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    fsim::GridDims g{};
    fsim_params prm{};
    std::string err;

    // particles (double-buffered for the binning gather)
    fsim::Particles P, Palt;
    uint32_t* key = nullptr;     // cell key per particle (Nc = removed)
    int32_t* rank = nullptr;     // slot within cell from the histogram atomics
    int32_t* perm = nullptr;     // sorted slot -> source slot
    int64_t pwork_cap = 0;
    uint8_t* removed = nullptr;  // sink removal flags (per particle)
    bool c_valid = true;         // APIC matrices carried (false after a PIC/FLIP bin)
    int64_t scan_tmp_cap = 0;

    // grid
    float *u = nullptr, *v = nullptr, *w = nullptr;
    float *u2 = nullptr, *v2 = nullptr, *w2 = nullptr;
    uint8_t* label = nullptr;
    uint8_t* valid = nullptr;
    float* density = nullptr;
    int32_t* cell_count = nullptr;   // Nc + 1 (last = removed particles)
    int32_t* cell_start = nullptr;   // Nc + 2
    int32_t* scan_tmp = nullptr;
    uint16_t* nbinfo = nullptr;
    uint8_t* colw = nullptr;          // WATER columns (y, z) of the current labels, for the wavefront kernels,
                                      // and behind them the x range of the WATER cells (WaveArgs::xrange)
                                      // and the chunk flags
    uint32_t* chunk_flags = nullptr;  // solver-vector chunks (256 values) holding a WATER cell, per solve

    // pressure solve
    float* vectors = nullptr;         // the allocation of the FP32 vectors below
    float *b = nullptr, *r = nullptr, *z = nullptr, *s = nullptr, *q = nullptr;
    float* s2 = nullptr;              // second search-direction buffer (swapped with s)
    float* t = nullptr;               // forward sweep's result
    float* r_next = nullptr;          // MIC(0)-PCG: second residual buffer
    float* P32 = nullptr;
    double* P64 = nullptr;
    double* x = nullptr;
    double* sor64 = nullptr;          // BasicMacGrid SOR: FP64 faces u, v, w (allocated on first use)
    double* partials = nullptr;       // block partial sums (FP64)
    unsigned* red_count = nullptr;    // blocks finished in the running reduction (0 between launches)
    unsigned scal_seq = 0;                 // last reduction that writes scal_host
    int last_mic_iterations = 0;      // MIC(0)-PCG iterations of the last solve that used it
    int learned_since_mic = 0;        // learned solves since that MIC(0) solve
    int learned_refresh = 50;         // learned solves between MIC(0) solves that renew the count (0: never)
    fsim::LearnedNet* learned = nullptr;   // learned preconditioner (network parameters and buffers)
    fsim::MgState* mg = nullptr;          // multigrid hierarchy of the learned preconditioner
    int mg_coarse = 0;                    // coarsest-level solve: FSIM_MG_COARSE_*
    int reliable_drop = 3;                // PCG: true residual after a 10^drop drop of the recursive one (0: at the tolerance)
    int mg_graph = 1;                     // replay the multigrid V-cycle as a HIP graph
    int p2g_rows = 0;                     // 1: the one-row-per-block P2G gather instead of the tiled one
    int wave_send_delay = 0;              // test option: sending-wave pause per step (s_sleep 127 units)
    int learned_gen = 0;                  // bumped when the network's per-size buffers are reallocated
    bool mg_harvesting = false;           // a solve run by fsim_learned_harvest
    fsim::SolveScalars* scal = nullptr;   // device
    fsim::SolveScalars* scal_host = nullptr;  // pinned host mirror
    double last_dt = 0.0;
    // wavefront sweeps
    fsim::WaveArgs wave{};
    uint4* ybnd = nullptr;
    uint4* zbnd = nullptr;
    unsigned long long* wave_ticket = nullptr;   // 3 counters: factor, fwd, bwd
    unsigned long long wave_ticket_base[3] = {0, 0, 0};
    int64_t wave_packets[2] = {0, 0};            // 16-byte packets of ybnd, zbnd
    int* wave_err = nullptr;
    int sweep_mode = 0;                          // 0 wavefront, 1 one launch per plane
    int learned_smoothing = 2;                   // red-black sweeps after the network on the coarsest level
    int learned_loss = 0;                        // training loss: 0 masked MSE, 1 energy norm
    int learned_conv_lds = 1;                    // 1: LDS-staged convolutions where they fit

    // renderer snapshot staging (grown on demand)
    fsim_gfx_particle* gfx_staging = nullptr;
    int64_t gfx_cap = 0;

    bool rb_counted = false;

    // obstacles
    std::vector<fsim_obstacle> obs;
    fsim_obstacle* obs_dev = nullptr;
    uint64_t spawn_calls = 0;

    // timing
    hipEvent_t ev[2 * FSIM_NUM_TIMERS + 4] = {};
    fsim_step_stats stats{};
    // per-kernel profiling
    bool prof_on = false;
    std::vector<hipEvent_t> prof_pool;
    size_t prof_next = 0;
    std::vector<int> prof_pending;   // triples: kernel id, start event, end event
    double prof_ms[fsim::KID_COUNT] = {};
    int64_t prof_n[fsim::KID_COUNT] = {};
};

namespace fsim {

// ---- error plumbing ------------------------------------------------------
int set_err(fsim_ctx* ctx, int code, const std::string& msg);
#define FSIM_HIP(ctx, expr)                                                              \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess)                                                            \
            return ::fsim::set_err((ctx), FSIM_ERR_HIP,                                  \
                                   std::string(#expr) + ": " + hipGetErrorString(e_));   \
    } while (0)
#define FSIM_TRY(expr)              \
    do {                            \
        int rc_ = (expr);           \
        if (rc_ != FSIM_OK) return rc_; \
    } while (0)

inline unsigned nblocks(int64_t n, int b = kBlock) { return (unsigned)((n + b - 1) / b); }

// ---- profiling (fsim_capi.hip) ----------------------------------------------
int set_profiling(fsim_ctx* ctx, bool on);
int prof_event(fsim_ctx* ctx);          // records a pooled event, returns its index (-1 if off)
void prof_close(fsim_ctx* ctx, int kid, int start);
int prof_collect(fsim_ctx* ctx);        // after a stream synchronisation

// Times the enclosed launches as kernel group `kid` when profiling is on.
struct ProfRange {
    fsim_ctx* c;
    int kid, start;
    ProfRange(fsim_ctx* ctx, int k) : c(ctx), kid(k), start(prof_event(ctx)) {}
    ~ProfRange() {
        if (start >= 0) prof_close(c, kid, start);
    }
};
#define FSIM_CAT2(a, b) a##b
#define FSIM_CAT(a, b) FSIM_CAT2(a, b)
#define FSIM_PROF(ctx, kid) ::fsim::ProfRange FSIM_CAT(prof_range_, __LINE__)((ctx), (kid))

// ---- particle stages (fsim_particles.hip) ---------------------------------
int particles_reserve(fsim_ctx* ctx, int64_t n);
int stage_spawn(fsim_ctx* ctx, double dt);
// flags: 1 = advect, 2 = push out, 4 = stop particles
int stage_move(fsim_ctx* ctx, double dt, int flags);
int stage_bin(fsim_ctx* ctx);
int stage_push_apart(fsim_ctx* ctx);
int upload_obstacles(fsim_ctx* ctx);

// ---- grid stages (fsim_grid.hip) ------------------------------------------
int stage_p2g(fsim_ctx* ctx);
int stage_mark(fsim_ctx* ctx);
int stage_obstacles(fsim_ctx* ctx);
int stage_borders(fsim_ctx* ctx);
int stage_post_p2g(fsim_ctx* ctx, double grav_inc);
int stage_extrapolate(fsim_ctx* ctx);
int stage_g2p(fsim_ctx* ctx);
int fill_u8(fsim_ctx* ctx, uint8_t* p, uint8_t v, int64_t n);
int fill_f32(fsim_ctx* ctx, float* p, float v, int64_t n);
int fill_f64(fsim_ctx* ctx, double* p, double v, int64_t n);
int fill_i32(fsim_ctx* ctx, int32_t* p, int32_t v, int64_t n);

// ---- pressure solve (fsim_solver.hip) -------------------------------------
int stage_solve(fsim_ctx* ctx, double dt);
// WAVE_FWD_UPDATE: the forward sweep of in - alpha side->q; side: null or what further blocks do (fsim_reduce.hpp)
// WAVE_FWD_ALONE and WAVE_BWD_ALONE: the sweeps outside a solve, which hold the cells off WATER at 0 whatever the input
enum WaveKind {
    WAVE_FACTOR = 0, WAVE_FWD = 1, WAVE_BWD = 2, WAVE_FWD_UPDATE = 3, WAVE_FWD_ALONE = 4, WAVE_BWD_ALONE = 5
};
struct SideWork;
int wave_launch(fsim_ctx* ctx, WaveKind kind, const float* in, float* out, double scale, const SideWork* side);
int wave_init(fsim_ctx* ctx);
int solver_apply(fsim_ctx* ctx, int op, double dt, const double* in, double* out);

// ---- renderer snapshot (fsim_gfx.hip) --------------------------------------
int gfx_snapshot(fsim_ctx* ctx, fsim_gfx_particle* host_out);
int gfx_snapshot_noalloc(fsim_ctx* ctx, fsim_gfx_particle* host_out);
int scratch_init(fsim_ctx* ctx);
int64_t scratch_particles();
void gfx_free(fsim_ctx* ctx);

// ---- results to host memory (fsim_readback.hip) ------------------------------
// dst = src after the stream's work so far; returns when dst is complete
int read_back(fsim_ctx* ctx, void* dst, const void* src, size_t bytes);
// positions, velocities and C in the reference's particle order; each may be null
int particles_out(fsim_ctx* ctx, float* pos, float* vel, float* c);
void readback_init(fsim_ctx* ctx);
void readback_free(fsim_ctx* ctx);

// ---- multigrid of the learned preconditioner (fsim_mg.hip) ------------------
int mg_levels_for(int nx, int ny, int nz);
int mg_setup(fsim_ctx* ctx);                                        // coarse operators of the current labels
int mg_apply(fsim_ctx* ctx, const float* r, float* z, double scale);  // z = V-cycle(r), rotated layout
int mg_info(fsim_ctx* ctx, int* levels, int* dims);
int mg_harvest_begin(fsim_ctx* ctx, int cap);
int mg_harvest_end(fsim_ctx* ctx, int cap, float* b, float* op, float* x, int* n_out);
void mg_free(fsim_ctx* ctx);

// ---- learned preconditioner (fsim_learned.hip) ------------------------------
// the network on the coarsest multigrid level (flat, operator arrays): x = out * max|b| * norm
int learned_apply_level(fsim_ctx* ctx, int nx, int ny, int nz, const float* b, const float* diag, const float* ox,
                        const float* oy, const float* oz, double norm, float* x);
// the network on the solve's own grid (rotated layout): z = out * max|r| * binv
int learned_prepare(fsim_ctx* ctx, int nx, int ny, int nz);
int learned_apply_level0(fsim_ctx* ctx, const float* r, float* z, float binv);
int64_t learned_num_params();
int learned_init(fsim_ctx* ctx, uint64_t seed);
int learned_set_params(fsim_ctx* ctx, const float* params);
int learned_get_params(fsim_ctx* ctx, float* params);
bool learned_ready(const fsim_ctx* ctx);
void label_operator(int nx, int ny, int nz, const uint8_t* label, float* op);   // op[4][nc] of a label field
int learned_forward_host(fsim_ctx* ctx, const float* b, const float* op, float* out);
int learned_grad_host(fsim_ctx* ctx, const float* b, const float* op, const double* p, float* grad, double* loss);
int learned_train_batch(fsim_ctx* ctx, int n, const float* b, const float* op, const double* p, float lr,
                        double* mean_loss);
void learned_free(fsim_ctx* ctx);

}  // namespace fsim
