// Marching work split of the stencil kernels over solver vectors: a wave
// takes kMarchRows rows of one z-tile and walks along a run of plane groups.
// It holds the own and the next group of its rows in registers, so of the
// neighbours of a cell
//   +-x  are the lane's own registers (elements of the same or the next group,
//        the last element of the group before),
//   +-z  come from the neighbouring lane (the columns of a tile differ by one
//        plane per lane, so it is the same element shift as +-x); at the two
//        edges of the tile from one more load, in which lane r holds the column
//        before row r of the tile and lane kMarchRows + r the one after it,
//   +-y  are the other rows' registers, and one row below and above is loaded.
// Per row and group it loads (kMarchRows + 3) / kMarchRows times 16 bytes per
// lane and vector, where a lane that gathers takes 9 loads.
#pragma once
#include "fsim_internal.hpp"

namespace fsim {

// Sizes: the matrix product with 2 rows, 4 waves and 512 blocks takes
// 10 / 12.5 / 17.5 / 65 us on 32^3, 128 x 128 x 3, 128^3 and 256^3; 4 rows
// 12 / 12.5 / 17 / 65, 1 row 10 / 12.5 / 18 / 68, 1024 blocks 10 / 15 / 19 / 67
// (every block takes a ticket of the reduction), 8 waves 11 / 12 / 17 / 71.
constexpr int kMarchRows = 2;      // rows of a wave
constexpr int kMarchWaves = 4;     // waves of a block: consecutive row blocks
constexpr int kMarchBlocks = 512;  // blocks that the runs are cut for
constexpr int kMarchRun = 16;      // consecutive items of one XCD
constexpr unsigned kBesideMarch = 256;   // blocks that a kernel may run beside the march in the same reduction
static_assert(kMarchBlocks + kBesideMarch <= kMaxParts, "march grid within the reduction");

// Items are ordered row blocks first, then z-tiles, then runs of groups.
// Workgroups are dispatched round-robin over the 8 XCDs (blockIdx mod 8): each
// XCD takes kMarchRun consecutive items (rows next to each other share its L2)
// in turn, so that a fluid that fills one side of the grid loads them alike.
struct MarchPlan {
    int ntile, nrow, len, items;
};
static inline MarchPlan march_of(int ny, int nz, int nxp) {
    MarchPlan m;
    m.ntile = (nz - 2 + WF_TZ - 1) / WF_TZ;
    m.nrow = (ny - 2 + kMarchRows * kMarchWaves - 1) / (kMarchRows * kMarchWaves);
    const int ng = nxp / WF_G;
    const int64_t whole = (int64_t)m.ntile * m.nrow * ng;
    m.len = (int)std::min<int64_t>(ng, (whole + kMarchBlocks - 1) / kMarchBlocks);
    m.items = m.ntile * m.nrow * ((ng + m.len - 1) / m.len);
    return m;
}
static inline unsigned march_blocks(const MarchPlan& m) {
    const int unit = 8 * kMarchRun;
    return (unsigned)std::min<int64_t>((m.items + unit - 1) / unit * unit, (kMaxParts - kBesideMarch) / unit * unit);
}

__device__ inline float lane_next(float v, float last) {   // lane i + 1's value; lane 63: last
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, last), __builtin_bit_cast(int, v),
                                                                 0x130, 0xf, 0xf, false));
}
__device__ inline float lane_prev(float v, float first) {   // lane i - 1's value; lane 0: first
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, first), __builtin_bit_cast(int, v),
                                                                 0x138, 0xf, 0xf, false));
}
__device__ inline float lane_value(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// the cells of a lane in one row and group: info words, values and the six neighbours
struct MarchCells {
    u16x4 info;
    f32x4 own, xp, xm, yp, ym, zp, zm;
};

// Raw load(int64_t j): the vectors at index j (a multiple of 4), without
// branches; f32x4 value(const Raw&): what the stencil is applied to, 0 off
// WATER; blocks: the grid's first ones, that march (a multiple of 8 kMarchRun); body(int64_t j, const MarchCells&): called for the lanes with WATER.
// Columns without WATER read index 0, a border cell, whose values are zero.
template <class Load, class Value, class Body>
__device__ inline void march(const MarchPlan& m, unsigned blocks, int ny, int nz, int nxp,
                             const uint16_t* __restrict__ nbinfo, Load&& load, Value&& value, Body&& body) {
    constexpr int R = kMarchRows;
    using Raw = decltype(load((int64_t)0));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ng = nxp / WF_G;
    const int64_t gs = (int64_t)ny * nz * WF_G, rs = (int64_t)nz * WF_G;
    const int far = ng > 16 ? 16 : 16 % ng;
    auto any = [](u16x4 f) { return ((f[0] | f[1] | f[2] | f[3]) & NB_FLUID) != 0; };
    for (int b = blockIdx.x;; b += blocks) {
        const int j = b >> 3;
        const int item = (j / kMarchRun * 8 + (b & 7)) * kMarchRun + j % kMarchRun;
        if (j / kMarchRun * 8 * kMarchRun >= m.items) break;
        if (item >= m.items) continue;
        const int rest = item / m.nrow;
        const int y0 = 1 + (item % m.nrow * kMarchWaves + wave) * R;
        const int tz = rest % m.ntile * WF_TZ;
        const int g0 = rest / m.ntile * m.len, g1 = min(g0 + m.len, ng);
        if (y0 > ny - 2) continue;
        const int zc = 1 + tz + lane;
        const bool in = zc <= nz - 2;
        const int64_t col = ((int64_t)y0 * nz + zc) * WF_G;
        auto wrap = [&](int g) { return g >= ng ? g - ng : g; };
        // the tile's edge columns
        const int er = lane < R ? lane : lane - R;
        const int ez = lane < R ? tz : tz + WF_TZ + 1;
        const bool ein = lane < 2 * R && y0 + er <= ny - 2 && ez <= nz - 1;
        const int64_t ecol = ((int64_t)(y0 + er) * nz + ez) * WF_G;
        auto edge = [&](int g) {
            const int e = lane < R ? wrap(g + far) : (g >= far ? g - far : g - far + ng);
            return load(ein ? e * gs + ecol : 0);
        };
        auto info_at = [&](int g, int r) {
            const bool on = in && y0 + r <= ny - 2;
            const u16x4 v = *reinterpret_cast<const u16x4*>(nbinfo + (on ? g * gs + col + r * rs : 0));
            return on ? v : u16x4{0, 0, 0, 0};
        };
        u16x4 info[R], info_n[R];
        f32x4 own[R], e;
        float last[R], e_last;
        {
            const int gm = g0 == 0 ? ng - 1 : g0 - 1, gn = wrap(g0 + 1);
            Raw pr[R], ow[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                info[r] = info_at(g0, r);
                info_n[r] = info_at(gn, r);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const bool on = in && y0 + r <= ny - 2;   // not by the info words: one round trip for both
                pr[r] = load(on ? gm * gs + col + r * rs : 0);
                ow[r] = load(on ? g0 * gs + col + r * rs : 0);
            }
            const Raw ep = edge(gm), eo = edge(g0);
#pragma unroll
            for (int r = 0; r < R; r++) {
                last[r] = value(pr[r])[3];
                own[r] = value(ow[r]);
            }
            e_last = value(ep)[3];
            e = value(eo);
        }
        for (int g = g0; g < g1; g++) {
            const int gn = wrap(g + 1), gnn = wrap(gn + 1);
            Raw nx[R];
#pragma unroll
            for (int r = 0; r < R; r++) nx[r] = load(any(info_n[r]) ? gn * gs + col + r * rs : 0);
            const Raw hm = load(any(info[0]) ? g * gs + col - rs : 0);
            const Raw hp = load(any(info[R - 1]) ? g * gs + col + R * rs : 0);
            const Raw en = edge(gn);
            u16x4 info_nn[R];
#pragma unroll
            for (int r = 0; r < R; r++) info_nn[r] = info_at(gnn, r);
            f32x4 next[R];
#pragma unroll
            for (int r = 0; r < R; r++) next[r] = value(nx[r]);
            const f32x4 ym0 = value(hm), ypR = value(hp), e_next = value(en);
#pragma unroll
            for (int r = 0; r < R; r++) {
                MarchCells c;
                c.info = info[r];
                c.own = own[r];
                c.xp = f32x4{own[r][1], own[r][2], own[r][3], next[r][0]};
                c.xm = f32x4{last[r], own[r][0], own[r][1], own[r][2]};
                c.yp = r + 1 < R ? own[r + 1 < R ? r + 1 : r] : ypR;
                c.ym = r > 0 ? own[r > 0 ? r - 1 : 0] : ym0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    c.zp[k] = lane_next(c.xp[k], lane_value(k < 3 ? e[(k + 1) & 3] : e_next[0], R + r));
                    c.zm[k] = lane_prev(c.xm[k], lane_value(k > 0 ? e[(k + 3) & 3] : e_last, r));
                }
                if (any(c.info)) body(g * gs + col + r * rs, c);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                last[r] = own[r][3];
                own[r] = next[r];
                info[r] = info_n[r];
                info_n[r] = info_nn[r];
            }
            e_last = e[3];
            e = e_next;
        }
    }
}

}  // namespace fsim
