// The fused step over plane tiles (kernels.h, LatGeom): the same cell
// arithmetic as fused.h's k_fused, with the addresses of that layout.
// Included by fused_f64.hip and fused_lp.hip.
//
// A workgroup never spans two z planes, so the three planes a cell reads from
// are the same for all its lanes: a population's address is a scalar base
// (plane, population) plus one of nine 32-bit offsets per lane (the cells
// (y + b, x + a) of a plane), against 27 offsets over the structure of arrays.
// What bounds it is HBM; TGV 512^3 and others before and after: see k_tiled.
#pragma once

#include "fused.h"

namespace imx {

struct TileCtx {
    CellCtx k;         // what cell_collide and the boundary rules read
    uint32_t o[3][3];  // byte offsets within a plane, population 0: [y + b - 1][x + a - 1]
};

// (wrapped or clamped as cell_setup does; a clamped value is never used as a
// source)
template <typename S, int BC>
__device__ __forceinline__ void tile_setup(const FusedParams &P, uint32_t z, uint32_t p, TileCtx &t)
{
    const uint32_t nx = P.nx, ny = P.ny, plane = nx * ny;
    CellCtx &k = t.k;
    k.live = p < plane;
    if (!k.live) p = 0;  // loads and collides a cell like the others, stores nothing
    const uint32_t y = P.divx.div(p), x = p - y * nx;
    k.c = z * plane + p;
    k.m = 0;
    if constexpr (BC == BC_CHANNEL) {
        if (k.live) {
            k.m = *glb(P.mask + k.c);
            if (k.m == 1) k.live = false;  // solid: nothing streams from or to it
        }
    }
    constexpr bool XW = BC == BC_PERIODIC, YW = BC == BC_PERIODIC || BC == BC_CHANNEL;
    k.x0 = x == 0;
    k.x1 = x == nx - 1;
    k.y0 = y == 0;
    k.y1 = y == ny - 1;
    k.z0 = z == 0;
    k.z1 = z == (uint32_t)P.nz - 1;
    k.xv[0] = k.x0 ? (XW ? nx - 1 : 0) : x - 1;
    k.xv[1] = x;
    k.xv[2] = k.x1 ? (XW ? 0 : nx - 1) : x + 1;
    const uint32_t yv[3] = {k.y0 ? (YW ? ny - 1 : 0) : y - 1, y, k.y1 ? (YW ? 0 : ny - 1) : y + 1};
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const uint32_t q = yv[b] * nx + k.xv[a];
            t.o[b][a] = (__umul24(q >> P.geom.tl, P.geom.ts) + q) * (uint32_t)sizeof(S);
        }
    if constexpr (BC == BC_FAITHFUL) {
        k.z = z;
        k.y = y;
        k.rx0 = (z + 1) * (ny + 2) + y + 1;
        k.ry0 = (z + 1) * nx + x;
        k.rz0 = y * nx + x;
    }
}

// The place of population i in a tile (LatGeom::pos).
template <int PAT>
__device__ __forceinline__ constexpr int tile_slot(int i)
{
    return PAT == PAT_PULL ? i : EZ_POS.v[i];
}

// Population i of a plane at byte offset `o`: the plane's first element
// is the same for all lanes, the population's place is added to the 32-bit
// offset.
template <int PAT, typename S>
__device__ __forceinline__ S *tile_ptr(S *plane, const FusedParams &P, int i, uint32_t o)
{
    const int slot = tile_slot<PAT>(i);
    using B = typename std::conditional<std::is_const<S>::value, const char, char>::type;
    return (S *)((B *)plane + (uint32_t)(o + (uint32_t)slot * (uint32_t)(P.geom.is * sizeof(S))));
}

// A pointer that is the same for all lanes, through readfirstlane: opaque to
// the compiler, which otherwise adds it to the lanes' offsets in 64 bits.
template <typename S>
__device__ __forceinline__ S *uniform_ptr(S *p)
{
    const uint64_t a = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return (S *)(((uint64_t)hi << 32) | lo);
}

// The planes z - 1, z, z + 1 (wrapped or clamped).
template <typename S, int BC>
__device__ __forceinline__ void tile_planes(S *lat, const FusedParams &P, uint32_t z, S *(&pl)[3])
{
    constexpr bool ZW = BC == BC_PERIODIC || BC == BC_CHANNEL;
    const uint32_t nz = P.nz;
    const uint32_t zm = z == 0 ? (ZW ? nz - 1 : 0) : z - 1, zp = z == nz - 1 ? (ZW ? 0 : nz - 1) : z + 1;
    pl[0] = uniform_ptr(lat + (uint64_t)zm * P.geom.zs);
    pl[1] = uniform_ptr(lat + (uint64_t)z * P.geom.zs);
    pl[2] = uniform_ptr(lat + (uint64_t)zp * P.geom.zs);
}

// The 27 populations arriving at the cell (cell_gather's rules).  CLEAR: no
// lane of the wavefront is beside the channel's ball.
template <typename S, int BC, int PAT, bool NT, bool CLEAR = true>
__device__ __forceinline__ void tile_gather(const FusedParams &P, const TileCtx &t, const S *const (&pl)[3],
                                            typename RealOf<S>::type (&f)[Q])
{
    using R = typename RealOf<S>::type;
    constexpr bool F64 = std::is_same<S, double>::value;
    const CellCtx &k = t.k;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        if constexpr (PAT == PAT_AA_EVEN) {
            f[i] = ld_ptr<S, NT>(tile_ptr<PAT>(pl[1], P, i, t.o[1][1]), WCLASS[i]);
            if constexpr (BC == BC_CAVITY) {
                if (EZ[i] < 0) {
                    R lid;
                    if constexpr (F64) lid = f[i] + P.corr[i];
                    else lid = f[i] + (float)P.corr[i];
                    f[i] = k.z1 ? lid : f[i];
                }
            }
        } else {
            const int s = PAT == PAT_PULL ? i : BB[i];
            const S *const from = pl[1 - EZ[i]];
            const uint32_t o = t.o[1 - EY[i]][1 - EX[i]];
            // lines that no other wavefront reads are not kept
            const bool nt = NT && EX[i] == 0;
            if constexpr (BC == BC_PERIODIC) {
                const S *p = tile_ptr<PAT>(from, P, s, o);
                f[i] = nt ? ld_ptr<S, true>(p, WCLASS[i]) : ld_ptr<S, false>(p, WCLASS[i]);
            } else if constexpr (BC == BC_CAVITY) {
                // One base (the plane below), two offsets: where x - e_i is
                // outside, the cell's own population bb(i) (pull) or i (AA)
                const bool out = src_out(k, i);
                const uint32_t zb = (uint32_t)((pl[1] - pl[0]) * (int64_t)sizeof(S));
                const uint32_t is = (uint32_t)(P.geom.is * sizeof(S));
                const uint32_t in = (uint32_t)((from - pl[0]) * (int64_t)sizeof(S)) + (uint32_t)tile_slot<PAT>(s) * is + o;
                const uint32_t own = zb + (uint32_t)tile_slot<PAT>(BB[s]) * is + t.o[1][1];
                const S *p = (const S *)((const char *)pl[0] + (out ? own : in));
                R v = nt ? ld_ptr<S, true>(p, WCLASS[i]) : ld_ptr<S, false>(p, WCLASS[i]);
                if (EZ[i] < 0) {
                    R lid;
                    if constexpr (F64) lid = v + P.corr[i];
                    else lid = v + (float)P.corr[i];
                    v = k.z1 ? lid : v;
                }
                f[i] = v;
            } else if constexpr (BC == BC_FAITHFUL) {
                const bool ox = (EX[i] > 0 && k.x0) || (EX[i] < 0 && k.x1);
                const bool oy = (EY[i] > 0 && k.y0) || (EY[i] < 0 && k.y1);
                const bool oz = (EZ[i] > 0 && k.z0) || (EZ[i] < 0 && k.z1);
                const uint32_t nx = P.nx, ny = P.ny;
                const uint32_t rxi = (EX[i] < 0 ? P.ring_a : 0u) + k.rx0 - EZ[i] * (ny + 2) - EY[i];
                const uint32_t ryi = 2 * P.ring_a + (EY[i] < 0 ? P.ring_b : 0u) + k.ry0 - EZ[i] * nx - EX[i];
                const uint32_t rzi =
                    2 * (P.ring_a + P.ring_b) + (EZ[i] < 0 ? P.ring_c : 0u) + k.rz0 - EY[i] * nx - EX[i];
                const uint32_t r = ox ? rxi : (oy ? ryi : rzi);
                const S *p = tile_ptr<PAT>(from, P, s, o);
                if (i != 0) {
                    const S *g = (const S *)P.ring + (uint64_t)i * P.ring_n + r;
                    p = ox || oy || oz ? g : p;
                }
                f[i] = nt ? ld_ptr<S, true>(p, WCLASS[i]) : ld_ptr<S, false>(p, WCLASS[i]);
            } else {  // channel, pull only
                bool solid = false;
                const S *p = tile_ptr<PAT>(from, P, s, o);
                if constexpr (!CLEAR) {
                    if (i != 0 && k.m == 2) {
                        const uint32_t nz = P.nz, z = P.divy.div(P.divx.div(k.c));
                        const uint32_t zs = EZ[i] > 0 ? (z == 0 ? nz - 1 : z - 1) : EZ[i] < 0 ? (z == nz - 1 ? 0 : z + 1) : z;
                        const uint32_t y = P.divx.div(k.c) - z * P.ny;
                        const uint32_t ys = EY[i] > 0   ? (y == 0 ? P.ny - 1 : y - 1)
                                            : EY[i] < 0 ? (y == (uint32_t)P.ny - 1 ? 0 : y + 1)
                                                        : y;
                        solid = *glb(P.mask + ((uint64_t)zs * P.ny + ys) * P.nx + k.xv[1 - EX[i]]) == 1;
                    }
                    const S *own = tile_ptr<PAT>(pl[1], P, BB[i], t.o[1][1]);
                    p = solid ? own : p;
                }
                R v = ld_ptr<S, false>(p, WCLASS[i]);
                if constexpr (!F64 && !CLEAR) {
                    // shifted storage: see cell_gather
                    if (EX[i] != 0) v = solid ? ball_link<S>(P, i, v) : v;
                }
                if (EX[i] > 0) {
                    R in;
                    if constexpr (F64) in = P.feq_in[i];
                    else in = (float)P.feq_in[i];
                    v = k.x0 ? in : v;
                }
                f[i] = v;
            }
        }
    }
}

template <typename S, int BC, int PAT, bool NT>
__device__ __forceinline__ void tile_scatter(const FusedParams &P, const TileCtx &t, S *const (&pl)[3],
                                             const typename RealOf<S>::type (&f)[Q])
{
    const CellCtx &k = t.k;
    // The AA pattern stores to the addresses it loaded from.  Behind an empty
    // asm the offsets are new to the compiler, which would otherwise hold the
    // loads' 27 addresses, as 64-bit pairs, across the collision (FP64 even
    // step 146 instead of 120 registers).
    uint32_t o9[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            o9[b][a] = t.o[b][a];
            if (PAT == PAT_AA_ODD || (a == 1 && b == 1)) asm("" : "+v"(o9[b][a]));
        }
    if constexpr (PAT == PAT_PULL || PAT == PAT_AA_EVEN) {
        if constexpr (BC == BC_FAITHFUL) stage_rows(P, k, f);
#pragma unroll
        for (int i = 0; i < Q; ++i)
            st_ptr<S, NT>(tile_ptr<PAT>(pl[1], P, PAT == PAT_PULL ? i : BB[i], o9[1][1]), WCLASS[i], f[i]);
    } else {
        // to slot i of x + e_i, or bounced back into slot bb(i) at x
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            S *const to = pl[1 + EZ[i]];
            const uint32_t o = o9[1 + EY[i]][1 + EX[i]];
            S *p;
            if constexpr (BC == BC_CAVITY) {
                const uint32_t zb = (uint32_t)((pl[1] - pl[0]) * (int64_t)sizeof(S));
                const uint32_t is = (uint32_t)(P.geom.is * sizeof(S));
                const uint32_t in = (uint32_t)((to - pl[0]) * (int64_t)sizeof(S)) + (uint32_t)tile_slot<PAT>(i) * is + o;
                const uint32_t own = zb + (uint32_t)tile_slot<PAT>(BB[i]) * is + o9[1][1];
                p = (S *)((char *)pl[0] + (src_out(k, BB[i]) ? own : in));
            } else {
                p = tile_ptr<PAT>(to, P, i, o);
            }
            st_ptr<S, NT>(p, WCLASS[i], f[i]);
        }
    }
}

// Collision and stores of a gathered cell.  In FP64 a wavefront whose populations
// all allow it divides through reciprocals (fused.h div_by), with the same bits:
// 677 vector operations for a cell instead of 1055, us per step before /
// after: cavity 128^3 AA 146.7 / 136.0, TGV 96^3 AA 63.6 / 59.2, 64^3 AA 21.4 / 20.0, 32^3 pull
// 5.8 / 5.2, 256^3 pull 1211 / 1202 (HBM).
template <typename S, int BC, int PAT, bool NT>
__device__ __forceinline__ void tile_finish(const FusedParams &P, const TileCtx &t, S *const (&dst)[3],
                                            typename RealOf<S>::type (&f)[Q])
{
    if constexpr (std::is_same<S, double>::value) {
        if (P.inv_den == 0.0 || wave_any(!div_safe(f))) {
            cell_collide_f64<BC, false>(P, t.k, f, P.mom_p != nullptr);
            if (t.k.live) tile_scatter<S, BC, PAT, NT>(P, t, dst, f);
        } else {
            cell_collide_f64<BC, true>(P, t.k, f, P.mom_p != nullptr);
            if (t.k.live) tile_scatter<S, BC, PAT, NT>(P, t, dst, f);
        }
    } else {
        cell_collide<S, BC>(P, t.k, f, P.mom_p != nullptr);
        if (t.k.live) tile_scatter<S, BC, PAT, NT>(P, t, dst, f);
    }
}

// XCD-aware order of the workgroups over plane tiles (FusedParams::xcd_remap):
// 1: one contiguous run of the lattice per XCD, which finds the lines it wrote
// in the step before in its own L2 or, further out, still in the last-level
// cache; XCD_RUNS: runs of eight consecutive workgroups per XCD, the eight
// XCDs' runs side by side, so that the lines which the x-shifted rows of
// neighbouring workgroups share mostly stay in one L2 while the chip sweeps one
// window of the lattice.  tile_order chooses.  us per step, linear / one run /
// runs of 8, block 256: pull TGV 256^3 FP64 1292 / 1218 / 1209, FP32 605 / 621 / 603, FP16
// 310 / 310 / 297, 301x203x157 FP32 337 / 367 / 342, channel 512x256x256 FP16 640 / 702 /
// 637; in the last-level cache, with plain stores, 80^3 FP64 36.2 / 33.8 / 35.1, 96^3
// FP32 31.0 / 28.5 / 29.5, 48^3 FP32 9.9 / 5.4 / 8.2, 112^3 FP16 28.5 / 23.7 / 25.3; AA TGV
// 160^3 FP32 145 / 144 / 139, 128^3 66.0 / 64.1 / 65.3, 96^3 FP64 59.1 / 56.2 / 57.7, 48^3 11.9 / 8.4 /
// 10.9, 80^3 FP16 12.0 / 9.4 / 11.1.
__device__ __forceinline__ uint32_t tile_block_of(int order, uint32_t b, uint32_t nb)
{
    constexpr uint32_t RUN = 8, ALL = 8 * RUN;
    if (order == 1) return xcd_tile(b, nb);
    const uint32_t g = b / ALL, r = b % ALL;
    return order == XCD_RUNS && (g + 1) * ALL <= nb ? g * ALL + (r & 7u) * RUN + (r >> 3) : b;
}

// CPT cells per thread, blockDim.x apart, of plane z from cell p0; the loads of
// all are issued before any of them is collided.
template <typename S, int BC, int PAT, int CPT, bool NT>
__device__ __forceinline__ void tile_cells(const FusedParams &P, uint32_t z, uint32_t p0)
{
    using R = typename RealOf<S>::type;
    const S *src[3];
    S *dst[3];
    tile_planes<const S, BC>((const S *)P.src, P, z, src);
    tile_planes<S, BC>((S *)P.dst, P, z, dst);
    TileCtx t[CPT];
    R f[CPT][Q];
    bool near = false;
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
        tile_setup<S, BC>(P, z, p0 + (uint32_t)r * blockDim.x, t[r]);
        near |= BC == BC_CHANNEL && t[r].k.m == 2;
    }
    // Lanes beyond the plane and solid cells load and collide a cell like the
    // others and store nothing: a branch around it all would make the choices
    // below divergent regions, whose values the compiler holds twice.
    // Only wavefronts with a cell beside the channel's ball look at their
    // neighbours' mask and choose between two addresses.
    if (BC == BC_CHANNEL && wave_any(near)) {
#pragma unroll
        for (int r = 0; r < CPT; ++r) {
            tile_gather<S, BC, PAT, NT, false>(P, t[r], src, f[r]);
            tile_finish<S, BC, PAT, NT>(P, t[r], dst, f[r]);
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < CPT; ++r) tile_gather<S, BC, PAT, NT>(P, t[r], src, f[r]);
#pragma unroll
    for (int r = 0; r < CPT; ++r) tile_finish<S, BC, PAT, NT>(P, t[r], dst, f[r]);
}

// Before (structure of arrays, k_fused) and after, us per step, first
// allocations: TGV 256^3 FP64 pull 1342 -> 1202 (6.03 TB/s algorithmic), 301x203x157
// FP32 pull 414 -> 340, channel 512x256x256 FP16 712 -> 603, the reference's sphere
// 512x128x128 715 -> 627 with its boundary launch, cavity 128^3 FP64 AA 153 -> 136, TGV 64^3
// FP64 AA 21.0 -> 18.9.  NT: kernels.h tile_nt.
template <typename S, int BC, int PAT, int CPT, bool NT>
__global__ void __launch_bounds__(512) k_tiled(const FusedParams P)
{
    const uint32_t b = tile_block_of(P.xcd_remap, blockIdx.x, P.nblocks);
    const uint32_t z = P.divb.div(b);
    tile_cells<S, BC, PAT, CPT, NT>(P, z, (b - z * P.bpp) * blockDim.x * CPT + threadIdx.x);
}

// The value of the lane before (EXP 1) or after (EXP -1); the first (last)
// lane takes `edge`.
template <int EXP>
__device__ __forceinline__ float lane_shift(float v, float edge)
{
    constexpr int CTRL = EXP > 0 ? 0x138 : 0x130;  // wave_shr:1, wave_shl:1
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v),
                                                                 CTRL, 0xf, 0xf, false));
}
template <int EXP>
__device__ __forceinline__ double lane_shift(double v, double edge)
{
    constexpr int CTRL = EXP > 0 ? 0x138 : 0x130;
    const uint64_t a = __builtin_bit_cast(uint64_t, v), e = __builtin_bit_cast(uint64_t, edge);
    const uint32_t lo = __builtin_amdgcn_update_dpp((int)(uint32_t)e, (int)(uint32_t)a, CTRL, 0xf, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp((int)(uint32_t)(e >> 32), (int)(uint32_t)(a >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The AA odd step on rows that are whole wavefronts (nx a multiple of 64, at
// most 512): a workgroup is one or more whole rows, every population moves in
// x-aligned lines, and what crosses into a neighbouring cell in x crosses
// between lanes (DPP; LDS between wavefronts) instead of through shifted lines.  The shifted form loads a line twice and
// stores it in two parts, through L2: 5.2 TB/s against 5.9-6.1 for this
// pattern without arithmetic (TGV 512^3, FP64).  As every row is one
// wavefront's, its addresses are scalars and one lane offset serves all 27.
// NT is the loads': stores are non-temporal in both forms (with plain loads too they are
// faster, us per AA step, non-temporal / plain stores: 512^3 FP64 10490 / 10600, 448x256x256 FP64
// 2338 / 2343, FP32 1207 / 1200, 512x512x256 FP16 1267 / 1272; non-temporal loads 9590, 2107,
// 1077, 1161).
template <typename R>
struct RowEdges {
    // [wavefront][0: its last lane, e_x = 1; 1: its first lane, e_x = -1][XDIR_P / XDIR_M rank]
    R v[8][2][10];
};

template <typename S, int BC, bool NT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) k_tiled_rows(const FusedParams P)
{
    using R = typename RealOf<S>::type;
    constexpr bool F64 = std::is_same<S, double>::value;
    constexpr bool WALLS = BC == BC_CAVITY;
    __shared__ RowEdges<R> in, out;
    const uint32_t b = tile_block_of(P.xcd_remap, blockIdx.x, P.nblocks);
    const uint32_t nx = P.nx, ny = P.ny, nz = P.nz, plane = nx * ny;
    const uint32_t z = P.divb.div(b), lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), per_row = nx >> 6;
    const uint32_t row = wave / per_row, seg = wave - row * per_row;
    const uint32_t y0 = (b - z * P.bpp) * (blockDim.x / nx) + row;
    // a last workgroup's rows beyond the plane work on the last row and store
    // nothing
    const bool live = y0 < ny;
    const uint32_t y = live ? y0 : ny - 1, x = seg * 64u + lane;
    const uint32_t first = row * per_row;
    const uint32_t prev = seg == 0 ? first + per_row - 1 : wave - 1, next = seg + 1 == per_row ? first : wave + 1;

    const uint32_t zv[3] = {z == 0 ? (WALLS ? 0 : nz - 1) : z - 1, z, z == nz - 1 ? (WALLS ? z : 0) : z + 1};
    const uint32_t yv[3] = {y == 0 ? (WALLS ? 0 : ny - 1) : y - 1, y, y == ny - 1 ? (WALLS ? y : 0) : y + 1};
    const bool zo[3] = {WALLS && z == 0, false, WALLS && z == nz - 1};
    const bool yo[3] = {WALLS && y == 0, false, WALLS && y == ny - 1};
    S *const lat = (S *)P.dst;
    S *seg_of[3][3];  // this wavefront's cells in rows (z + a - 1, y + b - 1), population 0
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) seg_of[a][c] = uniform_ptr(lat + P.geom.off(0, zv[a], yv[c] * nx + seg * 64u));
    // population `slot` of lane `l` of row (z + a - 1, y + c - 1)
    auto at = [&](int a, int c, int slot, uint32_t l) {
        return (S *)((char *)seg_of[a][c] + (uint32_t)(l * (uint32_t)sizeof(S) + (uint32_t)tile_slot<PAT_AA_ODD>(slot) * (uint32_t)(P.geom.is * sizeof(S))));
    };

    R f[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        // from slot bb(i) of x - e_i; where that row lies outside the cavity,
        // the cell's own slot i, not shifted
        const bool o = zo[1 - EZ[i]] || yo[1 - EY[i]];
        f[i] = ld_ptr<S, NT>(o ? at(1, 1, i, lane) : at(1 - EZ[i], 1 - EY[i], BB[i], lane), WCLASS[i]);
    }
    // cells at an x wall take their own slot i
    R wall[9];
    const bool xw_lo = WALLS && seg == 0, xw_hi = WALLS && seg + 1 == per_row;
    R wall2[9];
    if (xw_lo) {
#pragma unroll
        for (int r = 0; r < 9; ++r) wall[r] = ld_ptr<S>(at(1, 1, XDIR_P[r], 0), WCLASS[XDIR_P[r]]);
    }
    if (xw_hi) {
#pragma unroll
        for (int r = 0; r < 9; ++r) wall2[r] = ld_ptr<S>(at(1, 1, XDIR_M[r], 63), WCLASS[XDIR_M[r]]);
    }
    auto exchange = [&](RowEdges<R> &e, bool gather) {
        if (lane == 0 || lane == 63) {
#pragma unroll
            for (int r = 0; r < 9; ++r) e.v[wave][lane == 0][r] = lane == 0 ? f[XDIR_M[r]] : f[XDIR_P[r]];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int p = XDIR_P[r], m = XDIR_M[r];
            R ep = e.v[prev][0][r], em = e.v[next][1][r];
            if (gather && xw_lo) ep = wall[r];
            if (gather && xw_hi) em = wall2[r];
            const R sp = lane_shift<1>(f[p], ep), sm = lane_shift<-1>(f[m], em);
            if constexpr (WALLS) {
                const bool op = gather ? zo[1 - EZ[p]] || yo[1 - EY[p]] : zo[1 + EZ[p]] || yo[1 + EY[p]];
                const bool om = gather ? zo[1 - EZ[m]] || yo[1 - EY[m]] : zo[1 + EZ[m]] || yo[1 + EY[m]];
                f[p] = op ? f[p] : sp;
                f[m] = om ? f[m] : sm;
            } else {
                f[p] = sp;
                f[m] = sm;
            }
        }
    };
    exchange(in, true);
    // FP64: 127 registers (four wavefronts per SIMD) instead of 129
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (WALLS) {
#pragma unroll
        for (int i = 0; i < Q; ++i)
            if (EZ[i] < 0) {
                R lid;
                if constexpr (F64) lid = f[i] + P.corr[i];
                else lid = f[i] + (float)P.corr[i];
                f[i] = z == nz - 1 ? lid : f[i];
            }
    }

    CellCtx k;
    k.c = z * plane + y * nx + x;
    k.live = live;
    // FP64 keeps the IEEE division: the choice of tile_finish takes 12 registers
    // more than four wavefronts per SIMD leave, and these lattices wait for HBM
    cell_collide<S, BC>(P, k, f, P.mom_p != nullptr);

    if constexpr (WALLS) {
        // what leaves through an x wall comes back into slot bb(i) of the cell
        if (live && xw_hi && lane == 63) {
#pragma unroll
            for (int r = 0; r < 9; ++r) st_ptr<S, false>(at(1, 1, XDIR_M[r], lane), WCLASS[XDIR_M[r]], f[BB[XDIR_M[r]]]);
        }
        if (live && xw_lo && lane == 0) {
#pragma unroll
            for (int r = 0; r < 9; ++r) st_ptr<S, false>(at(1, 1, XDIR_P[r], lane), WCLASS[XDIR_P[r]], f[BB[XDIR_P[r]]]);
        }
    }
    exchange(out, false);
    if (!live) return;
    uint32_t to = lane;  // see tile_scatter
    asm("" : "+v"(to));
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        // to slot i of x + e_i, or back into the cell's own slot bb(i)
        const bool o = zo[1 + EZ[i]] || yo[1 + EY[i]];
        S *const p = o ? at(1, 1, BB[i], to) : at(1 + EZ[i], 1 + EY[i], i, to);
        if constexpr (WALLS) {
            // nothing arrives at an x wall from beyond it
            if (EX[i] > 0 && xw_lo && !o && lane == 0) continue;
            if (EX[i] < 0 && xw_hi && !o && lane == 63) continue;
        }
        st_ptr<S, true>(p, WCLASS[i], f[i]);
    }
}

template <typename S, int CPT, bool NT>
hipError_t launch_tiled_cpt(int bc, int pattern, const FusedParams &P, int block, hipStream_t st)
{
    dim3 grid(P.nblocks), blk(block);
#define IMX_L(B, PT) hipLaunchKernelGGL((k_tiled<S, B, PT, CPT, NT>), grid, blk, 0, st, P)
    if (bc == BC_PERIODIC) {
        if (pattern == PAT_PULL) IMX_L(BC_PERIODIC, PAT_PULL);
        else if (pattern == PAT_AA_EVEN) IMX_L(BC_PERIODIC, PAT_AA_EVEN);
        else IMX_L(BC_PERIODIC, PAT_AA_ODD);
    } else if (bc == BC_CAVITY) {
        if (pattern == PAT_PULL) IMX_L(BC_CAVITY, PAT_PULL);
        else if (pattern == PAT_AA_EVEN) IMX_L(BC_CAVITY, PAT_AA_EVEN);
        else IMX_L(BC_CAVITY, PAT_AA_ODD);
    } else if (pattern != PAT_PULL) {
        return hipErrorInvalidValue;
    } else if (bc == BC_CHANNEL) {
        IMX_L(BC_CHANNEL, PAT_PULL);
    } else if constexpr (std::is_same<S, double>::value) {
        IMX_L(BC_FAITHFUL, PAT_PULL);
    } else {
        return hipErrorInvalidValue;
    }
#undef IMX_L
    return hipGetLastError();
}

template <typename S>
hipError_t launch_tiled(int bc, int pattern, const FusedParams &P0, int block, hipStream_t st)
{
    FusedParams P = P0;
    const uint64_t bytes = lattice_elems(P.geom, (uint32_t)P.nz) * sizeof(S);
    const uint32_t plane = (uint32_t)P.nx * (uint32_t)P.ny;
    block = tile_block_in_effect(plane, block);
    P.xcd_remap = P.xcd_remap ? tile_order(bytes, pattern != PAT_PULL) : 0;
    const uint32_t rows = tile_rows(P.nx, block, bytes, bc, sizeof(S));
    if (pattern == PAT_AA_ODD && rows > 0) {
        P.bpp = ((uint32_t)P.ny + rows - 1) / rows;
        P.divb.init(P.bpp);
        P.nblocks = P.bpp * (uint32_t)P.nz;
        const dim3 grid(P.nblocks), blk(rows * (uint32_t)P.nx);
#define IMX_L(B)                                                                                  \
    do {                                                                                          \
        if (P.ntl) hipLaunchKernelGGL((k_tiled_rows<S, B, true>), grid, blk, 0, st, P);           \
        else hipLaunchKernelGGL((k_tiled_rows<S, B, false>), grid, blk, 0, st, P);                \
    } while (0)
        if (bc == BC_PERIODIC) IMX_L(BC_PERIODIC);
        else if (bc == BC_CAVITY) IMX_L(BC_CAVITY);
        else return hipErrorInvalidValue;
#undef IMX_L
        return hipGetLastError();
    }
    const int cpt = P.cpt == 2 ? 2 : 1;
    const uint32_t per = (uint32_t)block * (uint32_t)cpt;
    P.bpp = (plane + per - 1) / per;
    P.divb.init(P.bpp);
    P.nblocks = P.bpp * (uint32_t)P.nz;
    if (cpt == 2) return P.ntl ? launch_tiled_cpt<S, 2, true>(bc, pattern, P, block, st)
                               : launch_tiled_cpt<S, 2, false>(bc, pattern, P, block, st);
    return P.ntl ? launch_tiled_cpt<S, 1, true>(bc, pattern, P, block, st)
                 : launch_tiled_cpt<S, 1, false>(bc, pattern, P, block, st);
}

}  // namespace imx
