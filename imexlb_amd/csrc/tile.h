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

#ifndef IMX_TILE_ODD_NT
#define IMX_TILE_ODD_NT 1
#endif
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
    if (!k.live) p = 0;  // keep the arithmetic in range; nothing is loaded
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

// Population `slot` of a plane at byte offset `o`: the plane's first element
// is the same for all lanes, the population's place is added to the 32-bit
// offset.
template <typename S>
__device__ __forceinline__ S *tile_ptr(S *plane, const FusedParams &P, int slot, uint32_t o)
{
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
template <typename S, int BC, int PAT, bool NTL, bool CLEAR = true>
__device__ __forceinline__ void tile_gather(const FusedParams &P, const TileCtx &t, const S *const (&pl)[3],
                                            typename RealOf<S>::type (&f)[Q])
{
    using R = typename RealOf<S>::type;
    constexpr bool F64 = std::is_same<S, double>::value;
    const CellCtx &k = t.k;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        if constexpr (PAT == PAT_AA_EVEN) {
            f[i] = ld_ptr<S, NTL>(tile_ptr(pl[1], P, i, t.o[1][1]), WCLASS[i]);
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
            const bool nt = NTL && EX[i] == 0;
            if constexpr (BC == BC_PERIODIC) {
                const S *p = tile_ptr(from, P, s, o);
                f[i] = nt ? ld_ptr<S, true>(p, WCLASS[i]) : ld_ptr<S, false>(p, WCLASS[i]);
            } else if constexpr (BC == BC_CAVITY) {
                // One base (the plane below), two offsets: where x - e_i is
                // outside, the cell's own population bb(i) (pull) or i (AA)
                const bool out = src_out(k, i);
                const uint32_t zb = (uint32_t)((pl[1] - pl[0]) * (int64_t)sizeof(S));
                const uint32_t is = (uint32_t)(P.geom.is * sizeof(S));
                const uint32_t in = (uint32_t)((from - pl[0]) * (int64_t)sizeof(S)) + (uint32_t)s * is + o;
                const uint32_t own = zb + (uint32_t)BB[s] * is + t.o[1][1];
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
                const S *p = tile_ptr(from, P, s, o);
                if (i != 0) {
                    const S *g = (const S *)P.ring + (uint64_t)i * P.ring_n + r;
                    p = ox || oy || oz ? g : p;
                }
                f[i] = nt ? ld_ptr<S, true>(p, WCLASS[i]) : ld_ptr<S, false>(p, WCLASS[i]);
            } else {  // channel, pull only
                bool solid = false;
                const S *p = tile_ptr(from, P, s, o);
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
                    const S *own = tile_ptr(pl[1], P, BB[i], t.o[1][1]);
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

template <typename S, int BC, int PAT>
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
            st_ptr<S>(tile_ptr(pl[1], P, PAT == PAT_PULL ? i : BB[i], o9[1][1]), WCLASS[i], f[i]);
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
                const uint32_t in = (uint32_t)((to - pl[0]) * (int64_t)sizeof(S)) + (uint32_t)i * is + o;
                const uint32_t own = zb + (uint32_t)BB[i] * is + o9[1][1];
                p = (S *)((char *)pl[0] + (src_out(k, BB[i]) ? own : in));
            } else {
                p = tile_ptr(to, P, i, o);
            }
            if (IMX_TILE_ODD_NT || EX[i] == 0) st_ptr<S, true>(p, WCLASS[i], f[i]);
            else st_ptr<S, false>(p, WCLASS[i], f[i]);
        }
    }
}

// XCD-aware order of the workgroups over plane tiles: runs of eight consecutive
// workgroups per XCD, the eight XCDs' runs side by side.  The lines that the
// x-shifted rows of neighbouring workgroups share then mostly stay in one L2
// while the chip sweeps one window of the lattice.  Step times in us, linear
// / one run per XCD / runs of 8, block 256 (pull unless said): TGV 256^3 FP64 1292 /
// 1218 / 1209, FP32 605 / 621 / 603, FP16 310 / 310 / 297, 301x203x157 FP32 337 / 367 / 342,
// channel 512x256x256 FP16 640 / 702 / 637, cavity 128^3 FP64 AA 149.6 / 149.6 / 146.0.
__device__ __forceinline__ uint32_t xcd_run(uint32_t b, uint32_t nb)
{
    constexpr uint32_t RUN = 8, ALL = 8 * RUN;
    const uint32_t g = b / ALL, r = b % ALL;
    return (g + 1) * ALL <= nb ? g * ALL + (r & 7u) * RUN + (r >> 3) : b;
}

// Before (structure of arrays, k_fused) and after, us per step, first
// allocations: TGV 256^3 FP64 pull 1342 -> 1209 (5.99 TB/s algorithmic), 301x203x157
// FP32 pull 414 -> 342, channel 512x256x256 FP16 712 -> 637, the reference's sphere
// 512x128x128 715 -> 642 with its boundary kernels, cavity 128^3 FP64 AA 153 -> 146.
template <typename S, int BC, int PAT, int CPT, bool NTL>
__global__ void __launch_bounds__(512) k_tiled(const FusedParams P)
{
    using R = typename RealOf<S>::type;
    uint32_t b = blockIdx.x;
    if (P.xcd_remap) b = xcd_run(b, P.nblocks);
    const uint32_t z = P.divb.div(b);
    const uint32_t p0 = (b - z * P.bpp) * blockDim.x * CPT + threadIdx.x;
    const S *src[3];
    S *dst[3];
    tile_planes<const S, BC>((const S *)P.src, P, z, src);
    tile_planes<S, BC>((S *)P.dst, P, z, dst);
    TileCtx t[CPT];
    R f[CPT][Q];
    if constexpr (BC == BC_CHANNEL) {
        // Only wavefronts with a cell beside the ball look at their
        // neighbours' mask and choose between two addresses.
        bool near = false;
#pragma unroll
        for (int r = 0; r < CPT; ++r) {
            tile_setup<S, BC>(P, z, p0 + (uint32_t)r * blockDim.x, t[r]);
            near |= t[r].k.m == 2;
        }
        if (wave_any(near)) {
#pragma unroll
            for (int r = 0; r < CPT; ++r) {
                if (!t[r].k.live) continue;
                tile_gather<S, BC, PAT, NTL, false>(P, t[r], src, f[r]);
                cell_collide<S, BC>(P, t[r].k, f[r], P.mom_p != nullptr);
                tile_scatter<S, BC, PAT>(P, t[r], dst, f[r]);
            }
            return;
        }
    }
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
        if constexpr (BC != BC_CHANNEL) tile_setup<S, BC>(P, z, p0 + (uint32_t)r * blockDim.x, t[r]);
        if (t[r].k.live) tile_gather<S, BC, PAT, NTL>(P, t[r], src, f[r]);
    }
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
        if (!t[r].k.live) continue;
        cell_collide<S, BC>(P, t[r].k, f[r], P.mom_p != nullptr);
        tile_scatter<S, BC, PAT>(P, t[r], dst, f[r]);
    }
}

template <typename S, int CPT, bool NTL>
hipError_t launch_tiled_cpt(int bc, int pattern, const FusedParams &P, int block, hipStream_t st)
{
    dim3 grid(P.nblocks), blk(block);
#define IMX_L(B, PT) hipLaunchKernelGGL((k_tiled<S, B, PT, CPT, NTL>), grid, blk, 0, st, P)
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
    const int cpt = P.cpt == 2 ? 2 : 1;
    const uint32_t plane = (uint32_t)P.nx * (uint32_t)P.ny, per = (uint32_t)block * (uint32_t)cpt;
    P.bpp = (plane + per - 1) / per;
    P.divb.init(P.bpp);
    P.nblocks = P.bpp * (uint32_t)P.nz;
    if (cpt == 2) return P.ntl ? launch_tiled_cpt<S, 2, true>(bc, pattern, P, block, st)
                               : launch_tiled_cpt<S, 2, false>(bc, pattern, P, block, st);
    return P.ntl ? launch_tiled_cpt<S, 1, true>(bc, pattern, P, block, st)
                 : launch_tiled_cpt<S, 1, false>(bc, pattern, P, block, st);
}

}  // namespace imx
