// Initialisation, population transfer, FP64 reductions and the copy kernel
// used to calibrate bandwidth.  Compiled with -ffp-contract=off: the initial
// state is the oracle's, bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fused.h"
#include "kernels.h"

namespace imx {

// feq in the reference's evaluation order (tgv/src/lbm.cpp:209-215).
__device__ __forceinline__ double feq_f64(int i, double p, double u, double v, double w)
{
    const double edu = edu_of<double>(i, u, v, w);
    const double udu = u * u + v * v + w * w;
    const double eu2 = edu * edu;
    return WVAL[WCLASS[i]] * p * 3.0 + WVAL[WCLASS[i]] * (3.0 * edu + 4.5 * eu2 - 1.5 * udu);
}

// Population f in the stored convention, g = f - s with s the direction's
// shift, of the weight class of slot `slot` (i or bb(i)).
template <typename S>
__device__ __forceinline__ S stored(int slot, double f, double s)
{
    if constexpr (std::is_same<S, double>::value)
        return f;
    else if constexpr (std::is_same<S, float>::value)
        return (float)(f - s);
    else
        return (_Float16)((float)(f - s) * H_SCALE[WCLASS[slot]]);
}

// The same into cell c of plane z.
template <typename S>
__device__ __forceinline__ void put(S *lat, const LatGeom &g, int slot, uint32_t z, uint32_t c, double f, double s)
{
    lat[g.off(g.pos(slot), z, c)] = stored<S>(slot, f, s);
}

template <typename S>
__device__ __forceinline__ double get(const S *lat, const LatGeom &g, int slot, uint32_t z, uint32_t c, double s)
{
    const S *p = lat + g.off(g.pos(slot), z, c);
    if constexpr (std::is_same<S, double>::value)
        return *p;
    else if constexpr (std::is_same<S, float>::value)
        return (double)*p + s;
    else
        return (double)((float)*p * H_INV_SCALE[WCLASS[slot]]) + s;
}

// Initial state = f0 = feq(p, u) of the analytic fields.  The reference's
// first Collision relaxes f0 towards the feq of the same fields, which is f0
// itself, so f0 is also the first post-collision state.
//
// Bound by its stores.  Over plane tiles workgroups stay within a plane, so that their
// lines are whole in a tile; over arrays they follow the cells (init_block).  Each XCD
// writes one run of the lattice.  us, the kernel over arrays in the cells' order / this:
// TGV 301x203x157 FP32 240 / 240, 256^3 FP64 735 / 690, 512^3 FP64 5840 / 5500, FP16 2400 / 2690,
// cavity 100^3 33 / 33, sphere 512x128x128 377 / 372, channel 512x256x256 FP16 537 / 665 (10 % more or
// less with the allocation).  The solid cells of the sphere's other lattice are written
// here rather than by a copy of the whole, another 770 in both.
template <typename S>
__global__ void k_init(const InitParams P)
{
    const uint32_t b = xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t plane = (uint32_t)P.nx * P.ny, first = P.divb.div(b) * plane;  // (0 over arrays)
    const uint32_t pc0 = (b - P.divb.div(b) * P.bpp) * blockDim.x + threadIdx.x;
    const uint32_t c = first + pc0;
    if (pc0 >= (P.geom.tl != 31 ? plane : P.ncell)) return;
    const uint32_t row = P.divx.div(c), z = P.divy.div(row);
    const uint32_t x = c - row * P.nx, y = row - z * P.ny, pc = c - z * plane;
    double u, v, w, p;
    if (P.kind == 0) {
        // tgv/src/lbm.cpp:197-204 with per-axis sin/cos tables
        const double *T = P.tab;
        const double sx = T[x], cx = T[P.nx + x], c2x = T[2 * P.nx + x];
        const double *Ty = T + 3 * P.nx;
        const double sy = Ty[y], cy = Ty[P.ny + y], c2y = Ty[2 * P.ny + y];
        const double *Tz = Ty + 3 * P.ny;
        const double cz = Tz[P.nz + z], c2z = Tz[2 * P.nz + z];
        u = P.u0 * sx * cy * cz;
        v = -P.u0 * cx * sy * cz;
        w = 0;
        p = P.rho0 * P.cs2 + P.rho0 * P.u0 * P.u0 / 16.0 * (c2x + c2y) * (c2z + 2.0);
    } else if (P.kind == 2) {
        // sphere/src/lbm.cpp:224-239: p = 0, a parabolic x velocity in z
        // masked by usr and perturbed by urand(100) (here the seeded hash of
        // the cell's index in the reference's ghost-3 layout)
        const uint64_t ly = (uint64_t)P.ny + 6, lz = (uint64_t)P.nz + 6;
        const uint64_t idx = ((uint64_t)(x + 3) * ly + (y + 3)) * lz + (z + 3);
        const int ran = (int)(mix64(P.seed + idx * 0x9E3779B97F4A7C15ULL) % 100ULL);
        const int usr = faithful_sphere_solid(P.nx, (int)x, (int)y, (int)z) ? 0 : 1;
        const int glz = P.nz, kz = (int)z;
        const double gm = (double)(glz - 1);
        u = (P.u0 * 4.0 * (double)kz * (double)(glz - 1 - kz) / (gm * gm)) * (double)usr * (1.0 + (double)ran * 0.001);
        v = 0.0;
        w = 0.0;
        p = 0.0;
    } else {
        const bool solid = P.mask && P.mask[c] == 1;
        u = solid ? 0.0 : P.u0;
        v = 0.0;
        w = 0.0;
        p = P.p0;
    }
    const bool solid = P.mask && P.mask[c] == 1;
    const uint64_t at = P.geom.off(0, z, pc);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        const uint64_t o = at + (uint64_t)P.geom.pos(P.layout == 1 ? BB[i] : i) * P.geom.is;
        const S f = stored<S>(i, feq_f64(i, p, u, v, w), P.sh[i]);
        ((S *)P.dst)[o] = f;
        if (solid && P.other) ((S *)P.other)[o] = f;
    }
    // the fields themselves are the moments of step 0, as the reference's
    // Initialize leaves them in p, ua, va, wa; a solid cell reports a fluid at
    // rest with p = 0, as every later step leaves it
    if (P.mom[0]) {
        P.mom[0][c] = solid ? 0.0 : p;
        P.mom[1][c] = u;
        P.mom[2][c] = v;
        P.mom[3][c] = w;
    }
}

hipError_t launch_init(int dtype, InitParams P, hipStream_t st)
{
    const uint32_t plane = (uint32_t)P.nx * P.ny, block = init_block(P.geom, plane);
    P.bpp = ((P.geom.tl != 31 ? plane : P.ncell) + block - 1) / block;
    P.divb.init(P.bpp);
    dim3 blk(block), grid(P.geom.tl != 31 ? P.bpp * (uint32_t)P.nz : P.bpp);
    if (dtype == DT_F64) hipLaunchKernelGGL(k_init<double>, grid, blk, 0, st, P);
    else if (dtype == DT_F32) hipLaunchKernelGGL(k_init<float>, grid, blk, 0, st, P);
    else hipLaunchKernelGGL(k_init<_Float16>, grid, blk, 0, st, P);
    return hipGetLastError();
}

// Lattice slot and cell (plane, cell of the plane) holding f*_i of cell
// (x, y, z) for each storage layout.
__device__ __forceinline__ void slot_of(const XferParams &P, int i, int x, int y, int z, int &slot, uint32_t &plane,
                                        uint32_t &cell)
{
    const uint32_t nx = P.nx, ny = P.ny, nz = P.nz;
    slot = P.layout == 1 ? BB[i] : i;
    plane = (uint32_t)z;
    cell = (uint32_t)y * nx + (uint32_t)x;
    if (P.layout < 2) return;
    // streamed (AA after an odd step): f*_i(x) sits at x + e_i in slot i, or
    // at x in slot bb(i) when x + e_i is a cavity wall
    int xd = x + EX[i], yd = y + EY[i], zd = z + EZ[i];
    if (P.bc == BC_CAVITY) {
        if (xd < 0 || xd >= (int)nx || yd < 0 || yd >= (int)ny || zd < 0 || zd >= (int)nz) {
            slot = BB[i];
            return;
        }
    } else {
        xd = xd < 0 ? xd + (int)nx : (xd >= (int)nx ? xd - (int)nx : xd);
        yd = yd < 0 ? yd + (int)ny : (yd >= (int)ny ? yd - (int)ny : yd);
        zd = zd < 0 ? zd + (int)nz : (zd >= (int)nz ? zd - (int)nz : zd);
    }
    plane = (uint32_t)zd;
    cell = (uint32_t)yd * nx + (uint32_t)xd;
}

template <typename S>
__global__ void k_get_f(const XferParams P)
{
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= P.ncell) return;
    const uint32_t t = P.divx.div(c), z = P.divy.div(t);
    const int x = (int)(c - t * P.nx), y = (int)(t - z * P.ny);
    const S *lat = (const S *)P.lat;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        int slot;
        uint32_t plane, cell;
        slot_of(P, i, x, y, (int)z, slot, plane, cell);
        double v = 0.0;
        // slot is i or bb(i); both share the weight class of i
        if (slot == i) v = get<S>(lat, P.geom, i, plane, cell, P.sh[i]);
        else v = get<S>(lat, P.geom, BB[i], plane, cell, P.sh[i]);
        P.buf[(uint64_t)i * P.ncell + c] = v;
    }
}

template <typename S>
__global__ void k_set_f(const XferParams P)
{
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= P.ncell) return;
    const uint32_t t = P.divx.div(c), z = P.divy.div(t);
    const int x = (int)(c - t * P.nx), y = (int)(t - z * P.ny);
    S *lat = (S *)P.lat;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
        int slot;
        uint32_t plane, cell;
        slot_of(P, i, x, y, (int)z, slot, plane, cell);
        const double v = P.buf[(uint64_t)i * P.ncell + c];
        if (slot == i) put<S>(lat, P.geom, i, plane, cell, v, P.sh[i]);
        else put<S>(lat, P.geom, BB[i], plane, cell, v, P.sh[i]);
    }
}

hipError_t launch_get_f(int dtype, const XferParams &P, hipStream_t st)
{
    dim3 blk(256), grid((P.ncell + 255) / 256);
    if (dtype == DT_F64) hipLaunchKernelGGL(k_get_f<double>, grid, blk, 0, st, P);
    else if (dtype == DT_F32) hipLaunchKernelGGL(k_get_f<float>, grid, blk, 0, st, P);
    else hipLaunchKernelGGL(k_get_f<_Float16>, grid, blk, 0, st, P);
    return hipGetLastError();
}

hipError_t launch_set_f(int dtype, const XferParams &P, hipStream_t st)
{
    dim3 blk(256), grid((P.ncell + 255) / 256);
    if (dtype == DT_F64) hipLaunchKernelGGL(k_set_f<double>, grid, blk, 0, st, P);
    else if (dtype == DT_F32) hipLaunchKernelGGL(k_set_f<float>, grid, blk, 0, st, P);
    else hipLaunchKernelGGL(k_set_f<_Float16>, grid, blk, 0, st, P);
    return hipGetLastError();
}

// ------------------------------------------------------------ reductions
// Two passes with a fixed assignment of cells to blocks and a fixed tree in
// each block, so the sums are reproducible run to run.

template <int N>
__device__ __forceinline__ void block_sum(double (&v)[N], double (*sh)[256])
{
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < N; ++k) sh[k][t] = v[k];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) {
#pragma unroll
            for (int k = 0; k < N; ++k) sh[k][t] += sh[k][t + s];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = sh[k][0];
}

__global__ void __launch_bounds__(256) k_diag_pass1(const double *p, const double *u, const double *v,
                                                    const double *w, uint32_t n, double *partials)
{
    __shared__ double sh[2][256];
    const uint32_t per = (n + gridDim.x - 1) / gridDim.x;
    const uint32_t lo = blockIdx.x * per, hi = min(n, lo + per);
    double acc[2] = {0.0, 0.0};
    for (uint32_t c = lo + threadIdx.x; c < hi; c += blockDim.x) {
        acc[0] += u[c] * u[c] + v[c] * v[c] + w[c] * w[c];
        acc[1] += 3.0 * p[c];
    }
    block_sum<2>(acc, sh);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = acc[0];
        partials[2 * blockIdx.x + 1] = acc[1];
    }
}

template <int N>
__global__ void __launch_bounds__(256) k_sum_partials(const double *partials, int nparts, double *out, double scale0)
{
    __shared__ double sh[N][256];
    double acc[N];
#pragma unroll
    for (int k = 0; k < N; ++k) acc[k] = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x)
#pragma unroll
        for (int k = 0; k < N; ++k) acc[k] += partials[N * b + k];
    block_sum<N>(acc, sh);
    if (threadIdx.x == 0) {
        out[0] = acc[0] * scale0;
#pragma unroll
        for (int k = 1; k < N; ++k) out[k] = acc[k];
    }
}

hipError_t launch_diag(const double *p, const double *u, const double *v, const double *w, const uint8_t *,
                       uint32_t n, double *partials, int nparts, double *out2, hipStream_t st)
{
    hipLaunchKernelGGL(k_diag_pass1, dim3(nparts), dim3(256), 0, st, p, u, v, w, n, partials);
    hipLaunchKernelGGL(k_sum_partials<2>, dim3(1), dim3(256), 0, st, partials, nparts, out2, 0.5);
    return hipGetLastError();
}

// Momentum handed to the solid by halfway bounce-back, from the
// post-collision populations of the channel (pull storage, natural layout):
// F = sum over fluid x, directions i with x + e_i solid, of 2 f*_i(x) e_i.
template <typename S>
__global__ void __launch_bounds__(256) k_force_pass1(const FusedParams P, double *partials)
{
    __shared__ double sh[3][256];
    const uint32_t n = P.ncell;
    const uint32_t per = (n + gridDim.x - 1) / gridDim.x;
    const uint32_t lo = blockIdx.x * per, hi = min(n, lo + per);
    double acc[3] = {0.0, 0.0, 0.0};
    const S *lat = (const S *)P.src;
    for (uint32_t c = lo + threadIdx.x; c < hi; c += blockDim.x) {
        if (P.mask[c] != 2) continue;
        const uint32_t t = P.divx.div(c);
        const int x = (int)(c - t * P.nx);
        const uint32_t zz = P.divy.div(t);
        const int y = (int)(t - zz * P.ny), z = (int)zz;
#pragma unroll
        for (int i = 1; i < Q; ++i) {
            const int xd = x + EX[i];
            if (xd < 0 || xd >= P.nx) continue;
            int yd = y + EY[i], zd = z + EZ[i];
            yd = yd < 0 ? yd + P.ny : (yd >= P.ny ? yd - P.ny : yd);
            zd = zd < 0 ? zd + P.nz : (zd >= P.nz ? zd - P.nz : zd);
            const uint32_t cd = ((uint32_t)zd * P.ny + (uint32_t)yd) * P.nx + (uint32_t)xd;
            if (P.mask[cd] != 1) continue;
            const double f = 2.0 * get<S>(lat, P.geom, i, zz, (uint32_t)y * P.nx + (uint32_t)x, P.sh[i]);
            acc[0] += f * (double)EX[i];
            acc[1] += f * (double)EY[i];
            acc[2] += f * (double)EZ[i];
        }
    }
    block_sum<3>(acc, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; ++k) partials[3 * blockIdx.x + k] = acc[k];
}

hipError_t launch_force(int dtype, const FusedParams &P, double *partials, int nparts, double *out3, hipStream_t st)
{
    if (dtype == DT_F64) hipLaunchKernelGGL(k_force_pass1<double>, dim3(nparts), dim3(256), 0, st, P, partials);
    else if (dtype == DT_F32) hipLaunchKernelGGL(k_force_pass1<float>, dim3(nparts), dim3(256), 0, st, P, partials);
    else hipLaunchKernelGGL(k_force_pass1<_Float16>, dim3(nparts), dim3(256), 0, st, P, partials);
    hipLaunchKernelGGL(k_sum_partials<3>, dim3(1), dim3(256), 0, st, partials, nparts, out3, 1.0);
    return hipGetLastError();
}

// Domain health: *flag stays 1 while every value of the four moment fields
// is finite and is set to 0 by any lane that finds one that is not (all
// writers store the same 0).  A moment sums all 27 populations of its cell,
// so a non-finite population shows in the moments of the same step.
__global__ void __launch_bounds__(256) k_nonfinite(const double *p, const double *u, const double *v,
                                                   const double *w, uint32_t n, int32_t *flag)
{
    bool bad = false;
    for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x)
        bad |= !(isfinite(p[c]) && isfinite(u[c]) && isfinite(v[c]) && isfinite(w[c]));
    if (bad) *flag = 0;
}

__global__ void k_fill_i32(int32_t *a, int n, int32_t v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

hipError_t launch_finite_flags(const double *const *mom, const uint32_t *ncell, int ndom, int32_t *flags,
                               hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_i32, dim3((ndom + 255) / 256), dim3(256), 0, st, flags, ndom, 1);
    for (int d = 0; d < ndom; ++d) {
        const uint32_t n = ncell[d];
        const int grid = (int)std::min<uint32_t>(1024u, (n + 255) / 256);
        hipLaunchKernelGGL(k_nonfinite, dim3(grid), dim3(256), 0, st, mom[4 * d], mom[4 * d + 1], mom[4 * d + 2],
                           mom[4 * d + 3], n, flags + d);
    }
    return hipGetLastError();
}

// Plain copy, one 16-byte vector per lane, one pass: the reference point for
// the hardware counters and the measured bandwidth ceiling.
typedef double dvec2 __attribute__((ext_vector_type(2)));

__global__ void __launch_bounds__(256) k_copy(const dvec2 *__restrict__ src, dvec2 *__restrict__ dst, size_t n2)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n2) dst[i] = src[i];
}

hipError_t launch_copy(const double *src, double *dst, size_t n, hipStream_t st)
{
    const size_t n2 = n / 2;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, (const dvec2 *)src,
                       (dvec2 *)dst, n2);
    return hipGetLastError();
}

// Bandwidth probes: copy, read-only and write-only streams with V 16-byte
// vectors per lane (a workgroup covers V * 256 consecutive vectors, each
// sub-pass coalesced), optionally non-temporal, or a grid-stride loop over a
// fixed grid.  They bound what any kernel with one read and one write stream
// per value can reach on the part.
template <int V, bool NT>
__global__ void __launch_bounds__(256) k_copy_v(const dvec2 *__restrict__ src, dvec2 *__restrict__ dst, size_t n2)
{
    const size_t base = (size_t)blockIdx.x * 256 * V + threadIdx.x;
    dvec2 x[V];
#pragma unroll
    for (int r = 0; r < V; ++r) {
        const size_t i = base + (size_t)r * 256;
        if (i < n2) x[r] = NT ? __builtin_nontemporal_load(src + i) : src[i];
    }
#pragma unroll
    for (int r = 0; r < V; ++r) {
        const size_t i = base + (size_t)r * 256;
        if (i < n2) {
            if (NT) __builtin_nontemporal_store(x[r], dst + i);
            else dst[i] = x[r];
        }
    }
}

template <bool NT>
__global__ void __launch_bounds__(256) k_copy_gs(const dvec2 *__restrict__ src, dvec2 *__restrict__ dst, size_t n2)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n2; i += (size_t)gridDim.x * 256) {
        if (NT) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
        else dst[i] = src[i];
    }
}

// Read-only: the loaded values feed a sum that is stored only if it equals a
// value the data never sums to, so no load can be dropped.
template <int V, bool NT>
__global__ void __launch_bounds__(256) k_read_v(const dvec2 *__restrict__ src, size_t n2, double never,
                                                double *__restrict__ sink)
{
    const size_t base = (size_t)blockIdx.x * 256 * V + threadIdx.x;
    double acc = 0.0;
#pragma unroll
    for (int r = 0; r < V; ++r) {
        const size_t i = base + (size_t)r * 256;
        if (i < n2) {
            const dvec2 x = NT ? __builtin_nontemporal_load(src + i) : src[i];
            acc += x.x + x.y;
        }
    }
    if (acc == never) sink[threadIdx.x] = acc;
}

template <int V, bool NT>
__global__ void __launch_bounds__(256) k_write_v(dvec2 *__restrict__ dst, size_t n2, double v)
{
    const size_t base = (size_t)blockIdx.x * 256 * V + threadIdx.x;
    const dvec2 x = {v, v};
#pragma unroll
    for (int r = 0; r < V; ++r) {
        const size_t i = base + (size_t)r * 256;
        if (i < n2) {
            if (NT) __builtin_nontemporal_store(x, dst + i);
            else dst[i] = x;
        }
    }
}

int bandwidth_probe_streams(int kind)
{
    switch (kind) {
    case 0: case 1: case 2: case 3: case 4: case 5: return 2;
    case 6: case 7: case 8: case 9: return 1;
    default: return 0;
    }
}

hipError_t launch_bandwidth_probe(int kind, const double *src, double *dst, size_t n, int cus, hipStream_t st)
{
    const size_t n2 = n / 2;
    const auto grid = [&](int v) { return dim3((unsigned)((n2 + 256 * (size_t)v - 1) / (256 * (size_t)v))); };
    const dvec2 *s2 = (const dvec2 *)src;
    dvec2 *d2 = (dvec2 *)dst;
    switch (kind) {
    case 0: hipLaunchKernelGGL((k_copy_v<1, false>), grid(1), dim3(256), 0, st, s2, d2, n2); break;
    case 1: hipLaunchKernelGGL((k_copy_v<1, true>), grid(1), dim3(256), 0, st, s2, d2, n2); break;
    case 2: hipLaunchKernelGGL((k_copy_v<4, false>), grid(4), dim3(256), 0, st, s2, d2, n2); break;
    case 3: hipLaunchKernelGGL((k_copy_v<4, true>), grid(4), dim3(256), 0, st, s2, d2, n2); break;
    case 4: hipLaunchKernelGGL((k_copy_gs<false>), dim3(cus * 8), dim3(256), 0, st, s2, d2, n2); break;
    case 5: hipLaunchKernelGGL((k_copy_gs<true>), dim3(cus * 8), dim3(256), 0, st, s2, d2, n2); break;
    case 6: hipLaunchKernelGGL((k_read_v<4, false>), grid(4), dim3(256), 0, st, s2, n2, -1.0, dst); break;
    case 7: hipLaunchKernelGGL((k_read_v<4, true>), grid(4), dim3(256), 0, st, s2, n2, -1.0, dst); break;
    case 8: hipLaunchKernelGGL((k_write_v<4, false>), grid(4), dim3(256), 0, st, d2, n2, 0.5); break;
    case 9: hipLaunchKernelGGL((k_write_v<4, true>), grid(4), dim3(256), 0, st, d2, n2, 0.5); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Faithful mode on the fused engine: Streaming's boundary phase on the ring
// (the first ghost layer), in the reference's order, before the fused pass
// reads it.  Interior values come from the post-collision lattice P.src.
// Ghost cells deeper than the first layer are never written, so they keep
// Initialize's values: 0 in the cavity, whose fields start at rest with
// p = 0; in the sphere channel the initial fields reach into the ghosts
// (sphere/src/lbm.cpp:224-239 loops over the whole ghosted box), and those
// values are recomputed where a wall reads them.

// the faithful sphere's initial population q at cell (i, j, k) of the
// ghosted box, in interior coordinates (k_init's kind 2 at any cell)
__device__ __forceinline__ double faithful_sphere_f0(const FusedParams &P, uint64_t seed, int q, int i, int j, int k)
{
    const uint64_t ly = (uint64_t)P.ny + 6, lz = (uint64_t)P.nz + 6;
    const uint64_t idx = ((uint64_t)(i + 3) * ly + (uint64_t)(j + 3)) * lz + (uint64_t)(k + 3);
    const int ran = (int)(mix64(seed + idx * 0x9E3779B97F4A7C15ULL) % 100ULL);
    const int usr = faithful_sphere_solid(P.nx, i, j, k) ? 0 : 1;
    const int glz = P.nz, kz = k;
    const double gm = (double)(glz - 1);
    const double u = (P.u0 * 4.0 * (double)kz * (double)(glz - 1 - kz) / (gm * gm)) * (double)usr * (1.0 + (double)ran * 0.001);
    return feq_f64(q, 0.0, u, 0.0, 0.0);
}

// Where population q of cell (i, j, k) is read from, in two steps so that a
// kernel can first place all its sources (the deep-ghost value is computed
// under a branch, with no load in it), then issue all its loads back to back
// (a value loaded before a divergent branch and still live after it would be
// waited for there), then pick.
struct GhostSrc {
    const double *p;  // always a valid address
    double deep;      // the value when the cell lies deeper than the first layer
    bool is_deep;
};

__device__ __forceinline__ GhostSrc faithful_src(const FusedParams &P, int q, int i, int j, int k)
{
    const int64_t r = ring_index(P, i, j, k);
    GhostSrc g;
    g.is_deep = r == -1;
    g.deep = 0.0;
    if (g.is_deep && P.faithful_sphere) g.deep = faithful_sphere_f0(P, P.seed, q, i, j, k);
    const uint64_t in_cell = r == -2 ? P.geom.off(q, (uint32_t)k, (uint32_t)j * P.nx + i) : 0;
    g.p = r == -2 ? (const double *)P.src + in_cell
                  : P.ring + (uint64_t)q * P.ring_n + (uint64_t)(r < 0 ? 0 : r);
    return g;
}

// The coordinates of cell r of the ring (ring_index backwards).
__device__ __forceinline__ void ring_cell(const FusedParams &P, uint32_t r, int &i, int &j, int &k)
{
    if (r < 2 * P.ring_a) {
        const bool high = r >= P.ring_a;
        r -= high ? P.ring_a : 0;
        i = high ? P.nx : -1;
        k = (int)(r / (uint32_t)(P.ny + 2));
        j = (int)(r - (uint32_t)k * (uint32_t)(P.ny + 2)) - 1;
        k -= 1;
        return;
    }
    r -= 2 * P.ring_a;
    const bool yf = r < 2 * P.ring_b;
    r -= yf ? 0 : 2 * P.ring_b;
    const uint32_t n = yf ? P.ring_b : P.ring_c;
    const bool high = r >= n;
    r -= high ? n : 0;
    const int row = (int)P.divx.div(r);
    i = (int)(r - (uint32_t)row * (uint32_t)P.nx);
    j = yf ? (high ? P.ny : -1) : row;
    k = yf ? row - 1 : (high ? P.nz : -1);
}

// Initialize for the ring: every first-layer ghost cell takes its initial
// populations (0 in the cavity).
__global__ void k_faithful_ring_init(const FusedParams P)
{
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= P.ring_n) return;
    int i, j, k;
    ring_cell(P, r, i, j, k);
#pragma unroll
    for (int q = 0; q < Q; ++q)
        P.ring[(uint64_t)q * P.ring_n + r] = P.faithful_sphere ? faithful_sphere_f0(P, P.seed, q, i, j, k) : 0.0;
}

hipError_t launch_faithful_ring_init(const FusedParams &P, hipStream_t st)
{
    hipLaunchKernelGGL(k_faithful_ring_init, dim3((P.ring_n + 255) / 256), dim3(256), 0, st, P);
    return hipGetLastError();
}

// "usrbc", sphere/src/lbm.cpp:350-356: a solid cell takes, for each
// direction q whose neighbour x + e_q is fluid, f_bb(q)(x + 2 e_q), in place
// in the post-collision lattice.  The reference's mask covers the ghost
// cells too: where the ball reaches the first ghost layer (ny or nz within r
// of its centre), a ghost neighbour can be solid, and its mask value is
// recomputed here.  A source is never a target: between two solid voxels of a
// ball the midpoint voxel is solid too, so that direction is not taken.  The
// (cell, q) pairs are therefore independent: thread t of direction q
// takes cell t of the box [lo, lo + n)^3 around the ball (clamped to the
// cavity), so that the few thousand cells of the box fill 27 times as many
// lanes.  Every thread loads (threads off the box from a valid cell) and only
// solid cells store: no load sits under a divergent branch.
__device__ __forceinline__ void faithful_usr(const FusedParams &P, int lo, int n, int q, int t)
{
    int e[3], bq;
    dir_of(q, e, bq);
    const int ex = e[0], ey = e[1], ez = e[2];
    const int tt = t < n * n * n ? t : 0;
    const int x0 = lo + tt % n, y0 = lo + (tt / n) % n, z0 = lo + tt / (n * n);
    const bool valid = (t < n * n * n) & (x0 < P.nx) & (y0 < P.ny) & (z0 < P.nz);
    const int x = valid ? x0 : 0, y = valid ? y0 : 0, z = valid ? z0 : 0;
    const uint32_t c = ((uint32_t)z * P.ny + y) * P.nx + x;
    const int xi = x + ex, yi = y + ey, zi = z + ez;
    const bool in = (xi >= 0) & (xi < P.nx) & (yi >= 0) & (yi < P.ny) & (zi >= 0) & (zi < P.nz);
    const uint64_t mi = in ? ((uint64_t)zi * P.ny + yi) * P.nx + xi : (uint64_t)c;
    const GhostSrc g = faithful_src(P, bq, x + 2 * ex, y + 2 * ey, z + 2 * ez);
    const uint8_t mc = P.mask[c];
    const uint8_t m = P.mask[mi];
    double v = *g.p;
    v = g.is_deep ? g.deep : v;
    const bool solid = valid & (mc == 1);
    const bool nb_solid = in ? m == 1 : faithful_sphere_solid(P.nx, xi, yi, zi);
    if (solid & !nb_solid) ((double *)P.src)[P.geom.off(q, (uint32_t)z, (uint32_t)y * P.nx + x)] = v;
}

__global__ void k_faithful_usr(const FusedParams P, int lo, int n)
{
    faithful_usr(P, lo, n, blockIdx.y, blockIdx.x * blockDim.x + threadIdx.x);
}

// The boundary phase on the ring, in one launch.  The reference fills the ghost
// cells in several passes, each reading what an earlier one wrote:
//   cavity: the one-rank unpack of lid_driven_cavity/src/mpi_view_transfer.cpp:
//     617-688 zeroes the planes x = -1, x = nx, y = ny and z = nz (it copies
//     receive buffers that nothing filled), then the x, y and z walls
//     (lid_driven_cavity/src/lbm.cpp:233-301) write, for every first-layer cell
//     of their plane and direction q pointing into the cavity,
//     f_q(cell) = f_bb(q)(cell + 2 e_q on the plane n - 2 or 1 of their axis; the
//     top wall takes one e_y instead of two);
//   sphere: the y and z walls, then the inlet copy f_q(-1, y, z) = f_q(0, y, z) and
//     the outlet copy f_q(nx, y, z) = f_q(nx - 1, y + e_y, z + e_z)
//     (sphere/src/lbm.cpp:277-347).
// Here every entry that a pass writes finds its value by itself: the last pass
// that writes it names a source, of which an earlier pass may be the last
// writer, and so on -- at most three times, always between q and bb(q) -- down to a
// cell of the lattice, a ghost cell deeper than the first layer, a zeroed
// plane, or an entry that no pass before it wrote this step and that therefore
// still holds the last step's value.  Those are read from the last step's ring,
// so the two rings change places every step and no thread reads what another
// writes.  Entries that no pass writes hold Initialize's values in both.
//
// It is bound by latency, not by what it moves: the launches, and per thread one
// load of what another XCD wrote last.  us a step, a launch per pass before / now:
// cavity 100^3 20 / 8 of a step of 92 / 84, sphere 512x128x128 45 / 20 of
// 640 / 626; whole steps: sphere 72x24x24 27 / 11, cavity 24x16x24 19 / 10.

// Workgroups of one face of each axis, of one direction of the edges' cells, and
// of one direction of the box [lo, lo + n)^3 around the ball (0: not here).
struct RingBlocks {
    uint32_t x, y, z, edges, ball;
    int lo, n;
};

// One entry of the ring on its way to its value: the cell, the direction there
// (q, or bb(q) when turned) and how many of the step's passes come before.
struct RingEntry {
    int i, j, k, turned, before;
};

// Follows the entry through the last pass before `before` that writes it
// (passes 0, 1, 2: the cavity's x, y, z walls; the sphere's y and z walls and
// its inlet and outlet); false: none does.
template <bool SPHERE>
__device__ __forceinline__ bool ring_hop(const FusedParams &P, const int e[3], RingEntry &t)
{
    const int nx = P.nx, ny = P.ny, nz = P.nz, sg = t.turned ? -1 : 1;
    const int ex = sg * e[0], ey = sg * e[1], ez = sg * e[2];
    const bool first = t.i >= -1 && t.i <= nx && t.j >= -1 && t.j <= ny && t.k >= -1 && t.k <= nz;
    // written by the pass of an axis: a first-layer ghost cell of that axis, the
    // direction pointing inward there
    const bool in_x = first && ((t.i < 0 && ex > 0) || (t.i >= nx && ex < 0));
    const bool in_y = first && ((t.j < 0 && ey > 0) || (t.j >= ny && ey < 0));
    const bool in_z = first && ((t.k < 0 && ez > 0) || (t.k >= nz && ez < 0));
    const bool copy = SPHERE && in_x && t.before > 2;
    const bool wz = !copy && in_z && t.before > (SPHERE ? 1 : 2);
    const bool wy = !copy && !wz && in_y && t.before > (SPHERE ? 0 : 1);
    const bool wx = !SPHERE && !wz && !wy && in_x && t.before > 0;
    const bool wall = wx || wy || wz;
    const bool out = copy && ex < 0;
    const int sy = wz && !SPHERE && ez < 0 ? 1 : 2;  // the cavity's top wall
    t.i = copy ? (out ? nx - 1 : 0) : wx ? (ex > 0 ? 1 : nx - 2) : wall ? t.i + 2 * ex : t.i;
    t.j = out ? t.j + ey : wy ? (ey > 0 ? 1 : ny - 2) : wall ? t.j + sy * ey : t.j;
    t.k = out ? t.k + ez : wz ? (ez > 0 ? 1 : nz - 2) : wall ? t.k + 2 * ez : t.k;
    t.before = copy ? 2 : wz ? (SPHERE ? 1 : 2) : wy ? (SPHERE ? 0 : 1) : 0;
    t.turned = wall ? !t.turned : t.turned;
    return copy || wall;
}

// What the entry holds once no pass before it writes it.
template <bool SPHERE>
__device__ __forceinline__ double ring_value(const FusedParams &P, const double *last, int q, int bq, const int e[3],
                                             const RingEntry &t)
{
    const int c = t.turned ? bq : q, cx = t.turned ? -e[0] : e[0];
    const int64_t rc = ring_index(P, t.i, t.j, t.k);
    const bool inside = rc == -2, deep = rc == -1;
    // an interior cell on the planes that the fused pass copies beside the
    // lattice, y fastest (one strided cell per row of the lattice otherwise)
    const bool lo = SPHERE ? t.i == 0 && cx > 0 : t.i == 1 && cx < 0;
    const bool hi = SPHERE ? t.i == P.nx - 1 && cx < 0 : t.i == P.nx - 2 && cx > 0;
    const double *p = last + (uint64_t)c * P.ring_n + (uint64_t)(rc < 0 ? 0 : rc);
    if (inside)
        p = lo || hi ? P.stage + (((uint64_t)(lo ? 0 : 1) * P.nz + t.k) * P.ny + t.j) * STAGE_ROW + x_rank(c)
                     : (const double *)P.src + P.geom.off(c, (uint32_t)t.k, (uint32_t)t.j * P.nx + t.i);
    double v = *p;
    if (SPHERE) {
        if (deep) v = faithful_sphere_f0(P, P.seed, c, t.i, t.j, t.k);
    } else if (!inside && (deep || t.i < 0 || t.i >= P.nx || t.j >= P.ny || t.k >= P.nz)) {
        v = 0.0;  // never written, or zeroed by the unpack
    }
    return v;
}

// Workgroups: where the ball lies clear of what the passes read, its usrbc; then
// the edges' cells, three directions of the 27 to a row (the long
// ways start early); then per face its cells with one ghost coordinate, row y the
// y-th of the nine directions entering there (the pass of that axis writes it, and
// nearly always its source lies inside).
template <bool SPHERE>
__global__ void __launch_bounds__(256) k_faithful_ring(const FusedParams P, const double *last, RingBlocks nb)
{
    const int nx = P.nx, ny = P.ny, nz = P.nz;
    uint32_t b = blockIdx.x;
    if (SPHERE && b < 3 * nb.ball) {
        faithful_usr(P, nb.lo, nb.n, 3 * (int)blockIdx.y + (int)(b % 3), (int)(b / 3 * 256 + threadIdx.x));
        return;
    }
    b -= 3 * nb.ball;
    if (b >= 3 * nb.edges) {
        b -= 3 * nb.edges;
        const int axis = b < 2 * nb.x ? 0 : b < 2 * (nb.x + nb.y) ? 1 : 2;
        b -= axis == 0 ? 0 : axis == 1 ? 2 * nb.x : 2 * (nb.x + nb.y);
        const uint32_t n = axis == 0 ? nb.x : axis == 1 ? nb.y : nb.z;
        const bool high = b >= n;
        const uint32_t t = (b - (high ? n : 0)) * 256 + threadIdx.x;
        const uint32_t la = axis == 0 ? ny : nx, lb = axis == 2 ? ny : nz;
        const uint32_t B = t / la, A = t - B * la;
        if (B >= lb) return;
        const int q = axis == 0 ? (high ? nth_dir<0, -1>(blockIdx.y) : nth_dir<0, 1>(blockIdx.y))
                    : axis == 1 ? (high ? nth_dir<1, -1>(blockIdx.y) : nth_dir<1, 1>(blockIdx.y))
                                : (high ? nth_dir<2, -1>(blockIdx.y) : nth_dir<2, 1>(blockIdx.y));
        int e[3], bq;
        dir_of(q, e, bq);
        RingEntry w;
        w.i = axis == 0 ? (high ? nx : -1) : (int)A;
        w.j = axis == 1 ? (high ? ny : -1) : axis == 0 ? (int)A : (int)B;
        w.k = axis == 2 ? (high ? nz : -1) : (int)B;
        const uint64_t r = (uint64_t)ring_index(P, w.i, w.j, w.k);
        const bool copy = SPHERE && axis == 0;
        const int s = copy ? (high ? 1 : 0) : 2, sy = !SPHERE && axis == 2 && high ? 1 : s;
        w.i = axis == 0 ? (high ? (copy ? nx - 1 : nx - 2) : (copy ? 0 : 1)) : w.i + s * e[0];
        w.j = axis == 1 ? (high ? ny - 2 : 1) : w.j + sy * e[1];
        w.k = axis == 2 ? (high ? nz - 2 : 1) : w.k + s * e[2];
        w.turned = !copy;
        w.before = SPHERE ? (axis + 2) % 3 : axis;
        if (w.i < 0 || w.i >= nx || w.j < 0 || w.j >= ny || w.k < 0 || w.k >= nz) {
            if (ring_hop<SPHERE>(P, e, w)) ring_hop<SPHERE>(P, e, w);
        }
        P.ring[(uint64_t)q * P.ring_n + r] = ring_value<SPHERE>(P, last, q, bq, e, w);
        return;
    }
    const int q = 3 * (int)blockIdx.y + (int)(b % 3);
    uint32_t t = b / 3 * 256 + threadIdx.x;
    RingEntry w;
    if (t < 4 * (uint32_t)(ny + 2)) {  // along y
        const int l = (int)(t / (uint32_t)(ny + 2));
        w.i = l & 1 ? nx : -1;
        w.k = l & 2 ? nz : -1;
        w.j = (int)t - l * (ny + 2) - 1;
    } else if ((t -= 4 * (uint32_t)(ny + 2)) < 4 * (uint32_t)nz) {  // along z
        const int l = (int)(t / (uint32_t)nz);
        w.i = l & 1 ? nx : -1;
        w.j = l & 2 ? ny : -1;
        w.k = (int)t - l * nz;
    } else if ((t -= 4 * (uint32_t)nz) < 4 * (uint32_t)nx) {  // along x
        const int l = (int)(t / (uint32_t)nx);
        w.j = l & 1 ? ny : -1;
        w.k = l & 2 ? nz : -1;
        w.i = (int)t - l * nx;
    } else {
        return;
    }
    w.turned = 0;
    w.before = 3;
    const uint64_t r = (uint64_t)ring_index(P, w.i, w.j, w.k);
    int e[3], bq;
    dir_of(q, e, bq);
    if (!ring_hop<SPHERE>(P, e, w)) return;  // no pass writes this entry
    if (ring_hop<SPHERE>(P, e, w)) ring_hop<SPHERE>(P, e, w);
    P.ring[(uint64_t)q * P.ring_n + r] = ring_value<SPHERE>(P, last, q, bq, e, w);
}

// FusedParams::stage from the lattice P.src: thread t is entry t of the
// stage (side, z, y, r).
__global__ void k_faithful_stage_fill(const FusedParams P)
{
    const uint64_t plane = (uint64_t)P.ny * P.nz;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 2 * plane * STAGE_ROW) return;
    const int r = (int)(t % STAGE_ROW);
    const uint64_t row = t / STAGE_ROW;  // side * plane + (z ny + y)
    const int side = row >= plane ? 1 : 0;
    const uint64_t yz = row - (side ? plane : 0);
    int q;
    uint32_t x;
    if (P.faithful_sphere) {  // inlet x = 0, e_x > 0; outlet x = nx - 1, e_x < 0
        q = side == 0 ? nth_dir<0, 1>(r) : nth_dir<0, -1>(r);
        x = side == 0 ? 0u : (uint32_t)P.nx - 1u;
    } else {  // walls: x = 1, e_x < 0; x = nx - 2, e_x > 0
        q = side == 0 ? nth_dir<0, -1>(r) : nth_dir<0, 1>(r);
        x = side == 0 ? 1u : (uint32_t)P.nx - 2u;
    }
    const uint32_t z = (uint32_t)(yz / P.ny), y = (uint32_t)(yz - (uint64_t)z * P.ny);
    P.stage[t] = ((const double *)P.src)[P.geom.off(q, z, y * P.nx + x)];
}

hipError_t launch_faithful_stage_fill(const FusedParams &P, hipStream_t st)
{
    const uint64_t n = 2ull * P.ny * P.nz * STAGE_ROW;
    hipLaunchKernelGGL(k_faithful_stage_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, P);
    return hipGetLastError();
}

hipError_t launch_faithful_boundaries(const FusedParams &P, const double *last_ring, hipStream_t st)
{
    auto blocks = [](int64_t n) { return (uint32_t)((n + 255) / 256); };
    RingBlocks nb{blocks((int64_t)P.ny * P.nz), blocks((int64_t)P.nx * P.nz), blocks((int64_t)P.nx * P.ny),
                  blocks(4ll * (P.nx + P.ny + 2 + P.nz)), 0, 0, 0};
    dim3 grid(2 * (nb.x + nb.y + nb.z) + 3 * nb.edges, 9);
    if (!P.faithful_sphere) {
        hipLaunchKernelGGL(k_faithful_ring<false>, grid, dim3(256), 0, st, P, last_ring, nb);
        return hipGetLastError();
    }
    // one rank: the unpack has nothing to write.  The ball lies within
    // [c - r, c + r] of its centre c on every axis.  Where that box stays two
    // cells off every face, usrbc reads no ghost cell and no pass reads a cell of
    // the box (their sources lie on the two outermost planes of an axis): one
    // launch does both.  Elsewhere usrbc follows in its own, as in the reference.
    const int cc = (P.nx - 1) / 8, rr = (int)std::ceil((P.nx - 1) / 64.0);
    nb.lo = cc - rr < 0 ? 0 : cc - rr;
    nb.n = cc + rr - nb.lo + 1;
    const int low = P.nx < P.ny ? P.nx : P.ny, least = low < P.nz ? low : P.nz;
    const uint32_t ball = blocks((int64_t)nb.n * nb.n * nb.n);
    const bool clear = nb.lo >= 2 && nb.lo + nb.n <= least - 2;
    if (clear) nb.ball = ball;
    grid.x += 3 * nb.ball;
    hipLaunchKernelGGL(k_faithful_ring<true>, grid, dim3(256), 0, st, P, last_ring, nb);
    if (!clear) hipLaunchKernelGGL(k_faithful_usr, dim3(ball, Q), dim3(256), 0, st, P, nb.lo, nb.n);
    return hipGetLastError();
}

// Device arrays into pinned host memory (CopyOut), 16 bytes per thread and pass,
// straight over the link, whose 54 GB/s bound it (2 MiB 39 us); a read of a few
// hundred KiB is bound by the launch and the wait, hence one launch for all four.
__global__ void __launch_bounds__(256) k_copy_out(const CopyOut C)
{
    typedef uint32_t Unit __attribute__((ext_vector_type(4)));
    for (uint64_t u = (uint64_t)blockIdx.x * 256 + threadIdx.x; u < C.at[4]; u += (uint64_t)gridDim.x * 256) {
        const int k = (u >= C.at[1]) + (u >= C.at[2]) + (u >= C.at[3]);
        const char *base = k == 0 ? C.src[0] : k == 1 ? C.src[1] : k == 2 ? C.src[2] : C.src[3];
        const uint64_t bytes = k == 0 ? C.bytes[0] : k == 1 ? C.bytes[1] : k == 2 ? C.bytes[2] : C.bytes[3];
        const uint64_t first = k == 0 ? C.at[0] : k == 1 ? C.at[1] : k == 2 ? C.at[2] : C.at[3];
        const uint64_t o = (u - first) * 16;
        const char *const s = base + o;
        char *const d = C.dst + u * 16;
        if (o + 16 <= bytes && (uintptr_t)base % 8 == 0) {
            if ((uintptr_t)base % 16 == 0) {
                __builtin_nontemporal_store(__builtin_nontemporal_load((const Unit *)s), (Unit *)d);
            } else {
                const uint64_t a = ((const uint64_t *)s)[0], b = ((const uint64_t *)s)[1];
                const Unit v = {(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
                __builtin_nontemporal_store(v, (Unit *)d);
            }
        } else {
            for (uint64_t b = 0; b < 16 && o + b < bytes; ++b) d[b] = s[b];
        }
    }
}

hipError_t launch_copy_out(const CopyOut &C, hipStream_t st)
{
    const uint64_t blocks = (C.at[4] + 255) / 256;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy_out, dim3((unsigned)(blocks < 512 ? blocks : 512)), dim3(256), 0, st, C);
    return hipGetLastError();
}

}  // namespace imx
