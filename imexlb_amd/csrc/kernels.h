// Kernel parameter blocks and host-side launchers shared by the HIP
// translation units and the C-ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lattice.h"

// Bytes added to each population stride of a fused-engine lattice (after
// rounding the cell count up to 256 bytes): 9 x 256 keeps the 27 streams off a
// common power-of-two alignment.
#ifndef IMEXLB_DEFAULT_PAD
#define IMEXLB_DEFAULT_PAD 2304
#endif

namespace imx {

// BC_FAITHFUL: the cavity with the reference's own wall, lid and halo rules;
// the first ghost layer lives in a ring of face arrays (FusedParams::ring).
enum Bc : int { BC_PERIODIC = 0, BC_CAVITY = 1, BC_CHANNEL = 2, BC_FAITHFUL = 3 };
enum Pattern : int { PAT_PULL = 0, PAT_AA_EVEN = 1, PAT_AA_ODD = 2 };
enum Dtype : int { DT_F64 = 0, DT_F32 = 1, DT_F16 = 2 };

// The faithful sphere's inlet perturbation replaces Kokkos' random pool by a
// seeded counter hash: the splitmix64 finaliser (Steele, Lea and Flood, "Fast
// splittable pseudorandom number generators", OOPSLA 2014).
__host__ __device__ __forceinline__ uint64_t mix64(uint64_t x)
{
    x ^= x >> 30;
    x *= 0xBF58476D1CE4E5B9ULL;
    x ^= x >> 27;
    x *= 0x94D049BB133111EBULL;
    x ^= x >> 31;
    return x;
}

// Division by a run-time invariant 32-bit divisor (Granlund & Montgomery,
// "Division by invariant integers using multiplication", PLDI 1994, fig. 4.1):
// exact for every 32-bit dividend.
struct FastDiv {
    uint32_t d, m, s1, s2;
    void init(uint32_t div)
    {
        d = div;
        uint32_t l = 0;
        while ((uint64_t(1) << l) < div) ++l;
        m = uint32_t(((uint64_t(1) << 32) * ((uint64_t(1) << l) - div)) / div + 1);
        s1 = l < 1 ? l : 1;
        s2 = l > 0 ? l - 1 : 0;
    }
#if defined(__HIPCC__)
    __device__ __forceinline__ uint32_t div(uint32_t n) const
    {
        uint32_t t = __umulhi(m, n);
        return (t + ((n - t) >> s1)) >> s2;
    }
#endif
};

// One fused stream + moments + collide launch over a single domain.
// The address mode the fused kernels run with (fused.h AddrMode): 2 (a
// uniform base per group of 16 / elem populations, 32-bit offsets) while such
// a group spans at most 4 GiB, else 1 (a uniform base per population) while a
// population does, else 0 (64-bit offsets); capped at am_max.
inline int fused_addr_mode(uint64_t elem, uint64_t pstride, int am_max)
{
    const uint64_t lim = uint64_t(1) << 32;
    if (am_max >= 2 && pstride * 16 <= lim) return 2;
    if (am_max >= 1 && pstride * elem <= lim) return 1;
    return 0;
}

// Doubles per row of FusedParams::stage: the nine populations of one row of
// the lattice, together.
constexpr int STAGE_ROW = 9;

// The cells per thread the fused kernels run with for a requested `cpt`:
// two adjacent cells (3) only on periodic lattices with nx even and grouped
// bases (address mode 2), two cells blockDim apart (2) only with grouped
// bases, else one.
inline int fused_cells_per_thread(int cpt, int bc, uint32_t nx, int am)
{
    if (am != 2) return 1;
    if (cpt == 3) return bc == BC_PERIODIC && nx % 2 == 0 ? 3 : 1;
    return cpt == 2 ? 2 : 1;
}

// Where population i of cell (z, p), p = y nx + x, lies in a lattice, in
// elements: z zs + pos(i) is + (p >> tl) ts + p, i.e. within a z plane the cells
// come in tiles of 2^tl, and a tile holds its populations one after the other.
//
// Two layouts:
// - structure of arrays: one tile per lattice (tl = 31), is = the population
//   stride, zs = nx ny.
// - plane tiles: each z plane is a row of tiles of T = 2^tl cells, is = T,
//   zs = 27 T tiles.  One population of a tile is at most 32 KiB, so the 27
//   accesses of a wavefront fall into neighbouring DRAM rows of the same
//   channels, where 27 arrays a gigabyte apart open 27 rows in banks that the
//   lattice's place in HBM decides.  In-place 27-stream pass over 512^3 FP64,
//   no arithmetic, TB/s (arrays / tiles of 4 / 8 / 16 / 32 / 64 / 128 KiB per
//   population): 5.5 / 6.0 / 6.3 / 6.5 / 6.5 / 6.3 / 5.7, at every offset in 200 GiB
//   for the tiles (6.5), 5.5 or 6.4 by offset for the arrays; a pull pass 5.3 / 5.9 / 6.0 /
//   6.1 / 6.2 / 6.0 / 5.5.  Tiles that are not a power of two, or padded
//   between populations, were slower (6.0).
//
// AA lattices in tiles keep the populations sorted by e_z (by_ez): the odd step
// reads and writes nine of them in each of three planes, and those nine are
// then neighbours.  TGV 512^3 passes without arithmetic, TB/s, index order /
// by e_z: odd step FP64 5.7 / 6.0, FP32 5.7 / 5.9, even step 6.6 / 6.5, 6.5 / 6.4;
// pull 6.3 / 6.2, so pull lattices keep the index order.
struct LatGeom {
    uint64_t zs, is;
    uint32_t ts, tl;
    int by_ez;
#if defined(__HIPCC__)
    // the place of population i among a tile's 27 (i: a compile-time constant)
    __host__ __device__ __forceinline__ int pos(int i) const { return by_ez ? EZ_POS.v[i] : i; }
    __host__ __device__ __forceinline__ uint64_t off(int place, uint32_t z, uint32_t p) const
    {
        return (uint64_t)z * zs + (uint64_t)place * is + (uint64_t)(p >> tl) * ts + p;
    }
#endif
};

inline LatGeom soa_geom(uint32_t nx, uint32_t ny, uint64_t pstride)
{
    return LatGeom{(uint64_t)nx * ny, pstride, 0, 31, 0};
}

// The layout in a tuner's cache key.
inline const char *layout_name(const LatGeom &g) { return g.tl == 31 ? "arrays" : "tiles"; }

// Elements of a lattice of nz planes.
inline uint64_t lattice_elems(const LatGeom &g, uint32_t nz)
{
    return g.tl == 31 ? (uint64_t)Q * g.is : (uint64_t)nz * g.zs;
}

// Plane tiles for a lattice: the largest tile, of 128 bytes (a line) to 32 KiB per
// population, whose last one leaves at most a sixteenth of the plane unused, else
// tiles of a line.  Not for planes below 64 cells, whose wavefronts would be mostly
// idle (a workgroup never spans two planes), nor where three planes exceed the 4 GiB
// that the kernels' 32-bit offsets reach.  Tiles of a line instead of 64 cells take
// a quarter (FP64) and a sixth (FP32) of the memory off planes of 10x13 and are as fast or
// faster: us per step, 64 cells / a line, 12x12x69444 FP64 pull 751 / 731, FP32 AA 440 / 428, 12x12x13889
// FP32 AA 83.6 / 64.0 (the lattice then fits the last-level cache).
inline bool tile_geom(uint32_t nx, uint32_t ny, uint64_t elem, bool aa, LatGeom &g)
{
    const uint64_t plane = (uint64_t)nx * ny;
    if (plane < 64) return false;
    const uint32_t line = elem == 8 ? 4 : elem == 4 ? 5 : 6;
    uint32_t tl = line;
    for (uint32_t t = line; (elem << t) <= 32768; ++t) {
        const uint64_t n = ((plane - 1) >> t) + 1;
        if (((n << t) - plane) * 16 <= plane) tl = t;
    }
    const uint64_t tiles = ((plane - 1) >> tl) + 1;
    const uint64_t zs = (tiles * Q) << tl;
    if (3 * zs * elem > (uint64_t(1) << 32)) return false;
    g = LatGeom{zs, uint64_t(1) << tl, (uint32_t)(Q - 1) << tl, tl, aa ? 1 : 0};
    return true;
}

// Whether a lattice that tile_geom lays out in tiles is better off in them than in
// arrays.  A plane in tiles starts on a line and in a wavefront of its own, so
// what its last line and its last wavefront hold beyond it is spent; arrays run
// through the planes.  us per step, arrays / tiles:
// - beyond the last-level cache the lines count.  Tiles of whole lines gain 9-10 %,
//   so a twelfth of a plane is the most to spend: of 1e7 cells, 16x16 FP16 pull (none)
//   231 / 213, 30x20 (a fifteenth) 221 / 214, 20x20 (an eighth) 209 / 223, 19x17 (a fifth)
//   213 / 242, 10x13 (half) 239 / 304, 13x5 (all) 243 / 421, 12x12 FP64 (none) 850 / 731;
// - in it tiles gain more, a fifth to a half: 2e6 cells FP16 pull 216 MB, 19x17 (a fifth)
//   48.0 / 36.7, 12x12 (a third) 49.6 / 53.2, 9x8 (three quarters) 50.8 / 65.4; 4e5
//   cells FP32 pull 86 MB, 9x8 (a third) 20.9 / 16.6, 10x13 (a quarter) 20.7 / 16.0;
// - in the L2s (32 MB) the wavefronts count: none while each has a SIMD of its own
//   (13x5x308 FP32 pull 4.23 / 3.97, 9x8x278 FP64 pull 6.22 / 6.21), few while all of
//   them are resident, four to a SIMD (12x12x694 FP32 pull 6.31 / 5.41, 10x13x769 FP32 AA
//   5.76 / 5.79, 9x8x1389 FP16 AA 4.97 / 6.01), more beyond (FP16 AA of 4e5 cells: 16x16
//   10.2 / 10.0, 12x12 10.3 / 10.6, 10x13 10.5 / 11.7, 9x8 10.6 / 14.0); both count just
//   beyond them (FP64 pull 43 MB, 13x5x1538 9.9 / 11.8, 9x8x1389 9.6 / 11.2).
// The rule leaves out, for want of a cause: FP64 pull of 36 to 46 MiB with a quarter
// or more of the lanes idle (12x12x700 9.4 / 10.4) and the config cavity's AA beyond the
// last-level cache with planes of 20x20, 24x24 and 40x40 (FP32 20x20x15000 242 / 257; 16x16
// 240 / 220).
// At other sizes tiles serve: TGV 8^3 FP64 5.6 / 4.1, 16^3 5.86 / 4.17, FP32 4.12 / 3.19, FP16 AA
// 3.88 / 3.15, 9x13x30 FP64 5.88 / 4.15, 22x18x22 6.03 / 4.32, faithful cavity 16^3 10.1 / 8.8.
constexpr uint64_t LAST_LEVEL = uint64_t(256) << 20;
inline bool tiles_serve(const LatGeom &g, uint32_t nx, uint32_t ny, uint32_t nz, uint64_t elem, bool aa)
{
    const uint64_t plane = (uint64_t)nx * ny, bytes = lattice_elems(g, nz) * elem * (aa ? 1 : 2);
    const uint64_t spent = (plane * elem + 127) / 128 * 128 - plane * elem;
    if (bytes > LAST_LEVEL) return spent * 12 <= plane * elem;
    if (bytes > LAST_LEVEL / 2) return spent * 4 <= plane * elem;
    const uint64_t waves = (plane + 63) / 64, idle = waves * 64 - plane, mib = uint64_t(1) << 20;
    if (bytes > 32 * mib) return spent * 2 <= plane * elem && (bytes > 48 * mib || idle * 2 <= plane);
    return waves * nz <= 1024 || idle * (waves * nz <= 4096 ? 2 : 4) <= plane;
}

// The XCD-aware order of the plane-tile kernels (tile.h tile_block_of, with the
// measurements): one run of the lattice per XCD (1) where the lattices of a
// step fit the 256 MB last-level cache, else runs of eight workgroups.
constexpr int XCD_RUNS = 2;
inline int tile_order(uint64_t lattice_bytes, bool aa)
{
    return (aa ? lattice_bytes : 2 * lattice_bytes) <= LAST_LEVEL ? 1 : XCD_RUNS;
}

// Default for non-temporal accesses (imexlb_config.nt_loads) over plane tiles: not
// where the lattices of a step fit the 256 MB last-level cache, which keeps what
// plain loads and stores bring in (an in-place pass over 64 to 256 MB: 6.4 TB/s
// non-temporal, 6.6-7.1 plain; over 448 MB 6.4 and 5.7).  us per step,
// non-temporal / plain: pull FP64 64^3 22.5 / 18.7, 80^3 41.8 / 34.9, FP32 96^3
// 34.7 / 29.4, FP16 96^3 19.7 / 17.0, faithful cavity 80^3 48.0 / 41.6, but FP64 96^3 (382 MB)
// 67.3 / 72.0; AA FP64 64^3 20.4 / 18.8, 96^3 59.6 / 56.1, 128^3 (453 MB) 138 / 161, FP32
// 128^3 66.2 / 63.9, FP16 128^3 40.1 / 34.2.
//
// FP64 pull lattices of about the L2s' 32 MB stay non-temporal: a bracket that the
// measurements draw, whose cause (why it ends between 44^3 and 52^3, where the pair
// leaves the L2s) is not known (32^3 5.34 / 5.31, 36^3 5.79 / 6.09, 40^3 6.38 / 7.18, 44^3 8.21 / 8.95, 48^3 10.14 / 10.24, 52^3 14.7 / 12.1).
inline bool tile_nt(uint64_t lattice_bytes, bool aa, uint64_t elem)
{
    const uint64_t bytes = aa ? lattice_bytes : 2 * lattice_bytes, mib = uint64_t(1) << 20;
    return bytes > LAST_LEVEL || (!aa && elem == 8 && bytes > 16 * mib && bytes <= 40 * mib);
}

// Threads per workgroup of the plane-tile kernels where the caller names
// none: 64 below 200000 cells, where the chip has more compute units than there are
// larger workgroups (us per step, 64 / 256: TGV 24^3 FP64 AA 4.9 / 5.8, 32^3 5.7 / 6.3, 40^3
// 7.4 / 9.0, 56^3 14.5 / 14.8, 64^3 20.3 / 20.3 and FP16 7.0 / 6.8); above, the largest of
// 256, 128 and 64 that leaves at most a sixteenth of the plane's threads idle, else
// the one that leaves the fewest.  192, from measurements alone (no cause is known), for
// the FP16 channel (`channel_f16`) once its two
// lattices exceed the 256 MB last-level cache: us per step, 128 / 192 / 256, 512x256x256
// 650 / 605 / 655, 448x288x184 443 / 426 / 430, 640x256x160 483 / 469 / 477, 512x256x128
// 318 / 299 / 315, 678x246x190 600 / 577 / 589, 300x150x150 129 / 125 / 128, 384x192x192
// 260 / 262 / 257, 224x128x128 72.4 / 70.8 / 72.6, but inside it 160x96x96 35.6 / 35.0 / 34.5; not for
// the periodic box (256^3 297 / 301, but 384x256x256 466 / 449) nor FP32 (1248 / 1227).
inline int tile_block(uint64_t plane, uint64_t cells, bool channel_f16)
{
    if (cells < 200000) return 64;
    if (channel_f16 && cells * Q * 2 * 2 > LAST_LEVEL && ((plane + 191) / 192 * 192 - plane) * 16 <= plane) return 192;
    int best = 256;
    uint64_t idle_best = ~uint64_t(0);
    for (int b = 256; b >= 64; b /= 2) {
        const uint64_t idle = (plane + b - 1) / b * b - plane;
        if (idle * 16 <= plane) return b;
        if (idle < idle_best) {
            idle_best = idle;
            best = b;
        }
    }
    return best;
}

// Threads per workgroup that the plane-tile kernels run with for a requested
// block: no more than the plane's wavefronts, since a workgroup stays within a plane.
// Threads then number less than twice the cells, below the 2^32 that HIP takes
// along one dimension of a launch (512 on planes of 64 cells: eight times).
inline int tile_block_in_effect(uint64_t plane, int block)
{
    const uint64_t most = (plane + 63) / 64 * 64;
    return (uint64_t)block > most ? (int)most : block;
}

// Rows per workgroup of the AA odd step's row kernel (tile.h k_tiled_rows)
// for a requested block: as many whole rows as fit it, at least one; 0 where
// the shifted form (k_tiled) serves better:
// - rows that are not a whole number of wavefronts or exceed 512 threads;
// - rows of one wavefront (64x256x256 FP32: 146 us with rows, 140 without);
// - lattices that the 256 MB last-level cache holds a good part of, where the
//   shifted form's second access to a line is cheap (us per AA step, rows /
//   shifted: cavity 128^3 FP64 148 / 146, FP32 78 / 66, TGV 192x80x80 FP64 93 / 85; above
//   512 MiB TGV 512^3 FP64 9580 / 10430, 448x256x256 FP64 2105 / 2355, FP16 513 / 536,
//   cavity 256^3 FP64 1179 / 1327, FP32 594 / 617);
// - the FP16 cavity, whose x walls split the rows' 128-byte lines (320x192x192:
//   257 / 208).
inline uint32_t tile_rows(int nx, int block, uint64_t lattice_bytes, int bc, uint64_t elem)
{
    if (nx % 64 != 0 || nx == 64 || nx > 512) return 0;
    if (lattice_bytes < (uint64_t(512) << 20) || (bc != BC_PERIODIC && elem == 2)) return 0;
    return block > nx ? (uint32_t)(block / nx) : 1u;
}

struct FusedParams {
    int nx, ny, nz;
    uint32_t ncell;          // nx * ny * nz
    uint64_t pstride;        // elements between consecutive populations (structure of arrays)
    LatGeom geom;            // the lattice's layout
    uint32_t bpp;            // plane tiles: workgroups per z plane
    FastDiv divb;            // division by bpp
    const void *src;         // pull: lattice read; AA: the single lattice
    void *dst;               // pull: lattice written; AA: same as src
    double *mom_p, *mom_u, *mom_v, *mom_w;  // written when mom_p != nullptr
    const uint8_t *mask;     // channel: 0 fluid, 1 solid, 2 fluid next to solid
    double tau0;             // f <- f - (f - feq) / (tau0 + 0.5)
    double inv_den;          // FP64: div_reciprocal(tau0 + 0.5)
    float omega_f;           // 1 / (tau0 + 0.5) for the FP32 collision
    double shift;            // reduced precision: S, with sum_i s_i = S (p = (sum g + S) / 3)
    double ush;              // reduced-precision channel: the shift's free-stream x velocity U
                             // (u = sum g e + U); 0 otherwise
    double sh[Q];            // s_i (storage_shift), for the transfer and force kernels
    double corr[Q];          // cavity: moving-lid term for a link crossing z = nz
    double feq_in[Q];        // channel: inlet equilibrium, stored convention
    uint32_t nblocks;        // grid size (for the XCD-aware block order)
    int xcd_remap;           // 1: give each XCD one contiguous run of tiles; plane tiles: tile_order
    int cpt;                 // cells per thread: 1, 2 (blockDim apart) or 3 (two adjacent
                             // x cells; periodic lattices with nx even, else 1)
    int ntl;                 // 1: non-temporal loads of unshared lines; plane tiles: and
                             // stores (0: plain; by whole rows stores are always
                             // non-temporal)
    int am_max;              // widest-saving address mode allowed (AddrMode in fused.h)
    int bc;                  // boundary kind (read by the ensemble kernel)
    FastDiv divx, divy;
    // BC_FAITHFUL: the first ghost layer, population-major (q * ring_n + r).
    // Cell r of the ring: the two x faces (x = -1, nx; y in [-1, ny], z in
    // [-1, nz]; ring_a cells each) first, then the two y faces (y = -1, ny;
    // x in [0, nx), z in [-1, nz]; ring_b each), then the two z faces (z =
    // -1, nz; x in [0, nx), y in [0, ny); ring_c each), each x fastest.
    double *ring;
    int64_t ring_rel;        // (ring - src) in elements: ring loads address from the lattice's base
    uint32_t ring_n, ring_a, ring_b, ring_c;
    int faithful_sphere;     // BC_FAITHFUL: 0 the cavity, 1 the sphere channel
    // faithful mode: the populations the x-face boundary kernels read,
    // written by each fused pass: stage[((side * nz + z) * ny + y) * STAGE_ROW
    // + r] holds, for the cavity's walls, the r-th population with e_x = -1
    // at x = 1 (side 0) or with e_x = +1 at x = nx - 2 (side 1); for the
    // sphere's inlet and outlet copies, the r-th with e_x = +1 at x = 0 (side
    // 0) or with e_x = -1 at x = nx - 1 (side 1); each row's nine together;
    // null elsewhere
    double *stage;
    double u0;               // faithful sphere: inlet speed of the parabolic profile
    uint64_t seed;           // faithful sphere: the initial perturbation's seed
};

// The ring index of ghost cell (i, j, k), -2 for an interior cell and -1 for
// a ghost cell deeper than the first layer (those stay 0 in the faithful
// cavity: nothing writes them and Initialize makes f = 0).
// (selects rather than branches: a kernel's loads stay free of waits)
__host__ __device__ __forceinline__ int64_t ring_index(const FusedParams &P, int i, int j, int k)
{
    const bool deep = i < -1 || i > P.nx || j < -1 || j > P.ny || k < -1 || k > P.nz;
    const bool xf = i == -1 || i == P.nx, yf = j == -1 || j == P.ny, zf = k == -1 || k == P.nz;
    const int64_t rx = (i == P.nx ? (int64_t)P.ring_a : 0) + (int64_t)(k + 1) * (P.ny + 2) + (j + 1);
    const int64_t ry = 2 * (int64_t)P.ring_a + (j == P.ny ? (int64_t)P.ring_b : 0) + (int64_t)(k + 1) * P.nx + i;
    const int64_t rz =
        2 * (int64_t)(P.ring_a + P.ring_b) + (k == P.nz ? (int64_t)P.ring_c : 0) + (int64_t)j * P.nx + i;
    return deep ? -1 : (xf ? rx : (yf ? ry : (zf ? rz : -2)));
}

// Up to four device arrays, one after the other from dst on (pinned host
// memory), each from the next 16-byte unit; at[k] is array k's first unit, at[n] the
// number of units.
struct CopyOut {
    const char *src[4];
    uint64_t bytes[4];
    uint64_t at[5];
    char *dst;
};
hipError_t launch_copy_out(const CopyOut &C, hipStream_t st);

// Streaming's boundary phase on the ring (aux.hip k_faithful_ring), before the
// fused pass: P.ring from the lattice P.src and the last step's ring.
hipError_t launch_faithful_boundaries(const FusedParams &P, const double *last_ring, hipStream_t st);
// Initialize's values for the ring (0 in the cavity)
hipError_t launch_faithful_ring_init(const FusedParams &P, hipStream_t st);
// fills FusedParams::stage from the lattice P.src (after Initialize, set_f)
hipError_t launch_faithful_stage_fill(const FusedParams &P, hipStream_t st);

// The faithful sphere: solid iff (x-c)^2 + (y-c)^2 + (z-c)^2 <= r^2 with the
// integer centre c = (glx - 1) / 8 on every axis and r = (glx - 1) / 64
// (sphere/src/lbm.cpp:238).
__host__ __device__ __forceinline__ bool faithful_sphere_solid(int glx, int x, int y, int z)
{
    const int c = (glx - 1) / 8;
    const int di = x - c, dj = y - c, dk = z - c;
    const double r = (glx - 1) / 64.0;
    return (double)di * (double)di + (double)dj * (double)dj + (double)dk * (double)dk <= r * r;
}

// Storage shift of direction i: FP32/FP16 lattices store g_i = f_i - s_i.
// The TGV and the cavity (U = 0) subtract s_i = w_i S, S = rho0; the open
// channel subtracts its inflow equilibrium feq_i(S/3, (U, 0, 0)) in the
// oracle's evaluation order, so that the stored values are the flow's
// departure from the free stream and the inflow itself is stored as 0.
inline void storage_shift(double S, double U, double out[Q])
{
    const double pin = S * (1.0 / 3.0);
    for (int i = 0; i < Q; ++i) {
        if (U == 0.0) {
            out[i] = w(i) * S;
        } else {
            const double edu = (double)EX[i] * U, udu = U * U, eu2 = edu * edu;
            out[i] = w(i) * pin * 3.0 + w(i) * (3.0 * edu + 4.5 * eu2 - 1.5 * udu);
        }
    }
}

// RN(1 / b) for a divisor the kernels may divide by through its reciprocal
// (fused.h div_by), 0 for one beyond [2^-10, 2^30].
inline double div_reciprocal(double b) { return b >= 0x1p-10 && b <= 0x1p30 ? 1.0 / b : 0.0; }

// Launchers (defined next to their kernels).
hipError_t launch_fused(int dtype, int bc, int pattern, const FusedParams &P, int block, hipStream_t st);

struct InitParams {
    int nx, ny, nz;
    uint32_t ncell;
    LatGeom geom;
    void *dst;               // lattice written (stored convention)
    void *other;             // pull with solid cells: the other lattice, where
                             // only they are written (no step does); or null
    int layout;              // 0 natural (pull), 1 swapped (AA after an even step)
    int kind;                // 0 TGV from the per-axis tables, 1 uniform (u0,0,0)/p0, masked,
                             // 2 the faithful sphere (parabolic inlet profile, seeded perturbation)
    const double *tab;       // TGV: 9 tables [sx cx c2x | sy cy c2y | sz cz c2z]
    double u0, rho0, cs2, p0;
    double sh[Q];            // storage shift s_i
    const uint8_t *mask;
    uint64_t seed;           // kind 2
    double *mom[4];          // p, u, v, w of the initial fields (solid cells: 0);
                             // null: not written
    FastDiv divx, divy;
    uint32_t bpp;            // workgroups of a plane (set by launch_init)
    FastDiv divb;
};
// Threads per workgroup of k_init: 256, over plane tiles no more than the plane's
// wavefronts.  Threads then number less than twice the cells, below the 2^32
// that HIP takes along one dimension of a launch (a subdomain has fewer than
// 2^31 cells); whole workgroups of 256 for each plane reach it at 2^24 planes.
inline uint32_t init_block(const LatGeom &g, uint32_t plane)
{
    return g.tl == 31 || plane > 192 ? 256u : (plane + 63) / 64 * 64;
}
hipError_t launch_init(int dtype, InitParams P, hipStream_t st);

// Copy between the stored lattice (any dtype, pull or AA layout after step
// count parity) and a natural-order FP64 array of post-collision populations.
struct XferParams {
    int nx, ny, nz;
    uint32_t ncell;
    LatGeom geom;
    void *lat;
    double *buf;             // [Q][nz][ny][nx]
    int layout;              // 0 natural, 1 swapped (AA even), 2 streamed (AA odd)
    int bc;                  // periodic or cavity (AA streamed layout needs the rule)
    double sh[Q];            // storage shift s_i
    double corr[Q];
    FastDiv divx, divy;
};
hipError_t launch_get_f(int dtype, const XferParams &P, hipStream_t st);
hipError_t launch_set_f(int dtype, const XferParams &P, hipStream_t st);

// Deterministic FP64 reductions.
hipError_t launch_diag(const double *p, const double *u, const double *v, const double *w,
                       const uint8_t *mask, uint32_t n, double *partials, int nparts,
                       double *out2, hipStream_t st);
hipError_t launch_force(int dtype, const FusedParams &P, double *partials, int nparts,
                        double *out3, hipStream_t st);

hipError_t launch_copy(const double *src, double *dst, size_t n, hipStream_t st);

// Sets the message imexlb_last_error(NULL) returns on this thread (entry
// points without a handle).
void set_call_error(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
// Bandwidth probe `kind` (imexlb_bandwidth_probe) over n doubles; returns the
// number of streams it moves (2 for copies, 1 for read- or write-only), 0 for
// an unknown kind.
int bandwidth_probe_streams(int kind);
hipError_t launch_bandwidth_probe(int kind, const double *src, double *dst, size_t n, int cus, hipStream_t st);

// flags[d] = 1 if the moments mom[4d .. 4d+3] (ncell[d] cells each) are all
// finite, else 0.
hipError_t launch_finite_flags(const double *const *mom, const uint32_t *ncell, int ndom, int32_t *flags,
                               hipStream_t st);

}  // namespace imx

#include <string>

namespace imx {

// Autotuner cache (JSON lines), shared by the single-domain and ensemble tuners.
struct TuneChoice {
    int block, cpt, grid_or_xcd, ntl;
    float ms;
};
std::string tune_key(int device, const char *kind, int dtype, int storage, const std::string &shape);
bool tune_cache_read(const char *path, const std::string &key, TuneChoice &out);
void tune_cache_write(const char *path, const std::string &key, const TuneChoice &c);

}  // namespace imx
