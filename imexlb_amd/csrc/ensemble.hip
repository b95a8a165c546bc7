// Batched ensemble: many independent domains of uneven size and Reynolds
// number advanced by one persistent launch per step, optionally replayed from
// a captured HIP graph.  Each domain is a TGV box (periodic) or a config-mode
// lid-driven cavity; all share one storage type and step in lockstep.
//
// The work list is a table of tiles (domain, first cell); a fixed grid of
// workgroups walks it, workgroup b taking tiles b, b + G, b + 2G, ...  Every
// tile runs the single-domain cell code (fused.h) with that domain's
// parameters, so an ensemble member steps bit for bit as it would alone.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <random>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/imexlb.h"
#include "tile.h"
#include "readback.h"
#include "window.h"
#include "kernels.h"

namespace imx {

struct EnsParams {
    const FusedParams *doms;  // two entries per domain: [2 d + parity]
    const uint2 *tiles;       // (domain, first cell; plane tiles: workgroup of the domain)
    uint32_t t0, ntiles;      // this launch's tiles: [t0, ntiles)
    int order;                // tile.h tile_block_of
    bool nt;                  // kernels.h tile_nt
    int parity;               // pull: which lattice of each pair is read
    int write_moments;
};

template <typename S, int BC, int PAT, int CPT, bool NTL>
__device__ __forceinline__ void tile_run(const FusedParams &P, uint32_t first, bool wm)
{
    using R = typename RealOf<S>::type;
    CellCtx k[CPT];
    R f[CPT][Q];
    const S *at[CPT][Q];
    // every member holds at most 2^28 cells per population
    // (imexlb_ensemble_create checks): 32-bit offsets, grouped populations
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
        cell_setup<BC>(P, first + (uint32_t)r * blockDim.x + threadIdx.x, k[r]);
        if (k[r].live) cell_gather<S, BC, PAT, NTL, AM_GROUP>(P, k[r], f[r], at[r]);
    }
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
        if (!k[r].live) continue;
        cell_collide<S, BC>(P, k[r], f[r], wm);
        cell_scatter<S, BC, PAT, AM_GROUP, PAT == PAT_AA_ODD && CPT == 1>(P, k[r], f[r], at[r]);
    }
}

// The tile and domain tables are not written while the kernel runs: read
// them through the constant address space, so that they come in by scalar
// loads, once per workgroup and tile, instead of vector loads that every use
// of a parameter would wait for.  (The host pass only checks the kernel's
// source; the address space exists on the device side.)
template <typename T>
__device__ __forceinline__ T read_const(const T *p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const __attribute__((address_space(4))) T *)p;
#else
    return *p;
#endif
}

// Persistent over one run of the tile table (or one workgroup per tile, grid
// 0): every workgroup exits after its last tile.  Members in plane tiles
// (TILED: every plane of 512 cells or more) run tile.h's cells, periodic and cavity
// in one launch, the choice being the workgroup's (NT: tile_nt of all of them);
// members in arrays run
// fused.h's, one launch per boundary kind (BC), since both kinds in one kernel
// would hold the registers of the larger.  15 members of 32^3-96^3, us a step: FP32
// pull 243 in arrays with 2048 persistent workgroups (the default before), 233 in
// arrays with one workgroup per tile, 202 in tiles, 196 with one launch for both
// kinds (218 persistent); FP64 pull 475 -> 389, FP16 AA 142 -> 113.
template <typename S, int BC, int PAT, int CPT, bool TILED, bool NT>
__global__ void __launch_bounds__(512) k_ensemble(const EnsParams EP)
{
    const bool wm = EP.write_moments != 0;
    const uint32_t count = EP.ntiles - EP.t0;
    for (uint32_t v = blockIdx.x; v < count; v += gridDim.x) {
        // XCD-aware order (v and blockIdx.x agree mod 8 when the grid is a
        // multiple of 8, as the tuned grids are)
        const uint32_t t = EP.t0 + (TILED ? tile_block_of(EP.order, v, count) : xcd_tile(v, count));
        const uint2 tl = read_const(EP.tiles + t);
        FusedParams P = read_const(EP.doms + 2 * tl.x + (uint32_t)EP.parity);
        if constexpr (TILED) {
            if (!wm) P.mom_p = nullptr;
            const uint32_t z = P.divb.div(tl.y);
            const uint32_t p0 = (tl.y - z * P.bpp) * blockDim.x * CPT + threadIdx.x;
            if (P.bc == BC_PERIODIC) tile_cells<S, BC_PERIODIC, PAT, CPT, NT>(P, z, p0);
            else tile_cells<S, BC_CAVITY, PAT, CPT, NT>(P, z, p0);
        } else {
            tile_run<S, BC, PAT, CPT, NT>(P, tl.y, wm);
        }
    }
}

template <typename S, int BC, int CPT, bool TILED, bool NT>
static hipError_t launch_ens_bc(int pattern, const EnsParams &EP, int grid, int block, hipStream_t st)
{
    if (pattern == PAT_PULL)
        hipLaunchKernelGGL((k_ensemble<S, BC, PAT_PULL, CPT, TILED, NT>), dim3(grid), dim3(block), 0, st, EP);
    else if (pattern == PAT_AA_EVEN)
        hipLaunchKernelGGL((k_ensemble<S, BC, PAT_AA_EVEN, CPT, TILED, NT>), dim3(grid), dim3(block), 0, st, EP);
    else hipLaunchKernelGGL((k_ensemble<S, BC, PAT_AA_ODD, CPT, TILED, NT>), dim3(grid), dim3(block), 0, st, EP);
    return hipGetLastError();
}

template <typename S, int CPT>
static hipError_t launch_ens_cpt(int bc, bool tiled, int pattern, const EnsParams &EP, int grid, int block,
                                 hipStream_t st)
{
    if (tiled && EP.nt) return launch_ens_bc<S, BC_PERIODIC, CPT, true, true>(pattern, EP, grid, block, st);
    if (tiled) return launch_ens_bc<S, BC_PERIODIC, CPT, true, false>(pattern, EP, grid, block, st);
    if (bc == BC_PERIODIC) return launch_ens_bc<S, BC_PERIODIC, CPT, false, true>(pattern, EP, grid, block, st);
    return launch_ens_bc<S, BC_CAVITY, CPT, false, true>(pattern, EP, grid, block, st);
}

static hipError_t launch_ensemble(int dtype, int cpt, int bc, bool tiled, int pattern, const EnsParams &EP, int grid,
                                  int block, hipStream_t st)
{
    if (dtype == DT_F64) return cpt == 2 ? launch_ens_cpt<double, 2>(bc, tiled, pattern, EP, grid, block, st)
                                         : launch_ens_cpt<double, 1>(bc, tiled, pattern, EP, grid, block, st);
    if (dtype == DT_F32) return cpt == 2 ? launch_ens_cpt<float, 2>(bc, tiled, pattern, EP, grid, block, st)
                                         : launch_ens_cpt<float, 1>(bc, tiled, pattern, EP, grid, block, st);
    return cpt == 2 ? launch_ens_cpt<_Float16, 2>(bc, tiled, pattern, EP, grid, block, st)
                    : launch_ens_cpt<_Float16, 1>(bc, tiled, pattern, EP, grid, block, st);
}

}  // namespace imx

using namespace imx;

struct imexlb_ensemble {
    int n = 0, dtype = 0, storage = 0, device = 0;
    hipStream_t stream = nullptr;
    std::vector<imexlb_domain> doms;
    std::vector<FusedParams> hp;         // host copy of the domain table
    FusedParams *dp = nullptr;           // device domain table
    // one run per boundary kind and layout (run_of), the periodic first
    std::vector<uint2> tiles;
    uint32_t bounds[4] = {0, 0, 0, 0};
    uint2 *dtiles = nullptr;
    void *pool = nullptr;                // every lattice, in one allocation
    ChunkedWindow win;                   // the address range pool lies in when a window search placed it
    size_t pool_bytes = 0;
    std::vector<size_t> lat_off;         // offset of each lattice in the pool
    std::vector<void *> lat;             // 2 per domain (second null for AA)
    std::vector<double *> mom;           // 4 per domain
    std::vector<double *> tabs;          // TGV init tables per domain
    int32_t *dflags = nullptr;           // per-domain finite flags (imexlb_ensemble_status)
    double *dummy = nullptr;
    ReadBack back;                       // reads of the members' fields
    int block = 256, cpt = 1, grid = 0, cus = 256;
    int64_t steps = 0, mom_step = -1, cells = 0, device_bytes = 0;
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    int graph_parity = -1;               // step parity the captured pair starts from
    std::string err;
};

static int efail(imexlb_ensemble *e, int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    static thread_local std::string g;
    if (e) e->err = buf;
    else g = buf;
    return code;
}

#define ECHK(e, expr)                                                                             \
    do {                                                                                          \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess) return efail((e), IMEXLB_EHIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

static void drop_graph(imexlb_ensemble *e)
{
    if (e->gexec) (void)hipGraphExecDestroy(e->gexec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    e->gexec = nullptr;
    e->graph = nullptr;
    e->graph_parity = -1;
}

// The run of the tile table a member belongs to.
static int run_of(const FusedParams &P) { return P.geom.tl != 31 ? 0 : P.bc == BC_PERIODIC ? 1 : 2; }

static void build_tiles(imexlb_ensemble *e)
{
    e->tiles.clear();
    const uint32_t tile = (uint32_t)e->block * (uint32_t)e->cpt;
    // largest domains first within each run, so that its tail is made of
    // small work
    std::vector<int> order(e->n);
    for (int d = 0; d < e->n; ++d) order[d] = d;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        const FusedParams &A = e->hp[2 * a], &B = e->hp[2 * b];
        if (run_of(A) != run_of(B)) return run_of(A) < run_of(B);
        if (run_of(A) == 0 && A.bc != B.bc) return A.bc == BC_PERIODIC;
        return A.ncell > B.ncell;
    });
    for (uint32_t &b : e->bounds) b = 0;
    for (int d : order) {
        const FusedParams &A = e->hp[2 * d];
        const uint32_t plane = (uint32_t)A.nx * (uint32_t)A.ny;
        if (A.geom.tl == 31) {
            for (uint32_t c = 0; c < A.ncell; c += tile) e->tiles.push_back(make_uint2((uint32_t)d, c));
        } else {
            const uint32_t bpp = (plane + tile - 1) / tile;
            for (int par = 0; par < 2; ++par) {
                e->hp[2 * d + par].bpp = bpp;
                e->hp[2 * d + par].divb.init(bpp);
            }
            for (uint32_t b = 0; b < bpp * (uint32_t)A.nz; ++b) e->tiles.push_back(make_uint2((uint32_t)d, b));
        }
        for (int r = run_of(A) + 1; r < 4; ++r) e->bounds[r] = (uint32_t)e->tiles.size();
    }
}

static int upload_tables(imexlb_ensemble *e)
{
    if (e->dtiles) (void)hipFree(e->dtiles);
    e->dtiles = nullptr;
    ECHK(e, hipMalloc(&e->dtiles, e->tiles.size() * sizeof(uint2)));
    ECHK(e, hipMemcpy(e->dtiles, e->tiles.data(), e->tiles.size() * sizeof(uint2), hipMemcpyHostToDevice));
    for (auto &P : e->hp) {
        P.cpt = e->cpt;
        const uint32_t tile = (uint32_t)e->block * (uint32_t)e->cpt;
        P.nblocks = (P.ncell + tile - 1) / tile;
    }
    ECHK(e, hipMemcpy(e->dp, e->hp.data(), e->hp.size() * sizeof(FusedParams), hipMemcpyHostToDevice));
    drop_graph(e);
    return IMEXLB_OK;
}

// Point every lattice, and the domain table's src/dst, into `pool`.
static int use_pool(imexlb_ensemble *e, void *pool)
{
    e->pool = pool;
    const bool pull = e->storage == IMEXLB_PULL;
    for (int d = 0; d < e->n; ++d) {
        for (int k = 0; k < (pull ? 2 : 1); ++k) e->lat[2 * d + k] = (char *)pool + e->lat_off[2 * d + k];
        for (int par = 0; par < 2; ++par) {
            FusedParams &P = e->hp[2 * d + par];
            P.src = pull ? e->lat[2 * d + par] : e->lat[2 * d];
            P.dst = pull ? e->lat[2 * d + 1 - par] : e->lat[2 * d];
        }
    }
    return upload_tables(e);
}

static int pattern_of(const imexlb_ensemble *e)
{
    if (e->storage == IMEXLB_PULL) return PAT_PULL;
    return (e->steps % 2 == 0) ? PAT_AA_ODD : PAT_AA_EVEN;
}

// every member's lattice, and their accesses in plane tiles
static uint64_t lattice_bytes(const imexlb_ensemble *e) { return e->pool_bytes / (e->storage == IMEXLB_PULL ? 2 : 1); }
static bool nt_of(const imexlb_ensemble *e)
{
    return tile_nt(lattice_bytes(e), e->storage == IMEXLB_AA, e->dtype == IMEXLB_F64 ? 8 : e->dtype == IMEXLB_F32 ? 4 : 2);
}

static int launch_persistent(imexlb_ensemble *e, int pattern, int parity, bool wm)
{
    EnsParams EP;
    EP.doms = e->dp;
    EP.tiles = e->dtiles;
    EP.parity = parity;
    EP.write_moments = wm ? 1 : 0;
    EP.order = tile_order(lattice_bytes(e), e->storage == IMEXLB_AA);
    EP.nt = nt_of(e);
    // HIP takes fewer than 2^32 work-items along one dimension of a launch
    const int most = (int)(((uint64_t(1) << 32) - 1) / (uint64_t)e->block / 8 * 8);
    // the runs, back to back on the stream
    for (int r = 0; r < 3; ++r) {
        if (e->bounds[r + 1] == e->bounds[r]) continue;
        EP.t0 = e->bounds[r];
        EP.ntiles = e->bounds[r + 1];
        const int count = (int)(EP.ntiles - EP.t0);
        const int grid = std::min(e->grid == 0 ? count : std::min<int>(e->grid, count), most);
        ECHK(e, launch_ensemble(e->dtype, e->cpt, r == 2 ? BC_CAVITY : BC_PERIODIC, r == 0, pattern, EP, grid, e->block,
                                e->stream));
    }
    return IMEXLB_OK;
}

// one step of every domain; per_domain = one single-domain launch each
static int ens_step(imexlb_ensemble *e, bool per_domain, bool wm)
{
    const int pattern = pattern_of(e);
    const int parity = e->storage == IMEXLB_PULL ? (int)(e->steps & 1) : 0;
    if (per_domain) {
        for (int d = 0; d < e->n; ++d) {
            FusedParams P = e->hp[2 * d + parity];
            P.xcd_remap = 0;
            if (P.geom.tl != 31) P.ntl = nt_of(e) ? 1 : 0;
            if (!wm) P.mom_p = P.mom_u = P.mom_v = P.mom_w = nullptr;
            ECHK(e, launch_fused(e->dtype, P.bc, pattern, P, e->block, e->stream));
        }
    } else {
        int rc = launch_persistent(e, pattern, parity, wm);
        if (rc) return rc;
    }
    e->steps++;
    if (wm) e->mom_step = e->steps;
    return IMEXLB_OK;
}

// capture two consecutive steps (a full period of the pull parity and of the
// AA odd/even pair) starting from the current parity
static int capture_pair(imexlb_ensemble *e)
{
    drop_graph(e);
    const int64_t s0 = e->steps;
    ECHK(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    int rc = ens_step(e, false, false);
    if (!rc) rc = ens_step(e, false, false);
    hipGraph_t g = nullptr;
    hipError_t ce = hipStreamEndCapture(e->stream, &g);
    e->steps = s0;  // capture recorded the launches; nothing ran
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (ce != hipSuccess) return efail(e, IMEXLB_EHIP, "hipStreamEndCapture: %s", hipGetErrorString(ce));
    e->graph = g;
    ECHK(e, hipGraphInstantiate(&e->gexec, g, nullptr, nullptr, 0));
    e->graph_parity = (int)(s0 & 1);
    return IMEXLB_OK;
}

extern "C" {

// The ensemble of the batched benchmark: n domains from a 64-bit seed, half
// TGV and half config-mode cavity (alternating), edge from {32,48,64,80,96},
// Re uniform in [50, 1000], lid speed uniform in [0.05, 0.1], TGV U0 = 0.05.
// Drawn with std::mt19937_64 and explicit 53-bit scaling so every platform
// draws the same domains.
int imexlb_ensemble_generate(uint64_t seed, int n, imexlb_domain *out)
{
    if (n < 1 || !out) return IMEXLB_EINVAL;
    std::mt19937_64 rng(seed);
    auto unif = [&]() { return (double)(rng() >> 11) * (1.0 / 9007199254740992.0); };
    static const int edges[5] = {32, 48, 64, 80, 96};
    for (int d = 0; d < n; ++d) {
        imexlb_domain &D = out[d];
        std::memset(&D, 0, sizeof D);
        D.case_id = (d % 2 == 0) ? IMEXLB_CASE_TGV : IMEXLB_CASE_CAVITY;
        const int edge = edges[rng() % 5];
        D.nx = D.ny = D.nz = edge;
        const double re = 50.0 + 950.0 * unif();
        const double lid = 0.05 + 0.05 * unif();
        D.rho0 = 1.0;
        if (D.case_id == IMEXLB_CASE_TGV) {
            D.u0 = 0.05;
            D.lid_u = 0.0;
            D.tau0 = D.u0 * edge / re / (1.0 / 3.0) / 2 / 3.1415926;  // tgv/src/System.cpp:21
        } else {
            D.u0 = 0.0;
            D.lid_u = lid;
            D.tau0 = lid * edge / re / (1.0 / 3.0);  // lid_driven_cavity/src/System.cpp:19, R = edge
        }
    }
    return IMEXLB_OK;
}

int imexlb_ensemble_destroy(imexlb_ensemble *e)
{
    if (!e) return IMEXLB_OK;
    (void)hipSetDevice(e->device);
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    drop_graph(e);
    if (!e->win.empty()) window_destroy(e->win);
    else if (e->pool) (void)hipFree(e->pool);
    for (double *p : e->mom)
        if (p) (void)hipFree(p);
    for (double *p : e->tabs)
        if (p) (void)hipFree(p);
    if (e->dp) (void)hipFree(e->dp);
    if (e->dtiles) (void)hipFree(e->dtiles);
    if (e->dflags) (void)hipFree(e->dflags);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
    return IMEXLB_OK;
}

int imexlb_ensemble_create(const imexlb_domain *doms, int n, int dtype, int storage, int device,
                           imexlb_ensemble **out)
{
    if (!doms || n < 1 || !out || dtype < 0 || dtype > 2 || storage < 0 || storage > 1) return IMEXLB_EINVAL;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return IMEXLB_ENODEV;
    if (device < 0 || device >= ndev) return IMEXLB_EINVAL;
    for (int d = 0; d < n; ++d) {
        const imexlb_domain &D = doms[d];
        if ((D.case_id != IMEXLB_CASE_TGV && D.case_id != IMEXLB_CASE_CAVITY) || D.nx < 2 || D.ny < 2 || D.nz < 2 ||
            (uint64_t)D.nx * D.ny * D.nz >= (1ull << 31) || !(D.tau0 > -0.5))
            return IMEXLB_EINVAL;
    }
    imexlb_ensemble *e = new imexlb_ensemble;
    e->n = n;
    e->dtype = dtype;
    e->storage = storage;
    e->device = device;
    e->doms.assign(doms, doms + n);
    auto bail = [&](int code) {
        imexlb_ensemble_destroy(e);
        return code;
    };
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&e->stream) != hipSuccess) return bail(IMEXLB_EHIP);
    int cus = 256;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0) e->cus = cus;
    const size_t elem = dtype == IMEXLB_F64 ? 8 : (dtype == IMEXLB_F32 ? 4 : 2);
    e->hp.resize(2 * (size_t)n);
    e->lat.assign(2 * (size_t)n, nullptr);
    e->lat_off.assign(2 * (size_t)n, 0);
    // One pool for all lattices, each on a 4 KiB boundary: the step rate
    // depends on where a lattice's pages land, and a single allocation can be
    // swapped for a faster one as a whole (imexlb_ensemble_tune_placement).
    // Plane tiles or, for small planes or where only those fit, arrays with the
    // population stride of the single-domain engine: the cell count rounded up
    // to 256 bytes plus the pad that staggers the 27 streams.
    const int nl = storage == IMEXLB_PULL ? 2 : 1;
    std::vector<uint64_t> pstride(n);
    std::vector<LatGeom> geom(n);
    e->mom.assign(4 * (size_t)n, nullptr);
    auto alloc = [&](bool tiles) {  // the pool and the members' fields
        e->pool_bytes = 0;
        for (int d = 0; d < n; ++d) {
            geom[d] = soa_geom((uint32_t)doms[d].nx, (uint32_t)doms[d].ny, pstride[d]);
            // smaller planes would leave most of a workgroup of 256 idle
            if (tiles && (uint64_t)doms[d].nx * doms[d].ny >= 512)
                tile_geom((uint32_t)doms[d].nx, (uint32_t)doms[d].ny, elem, storage == IMEXLB_AA, geom[d]);
            for (int k = 0; k < nl; ++k) {
                e->lat_off[2 * d + k] = e->pool_bytes;
                e->pool_bytes += ((size_t)lattice_elems(geom[d], (uint32_t)doms[d].nz) * elem + 4095) / 4096 * 4096;
            }
        }
        bool ok = hipMalloc(&e->pool, e->pool_bytes) == hipSuccess;
        if (!ok) e->pool = nullptr;
        for (size_t k = 0; k < e->mom.size() && ok; ++k) {
            const imexlb_domain &D = doms[k / 4];
            ok = hipMalloc(&e->mom[k], (size_t)D.nx * D.ny * D.nz * 8) == hipSuccess;
            if (!ok) e->mom[k] = nullptr;
        }
        if (ok) return true;
        (void)hipGetLastError();
        if (e->pool) (void)hipFree(e->pool);
        e->pool = nullptr;
        for (double *&p : e->mom) {
            if (p) (void)hipFree(p);
            p = nullptr;
        }
        return false;
    };
    for (int d = 0; d < n; ++d) {
        const uint64_t nc = (uint64_t)doms[d].nx * doms[d].ny * doms[d].nz, per = 256 / elem;
        pstride[d] = (nc + per - 1) / per * per + (uint64_t)IMEXLB_DEFAULT_PAD / elem;
        // the member kernels address a group of populations (16 bytes of
        // stride per cell, PopGroup) with 32-bit byte offsets
        if (pstride[d] * 16 > (1ull << 32)) return bail(IMEXLB_EINVAL);
    }
    if (!alloc(true) && !alloc(false)) return bail(IMEXLB_ENOMEM);
    e->device_bytes += (int64_t)e->pool_bytes;
    for (int d = 0; d < n; ++d)
        for (int k = 0; k < nl; ++k) e->lat[2 * d + k] = (char *)e->pool + e->lat_off[2 * d + k];
    e->tabs.assign((size_t)n, nullptr);
    for (int d = 0; d < n; ++d) {
        const imexlb_domain &D = doms[d];
        const uint32_t nc = (uint32_t)((uint64_t)D.nx * D.ny * D.nz);
        e->cells += nc;
        e->device_bytes += 4 * (int64_t)nc * 8;
        for (int par = 0; par < 2; ++par) {
            FusedParams &P = e->hp[2 * d + par];
            std::memset(&P, 0, sizeof P);
            P.nx = D.nx;
            P.ny = D.ny;
            P.nz = D.nz;
            P.ncell = nc;
            P.pstride = pstride[d];
            P.geom = geom[d];
            if (storage == IMEXLB_PULL) {
                P.src = e->lat[2 * d + par];
                P.dst = e->lat[2 * d + 1 - par];
            } else {
                P.src = P.dst = e->lat[2 * d];
            }
            P.mom_p = e->mom[4 * d];
            P.mom_u = e->mom[4 * d + 1];
            P.mom_v = e->mom[4 * d + 2];
            P.mom_w = e->mom[4 * d + 3];
            P.tau0 = D.tau0;
            P.inv_den = div_reciprocal(D.tau0 + 0.5);
            P.omega_f = (float)(1.0 / (D.tau0 + 0.5));
            P.shift = dtype == IMEXLB_F64 ? 0.0 : D.rho0;
            if (dtype != IMEXLB_F64) storage_shift(P.shift, 0.0, P.sh);
            P.bc = D.case_id == IMEXLB_CASE_TGV ? BC_PERIODIC : BC_CAVITY;
            if (D.case_id == IMEXLB_CASE_CAVITY)
                for (int i = 0; i < Q; ++i) P.corr[i] = 6.0 * w(i) * D.rho0 * ((double)EX[i] * D.lid_u);
            P.divx.init(D.nx);
            P.divy.init(D.ny);
        }
        if (D.case_id == IMEXLB_CASE_TGV) {
            std::vector<double> tab(3 * ((size_t)D.nx + D.ny + D.nz));
            size_t o = 0;
            const int ext[3] = {D.nx, D.ny, D.nz};
            for (int a = 0; a < 3; ++a) {
                const int m = ext[a];
                for (int k = 0; k < m; ++k) tab[o + k] = std::sin((double)k / (double)m * 2.0 * PI_REF);
                for (int k = 0; k < m; ++k) tab[o + m + k] = std::cos((double)k / (double)m * 2.0 * PI_REF);
                for (int k = 0; k < m; ++k) tab[o + 2 * m + k] = std::cos((double)k / (double)m * 2.0 * PI_REF * 2.0);
                o += 3 * (size_t)m;
            }
            if (hipMalloc(&e->tabs[d], tab.size() * 8) != hipSuccess) return bail(IMEXLB_ENOMEM);
            if (hipMemcpy(e->tabs[d], tab.data(), tab.size() * 8, hipMemcpyHostToDevice) != hipSuccess)
                return bail(IMEXLB_EHIP);
        }
    }
    if (hipMalloc(&e->dp, e->hp.size() * sizeof(FusedParams)) != hipSuccess) return bail(IMEXLB_ENOMEM);
    if (hipMalloc(&e->dflags, (size_t)n * sizeof(int32_t)) != hipSuccess) return bail(IMEXLB_ENOMEM);
    build_tiles(e);
    if (upload_tables(e)) return bail(IMEXLB_EHIP);
    *out = e;
    return IMEXLB_OK;
}

int imexlb_ensemble_initialize(imexlb_ensemble *e)
{
    if (!e) return IMEXLB_EINVAL;
    ECHK(e, hipSetDevice(e->device));
    for (int d = 0; d < e->n; ++d) {
        const imexlb_domain &D = e->doms[d];
        const FusedParams &F = e->hp[2 * d];
        InitParams P;
        std::memset(&P, 0, sizeof P);
        P.nx = D.nx;
        P.ny = D.ny;
        P.nz = D.nz;
        P.ncell = F.ncell;
        P.geom = F.geom;
        P.dst = e->lat[2 * d];
        P.layout = e->storage == IMEXLB_AA ? 1 : 0;
        P.kind = D.case_id == IMEXLB_CASE_TGV ? 0 : 1;
        P.tab = e->tabs[d];
        P.u0 = D.case_id == IMEXLB_CASE_TGV ? D.u0 : 0.0;
        P.rho0 = D.rho0;
        P.cs2 = 1.0 / 3.0;
        P.p0 = D.rho0 * P.cs2;
        std::memcpy(P.sh, F.sh, sizeof P.sh);
        for (int k = 0; k < 4; ++k) P.mom[k] = e->mom[4 * d + k];
        P.divx.init(D.nx);
        P.divy.init(D.ny);
        ECHK(e, launch_init(e->dtype, P, e->stream));
    }
    ECHK(e, hipStreamSynchronize(e->stream));
    e->steps = 0;
    e->mom_step = 0;  // k_init wrote the initial fields
    return IMEXLB_OK;
}

// mode 0: persistent launch per step; 1: persistent launches replayed from a
// captured graph; 2: one single-domain launch per domain per step.
int imexlb_ensemble_step(imexlb_ensemble *e, int nsteps, int mode, int moments_every)
{
    if (!e || nsteps < 0 || mode < 0 || mode > 2 || moments_every < 0) return IMEXLB_EINVAL;
    ECHK(e, hipSetDevice(e->device));
    int rc;
    int k = 0;
    while (k < nsteps) {
        const int64_t idx = e->steps + 1;
        const bool last = k == nsteps - 1;
        const bool wm = moments_every > 0 && (idx % moments_every == 0 || last);
        if (mode == 1 && !wm && nsteps - k >= 2) {
            // graph pairs until two steps before the next moments step
            const bool wm2 = moments_every > 0 && ((idx + 1) % moments_every == 0 || k + 1 == nsteps - 1);
            if (!wm2) {
                if (e->graph_parity != (int)(e->steps & 1) || !e->gexec) {
                    if ((rc = capture_pair(e))) return rc;
                }
                ECHK(e, hipGraphLaunch(e->gexec, e->stream));
                e->steps += 2;
                k += 2;
                continue;
            }
        }
        if ((rc = ens_step(e, mode == 2, wm))) return rc;
        ++k;
    }
    return IMEXLB_OK;
}

int imexlb_ensemble_step_timed(imexlb_ensemble *e, int nsteps, int mode, int moments_every, float *ms)
{
    if (!e || !ms) return IMEXLB_EINVAL;
    ECHK(e, hipSetDevice(e->device));
    // build the graph outside the timed region
    if (mode == 1 && (e->graph_parity != (int)(e->steps & 1) || !e->gexec)) {
        int rc = capture_pair(e);
        if (rc) return rc;
    }
    hipEvent_t a, b;
    ECHK(e, hipEventCreate(&a));
    ECHK(e, hipEventCreate(&b));
    ECHK(e, hipEventRecord(a, e->stream));
    int rc = imexlb_ensemble_step(e, nsteps, mode, moments_every);
    if (!rc) {
        ECHK(e, hipEventRecord(b, e->stream));
        ECHK(e, hipEventSynchronize(b));
        ECHK(e, hipEventElapsedTime(ms, a, b));
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return rc;
}

int imexlb_ensemble_get_moments(imexlb_ensemble *e, int d, double *p, double *u, double *v, double *w)
{
    if (!e || d < 0 || d >= e->n) return IMEXLB_EINVAL;
    if (e->mom_step != e->steps) return efail(e, IMEXLB_ESTATE, "no moments for step %lld", (long long)e->steps);
    ECHK(e, hipSetDevice(e->device));
    double *out[4] = {p, u, v, w};
    const size_t nb = (size_t)e->hp[2 * d].ncell * 8;
    ReadBack::Part part[4];
    int n = 0;
    for (int k = 0; k < 4; ++k)
        if (out[k]) part[n++] = {out[k], e->mom[4 * d + k], nb};
    ECHK(e, e->back.copy(part, n, e->device, e->stream));
    return IMEXLB_OK;
}

// finite[d] = 1 while domain d's moments of the current step are all finite,
// 0 once the domain has blown up; *unstable = the number of zeros.
int imexlb_ensemble_status(imexlb_ensemble *e, int32_t *finite, int32_t *unstable)
{
    if (!e) return IMEXLB_EINVAL;
    if (e->mom_step != e->steps)
        return efail(e, IMEXLB_ESTATE, "status needs the moments of the current step %lld", (long long)e->steps);
    ECHK(e, hipSetDevice(e->device));
    std::vector<uint32_t> nc(e->n);
    for (int d = 0; d < e->n; ++d) nc[d] = e->hp[2 * d].ncell;
    ECHK(e, launch_finite_flags(e->mom.data(), nc.data(), e->n, e->dflags, e->stream));
    std::vector<int32_t> fl(e->n);
    const ReadBack::Part part{fl.data(), e->dflags, fl.size() * sizeof(int32_t)};
    ECHK(e, e->back.copy(&part, 1, e->device, e->stream));
    int32_t bad = 0;
    for (int d = 0; d < e->n; ++d) {
        bad += fl[d] == 0;
        if (finite) finite[d] = fl[d];
    }
    if (unstable) *unstable = bad;
    return IMEXLB_OK;
}

// out: cells, tiles, grid, block, cells per thread, device bytes, steps
int imexlb_ensemble_info(imexlb_ensemble *e, int64_t *out)
{
    if (!e || !out) return IMEXLB_EINVAL;
    out[0] = e->cells;
    out[1] = (int64_t)e->tiles.size();
    out[2] = e->grid == 0 ? (int64_t)e->tiles.size() : std::min<int64_t>(e->grid, (int64_t)e->tiles.size());
    out[3] = e->block;
    out[4] = e->cpt;
    out[5] = e->device_bytes;
    out[6] = e->steps;
    return IMEXLB_OK;
}

int imexlb_ensemble_set_launch(imexlb_ensemble *e, int block, int cpt, int grid)
{
    if (!e || block < 64 || block > 512 || block % 64 || (cpt != 1 && cpt != 2) || grid < 0) return IMEXLB_EINVAL;
    e->block = block;
    e->cpt = cpt;
    e->grid = grid;
    build_tiles(e);
    return upload_tables(e);
}

// As imexlb_tune_placement for one domain: time graph-replayed steps on the
// current pool and on up to trials - 1 fresh ones (each held until the end,
// so each has its own pages; 2 GiB stay free), keep the fastest, free the
// others and reset the ensemble to its initial state.  The results do not
// depend on the pool.
int imexlb_ensemble_tune_placement(imexlb_ensemble *e, int trials, int steps, float *ms_per_step, int32_t *chosen)
{
    if (!e) return IMEXLB_EINVAL;
    if (trials < 1 || trials > 16) return efail(e, IMEXLB_EINVAL, "placement trials %d must be in [1, 16]", trials);
    ECHK(e, hipSetDevice(e->device));
    if (steps < 2) steps = 2;
    steps += steps & 1;
    std::vector<void *> cand{e->pool};
    ChunkedWindow win0 = std::move(e->win);  // candidate 0 may lie in a window
    e->win = ChunkedWindow{};
    std::vector<float> ms(trials, 0.0f);
    auto time_current = [&](float &out) -> int {
        int r = imexlb_ensemble_initialize(e);
        if (!r) r = imexlb_ensemble_step(e, 2, IMEXLB_ENS_GRAPH, 0);
        if (!r) r = imexlb_ensemble_step_timed(e, steps, IMEXLB_ENS_GRAPH, 0, &out);
        if (!r) out /= (float)steps;
        return r;
    };
    int rc = time_current(ms[0]);
    for (int t = 1; !rc && t < trials; ++t) {
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess || free_b < e->pool_bytes + (2ull << 30)) break;
        void *p = nullptr;
        if (hipMalloc(&p, e->pool_bytes) != hipSuccess) {
            (void)hipGetLastError();
            break;
        }
        cand.push_back(p);
        rc = use_pool(e, p);
        if (!rc) rc = time_current(ms[t]);
    }
    int best = 0;
    if (!rc)
        for (int t = 1; t < (int)cand.size(); ++t)
            if (ms[t] < ms[best]) best = t;
    (void)hipStreamSynchronize(e->stream);
    for (int t = 1; t < (int)cand.size(); ++t)
        if (t != best) (void)hipFree(cand[t]);
    if (best == 0) {
        e->win = std::move(win0);
    } else if (!win0.empty()) {
        e->device_bytes -= (int64_t)win0.held() - (int64_t)e->pool_bytes;
        window_destroy(win0);
    } else {
        (void)hipFree(cand[0]);
    }
    int rc2 = use_pool(e, cand[best]);
    if (!rc2) rc2 = imexlb_ensemble_initialize(e);
    if (rc) return rc;
    if (ms_per_step)
        for (int t = 0; t < trials; ++t) ms_per_step[t] = ms[t];
    if (chosen) *chosen = best;
    return rc2;
}

// As imexlb_tune_placement_window, for the pool that holds every member's
// lattices: the pool slides through one allocation of pool + slack.
int imexlb_ensemble_tune_placement_window(imexlb_ensemble *e, int64_t slack_bytes, int64_t step_bytes, int steps,
                                          float *ms_per_pos, int32_t npos_max, int32_t *chosen)
{
    if (!e) return IMEXLB_EINVAL;
    const int64_t two_mib = 2ll << 20;
    if (step_bytes < two_mib || step_bytes % two_mib || slack_bytes < 0 || slack_bytes % step_bytes)
        return efail(e, IMEXLB_EINVAL, "window step must be a multiple of 2 MiB dividing the slack");
    const int64_t npos = slack_bytes / step_bytes + 1;
    if (npos > 256 || npos > npos_max)
        return efail(e, IMEXLB_EINVAL, "%lld window positions (at most %d)", (long long)npos,
                     std::min(256, (int)npos_max));
    ECHK(e, hipSetDevice(e->device));
    if (steps < 2) steps = 2;
    steps += steps & 1;
    const size_t total = e->pool_bytes + (size_t)slack_bytes;
    size_t free_b = 0, total_b = 0;
    ECHK(e, hipMemGetInfo(&free_b, &total_b));
    if (free_b < total + (2ull << 30))
        return efail(e, IMEXLB_ENOMEM, "window of %zu bytes does not fit (%zu free)", total, free_b);
    // one address range in chunks of physical memory: the chunks the kept
    // offset does not use are given back after the search
    ChunkedWindow w;
    if (window_create(w, e->device, total, (size_t)step_bytes) != hipSuccess) {
        (void)hipGetLastError();
        return efail(e, IMEXLB_ENOMEM, "window of %zu bytes", total);
    }
    char *const big = w.base;
    void *const old_pool = e->pool;
    std::vector<float> ms((size_t)npos, 0.0f);
    int rc = IMEXLB_OK;
    for (int64_t k = 0; k < npos && !rc; ++k) {
        rc = use_pool(e, (char *)big + k * step_bytes);
        if (!rc) rc = imexlb_ensemble_initialize(e);
        if (!rc) rc = imexlb_ensemble_step(e, 2, IMEXLB_ENS_GRAPH, 0);
        if (!rc) rc = imexlb_ensemble_step_timed(e, steps, IMEXLB_ENS_GRAPH, 0, &ms[k]);
        if (!rc) ms[k] /= (float)steps;
    }
    (void)hipStreamSynchronize(e->stream);
    if (rc) {  // keep the pool the ensemble had
        const int rc1 = use_pool(e, old_pool);
        window_destroy(w);
        const int rc2 = rc1 ? rc1 : imexlb_ensemble_initialize(e);
        return rc ? rc : rc2;
    }
    int64_t best = 0;
    for (int64_t k = 1; k < npos; ++k)
        if (ms[k] < ms[best]) best = k;
    if (!e->win.empty()) {
        e->device_bytes -= (int64_t)e->win.held();
        window_destroy(e->win);
    } else {
        e->device_bytes -= (int64_t)e->pool_bytes;
        (void)hipFree(old_pool);
    }
    // the pool stays on the pages it was timed on; the rest goes back
    window_keep(w, (size_t)(best * step_bytes), e->pool_bytes);
    e->device_bytes += (int64_t)w.held();
    e->win = std::move(w);
    rc = use_pool(e, (char *)big + best * step_bytes);
    if (ms_per_pos)
        for (int64_t k = 0; k < npos; ++k) ms_per_pos[k] = ms[k];
    if (chosen) *chosen = (int32_t)best;
    return rc ? rc : imexlb_ensemble_initialize(e);
}

const char *imexlb_ensemble_last_error(const imexlb_ensemble *e) { return e ? e->err.c_str() : ""; }

}  // extern "C"

// ------------------------------------------------------------------ autotuner

namespace imx {

std::string tune_key(int device, const char *kind, int dtype, int storage, const std::string &shape)
{
    hipDeviceProp_t prop;
    std::string arch = "unknown";
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) arch = prop.gcnArchName;
    for (char &c : arch)
        if (c == ' ' || c == '"') c = '_';
    std::ostringstream k;
    k << kind << "|" << arch << "|dt" << dtype << "|st" << storage << "|" << shape;
    return k.str();
}

// JSON lines: {"key": "...", "block": B, "cpt": C, "third": T, "ms": M}
bool tune_cache_read(const char *path, const std::string &key, TuneChoice &out)
{
    if (!path || !*path) return false;
    std::ifstream in(path);
    std::string line;
    bool found = false;
    while (std::getline(in, line)) {
        const std::string pat = "\"key\": \"" + key + "\"";
        if (line.find(pat) == std::string::npos) continue;
        TuneChoice c{};
        const char *s = line.c_str() + line.find(pat) + pat.size();
        if (sscanf(s, ", \"block\": %d, \"cpt\": %d, \"third\": %d, \"ntl\": %d, \"ms\": %f", &c.block, &c.cpt,
                   &c.grid_or_xcd, &c.ntl, &c.ms) == 5) {
            out = c;
            found = true;  // last entry for the key wins
        }
    }
    return found;
}

void tune_cache_write(const char *path, const std::string &key, const TuneChoice &c)
{
    if (!path || !*path) return;
    std::ofstream o(path, std::ios::app);
    o << "{\"key\": \"" << key << "\", \"block\": " << c.block << ", \"cpt\": " << c.cpt << ", \"third\": "
      << c.grid_or_xcd << ", \"ntl\": " << c.ntl << ", \"ms\": " << c.ms << "}\n";
}

}  // namespace imx

extern "C" {

// Time every launch shape (workgroup size x cells per thread x persistent
// grid) for a few graph-replayed steps, keep the fastest, record it in the
// JSON-lines cache at cache_path (NULL = no cache).  A cache hit skips the
// timing.  All shapes give bit-identical results; the ensemble is reset to
// its initial state afterwards.  chosen[3] receives block, cpt, grid.
int imexlb_ensemble_autotune(imexlb_ensemble *e, const char *cache_path, int steps, int32_t *chosen)
{
    if (!e) return IMEXLB_EINVAL;
    ECHK(e, hipSetDevice(e->device));
    std::ostringstream shape;
    // members in plane tiles run another kernel than those in arrays
    int tiled = 0;
    for (int d = 0; d < e->n; ++d) tiled += run_of(e->hp[2 * d]) == 0 ? 1 : 0;
    shape << "ens" << e->n << "_cells" << e->cells << "_tiles" << tiled;
    const std::string key = tune_key(e->device, "ensemble", e->dtype, e->storage, shape.str());
    TuneChoice best{};
    if (!tune_cache_read(cache_path, key, best)) {
        if (steps < 2) steps = 2;
        steps += steps & 1;
        best.ms = 1e30f;
        const int blocks[3] = {128, 256, 512};
        // persistent grids of 4 to 64 workgroups per CU, and 0: one
        // workgroup per tile
        const int grids[6] = {e->cus * 4, e->cus * 8, e->cus * 16, e->cus * 32, e->cus * 64, 0};
        for (int b : blocks)
            for (int c = 1; c <= 2; ++c)
                for (int g : grids) {
                    int rc = imexlb_ensemble_set_launch(e, b, c, g);
                    if (rc) return rc;
                    if ((rc = imexlb_ensemble_step(e, 2, 1, 0))) return rc;  // warm: capture + one replay
                    float ms = 0;
                    if ((rc = imexlb_ensemble_step_timed(e, steps, 1, 0, &ms))) return rc;
                    if (ms < best.ms) best = TuneChoice{b, c, g, 0, ms};
                }
        tune_cache_write(cache_path, key, best);
    }
    int rc = imexlb_ensemble_set_launch(e, best.block, best.cpt, best.grid_or_xcd);
    if (rc) return rc;
    if (chosen) {
        chosen[0] = best.block;
        chosen[1] = best.cpt;
        chosen[2] = best.grid_or_xcd;
    }
    return imexlb_ensemble_initialize(e);
}

}  // extern "C"
