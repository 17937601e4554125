// cnv_stencil7.hip -- 7-point Laplacian / forward-Euler diffusion over the
// ghost-extended blocks of a grid, with the lab assembled on the fly.
//
// Layout of the work: a workgroup owns one x-y plane of one block and marches
// through a chunk of z-planes.  Each plane (plus its one-cell x/y halo, read
// straight from the face-neighbour blocks or filled from the block's BCs) is
// staged in LDS; the z neighbours come from a register queue of planes that is
// loaded two planes ahead, so HBM reads of the next planes overlap the
// arithmetic of the current one.  No lab buffer is ever written to HBM.
//
// Arithmetic follows test/sandbox/Benchmarks/Kernel/Laplacian/Laplacian.cpp
// :125-129 operation for operation: ddx = ihx2*((u[+x] - 2u) + u[-x]), same
// for y and z, lap = (ddx + ddy) + ddz; the Euler update is lap*nu_dt then
// u + that (Block/Field.h:457-512, FieldOperator.h:43-114).  The library is
// compiled with -ffp-contract=off so no step is fused into an FMA and FP64
// results are bit-identical to the CPU evaluation of the same order.
#include "cnv_cols.h"
#include "cnv_march.h"

#include <cstdlib>
#include <map>
#include <tuple>

namespace cnv
{

constexpr int kMaxComp = 8;

struct S7Args {
    const char *u;   // input grid base (component slabs)
    char *out;       // output grid base
    char *lap;       // optional Laplacian grid base
    Geom G;
    int comp_in, comp_out;
    int ncomp;
    int nzc;         // z-chunks per block
    int zchunk;      // planes per chunk
    int tiles_per_comp;
    int has_bc[kMaxComp];
    const DevBCHead *heads[kMaxComp];
    double ih2[3];
    double nudt;
    double *partials;
    double *sumsq;
    // deferred norm of the previous step of a multi-step run: workgroup 0
    // sums prev_n[k] partials (written by the previous launch) into
    // *prev_out[k], k = 0, 1 (unused sets have prev_p[k] == nullptr)
    const double *prev_p[2];
    int prev_n[2];
    double *prev_out[2];
};

template <typename T, int NX, int NY, int WG, int MODE, bool SUMSQ>
__global__ __launch_bounds__(WG) void k_stencil7(const S7Args a)
{
    using S = S7Shape<T, NX, NY, WG>;
    __shared__ alignas(16) T lds[2 * S::PLANE];
    __shared__ double red[WG / 64];

    const int tid = threadIdx.x;
    if (blockIdx.x == 0)
        for (int k = 0; k < 2; ++k)
            if (a.prev_p[k])
                wg_sum_partials<WG>(a.prev_p[k], a.prev_n[k], a.prev_out[k], red);
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int comp = tile / a.tiles_per_comp;
    const int tt = tile - comp * a.tiles_per_comp;
    const long long blk = tt / a.nzc;
    const int zc = tt - (int)blk * a.nzc;
    const int NZ = a.G.n[2];
    const int z0 = zc * a.zchunk;
    const int z1 = min(NZ, z0 + a.zchunk);

    const T *cbase = reinterpret_cast<const T *>(a.u) + (long long)(a.comp_in + comp) * a.G.cstride;
    const T *ub = cbase + blk * a.G.bstride;
    T *ob = reinterpret_cast<T *>(a.out) + (long long)(a.comp_out + comp) * a.G.cstride + blk * a.G.bstride;
    T *lb = MODE == 2 ? reinterpret_cast<T *>(a.lap) + (long long)(a.comp_out + comp) * a.G.cstride +
                            blk * a.G.bstride
                      : nullptr;

    FaceSrc<T> F[6];
    block_faces<T>(a.G, a.heads[comp], a.has_bc[comp], blk, cbase, F);
    double acc = s7_march<T, NX, NY, WG, MODE, SUMSQ>(ub, ob, lb, F, NZ, z0, z1, (T)a.ih2[0], (T)a.ih2[1],
                                                      (T)a.ih2[2], (T)a.nudt, lds);

    if (SUMSQ) {
        // per-tile partial in a fixed wave tree and wave order; the tiles are
        // summed in tile order by k_finalize_sum after this kernel
        for (int o = 32; o > 0; o >>= 1)
            acc += __shfl_xor(acc, o, 64);
        if ((tid & 63) == 0)
            red[tid >> 6] = acc;
        __syncthreads();
        if (tid == 0) {
            double s = 0.0;
            for (int w = 0; w < WG / 64; ++w)
                s += red[w];
            a.partials[tile] = s;
        }
    }
}

// Sum of n partials in a fixed order (one workgroup of 1024 threads): every
// thread issues its loads for a round of 8 before adding them in index order,
// then a fixed wave tree and the waves in order.  Deterministic run to run.
__global__ __launch_bounds__(1024) void k_finalize_sum(const double *__restrict__ partials, int n,
                                                       double *__restrict__ out)
{
    __shared__ double red[16];
    const int tid = threadIdx.x;
    double s = 0.0;
    for (int base = 0; base < n; base += 8 * 1024) {
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int i = base + j * 1024 + tid;
            v[j] = i < n ? partials[i] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            s += v[j];
    }
    for (int o = 32; o > 0; o >>= 1)
        s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0)
        red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < 16; ++w)
            t += red[w];
        *out = t;
    }
}

// Blocks of any shape: a lane per VEC cells of a row and chunk of z planes
// (cnv_cols.h).  BC: some component's blocks carry BC lists.  Bound by load
// latency and the caches' bandwidth (a plane's rows are read three times, the
// row neighbours from L1).  Against one thread per cell with seven scalar
// loads and 64-bit index divisions: 3 x 1.66M FP32 cells in 24^3 blocks 107 ->
// 14 us per step (2.8 TB/s of one read and one write), 2.1M FP64 cells in 8^3
// blocks 41 -> 8.5 us (3.9 TB/s), 13.8M FP64 cells in 40^3 blocks 5.7 TB/s.
template <typename T, int VEC, int MODE, bool SUMSQ, bool BC>
__global__ __launch_bounds__(kColWG) void k_stencil7_cols(const S7Args a, const ColShape s)
{
    using V = VecT<T, VEC>;
    __shared__ double red[kColWG / 64];
    const int tid = threadIdx.x;
    if (wg_index(s.wgs) == 0)
        for (int k = 0; k < 2; ++k)
            if (a.prev_p[k])
                wg_sum_partials<kColWG>(a.prev_p[k], a.prev_n[k], a.prev_out[k], red);
    const ColLane c = col_lane<VEC>(s, a.G);
    double acc = 0.0;
    if (c.on) {
        const int nx = a.G.n[0], ny = a.G.n[1], nz = a.G.n[2];
        const long long nxy = (long long)nx * ny;
        const long long in = c.x0 + (long long)nx * c.y; // within a plane
        const T *cb = reinterpret_cast<const T *>(a.u) + (long long)(a.comp_in + c.comp) * a.G.cstride;
        const T *ub = cb + c.blk * a.G.bstride;
        const DevBCHead *h = nullptr;
        if (BC && a.has_bc[c.comp])
            h = a.heads[c.comp] + c.blk;
        auto nbr = [&](int f) { return cb + c.nbr[f] * a.G.bstride; };
        // the row's neighbours: inside the block, or through the face
        ColNb<T> xm{ub + in - 1, (T)1, false}, xp{ub + in + VEC, (T)1, false};
        ColNb<T> ym{ub + in - nx, (T)1, false}, yp{ub + in + nx, (T)1, false};
        if (c.x0 == 0)
            xm = col_ghost<T, BC>(h, 0, nbr(0) + in + nx - 1, ub + in, ub + in);
        if (c.x0 + VEC == nx)
            xp = col_ghost<T, BC>(h, 1, nbr(1) + in + VEC - nx, ub + in + VEC - 1, ub + in + VEC - 1);
        if (c.y == 0)
            ym = col_ghost<T, BC>(h, 2, nbr(2) + in + nxy - nx, ub + in, ub + in);
        if (c.y == ny - 1)
            yp = col_ghost<T, BC>(h, 3, nbr(3) + in + nx - nxy, ub + in, ub + in);
        const T *top = ub + in + nxy * (nz - 1);
        const V vlo = c.z0 == 0 ? col_load<T, VEC, BC>(col_ghost<T, BC>(h, 4, nbr(4) + in + nxy * (nz - 1), ub + in,
                                                                        ub + in), 0)
                                : load_vec<T, VEC>(ub + in + nxy * (c.z0 - 1));
        auto above = [&](int z) -> V { // plane z >= 1 of the column
            return z < nz ? load_vec<T, VEC>(ub + in + nxy * z)
                          : col_load<T, VEC, BC>(col_ghost<T, BC>(h, 5, nbr(5) + in, top, top), 0);
        };
        const T ihx2 = (T)a.ih2[0], ihy2 = (T)a.ih2[1], ihz2 = (T)a.ih2[2], nudt = (T)a.nudt;
        T *ob = reinterpret_cast<T *>(a.out) + (long long)(a.comp_out + c.comp) * a.G.cstride + c.blk * a.G.bstride + in;
        T *lb = MODE == 2 ? reinterpret_cast<T *>(a.lap) + (long long)(a.comp_out + c.comp) * a.G.cstride +
                                c.blk * a.G.bstride + in
                          : nullptr;
        // planes z - 1, z, z + 1 of the column and the neighbours of plane z
        // in registers; those of the next plane are loaded before plane z is
        // evaluated
        V um = vlo, uc = load_vec<T, VEC>(ub + in + nxy * c.z0), up = above(c.z0 + 1);
        long long o = nxy * c.z0;
        V vym = col_load<T, VEC, BC>(ym, o), vyp = col_load<T, VEC, BC>(yp, o);
        T vxm = col_load1<T, BC>(xm, o), vxp = col_load1<T, BC>(xp, o);
        for (int z = c.z0; z < c.z1; ++z, o += nxy) {
            V un_ = up, nym = vym, nyp = vyp;
            T nxm = vxm, nxp = vxp;
            if (z + 1 < c.z1) {
                un_ = above(z + 2);
                nym = col_load<T, VEC, BC>(ym, o + nxy);
                nyp = col_load<T, VEC, BC>(yp, o + nxy);
                nxm = col_load1<T, BC>(xm, o + nxy);
                nxp = col_load1<T, BC>(xp, o + nxy);
            }
            V res, lapv;
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                const T m = uc.v[v];
                const T l = v == 0 ? vxm : uc.v[v - 1], r = v == VEC - 1 ? vxp : uc.v[v + 1];
                const T ddx = ihx2 * (fms2(m, r) + l);
                const T ddy = ihy2 * (fms2(m, vyp.v[v]) + vym.v[v]);
                const T ddz = ihz2 * (fms2(m, up.v[v]) + um.v[v]);
                const T lap = ddx + ddy + ddz;
                lapv.v[v] = lap;
                if (MODE == 0) {
                    res.v[v] = lap;
                } else {
                    const T dl = lap * nudt;
                    const T un = m + dl;
                    res.v[v] = un;
                    if (SUMSQ)
                        acc = __builtin_fma((double)un, (double)un, acc);
                }
            }
            store_vec<T, VEC>(ob + o, res);
            if (MODE == 2)
                store_vec<T, VEC>(lb + o, lapv);
            um = uc;
            uc = up;
            up = un_;
            vym = nym;
            vyp = nyp;
            vxm = nxm;
            vxp = nxp;
        }
    }
    if (SUMSQ) {
        for (int o = 32; o > 0; o >>= 1)
            acc += __shfl_xor(acc, o, 64);
        if ((tid & 63) == 0)
            red[tid >> 6] = acc;
        __syncthreads();
        if (tid == 0)
            a.partials[wg_index(s.wgs)] = ((red[0] + red[1]) + red[2]) + red[3];
    }
}

// ---------------------------------------------------------------- host side

// Tile choice per (dtype, block edge): workgroup size and z-planes per tile.
struct S7Tune {
    int wg;
    int zchunk;
};

static std::mutex g_tune_mtx;
static std::map<std::tuple<int, int>, S7Tune> g_tune; // (dtype, edge) -> choice

// The tile in use; pinned: set to something else than the built-in one.
S7Tune s7_default_tune(int dtype, int edge, bool *pinned = nullptr)
{
    S7Tune d{64, 8};
    if (edge >= 64)
        d = {512, 16};
    else if (edge >= 32)
        d = {256, 8};
    else if (dtype == CNV_F64)
        d = {128, 8};
    std::lock_guard<std::mutex> lk(g_tune_mtx);
    auto it = g_tune.find({dtype, edge});
    const S7Tune t = it == g_tune.end() ? d : it->second;
    if (pinned)
        *pinned = t.wg != d.wg || t.zchunk != d.zchunk;
    return t;
}

void s7_set_tune(int dtype, int edge, int wg, int zchunk)
{
    std::lock_guard<std::mutex> lk(g_tune_mtx);
    g_tune[{dtype, edge}] = {wg, zchunk};
}

template <typename T, int NX, int WG>
constexpr bool s7_valid()
{
    return S7Shape<T, NX, NX, WG>::valid;
}

template <typename T, int NX, int WG, int MODE, bool SUMSQ>
static bool launch_spec(const S7Args &a, int ntiles, hipStream_t st)
{
    if constexpr (s7_valid<T, NX, WG>()) {
        hipLaunchKernelGGL((k_stencil7<T, NX, NX, WG, MODE, SUMSQ>), dim3(ntiles), dim3(WG), 0, st, a);
        return true;
    }
    return false;
}

template <typename T, int NX, int MODE, bool SUMSQ>
static bool dispatch_wg(const S7Args &a, int wg, int ntiles, hipStream_t st)
{
    switch (wg) {
    case 64:
        return launch_spec<T, NX, 64, MODE, SUMSQ>(a, ntiles, st);
    case 128:
        return launch_spec<T, NX, 128, MODE, SUMSQ>(a, ntiles, st);
    case 256:
        return launch_spec<T, NX, 256, MODE, SUMSQ>(a, ntiles, st);
    case 512:
        return launch_spec<T, NX, 512, MODE, SUMSQ>(a, ntiles, st);
    default:
        return false;
    }
}

template <typename T, int MODE, bool SUMSQ>
static bool dispatch_spec(const S7Args &a, int edge, int wg, int ntiles, hipStream_t st)
{
    switch (edge) {
    case 16:
        return dispatch_wg<T, 16, MODE, SUMSQ>(a, wg, ntiles, st);
    case 32:
        return dispatch_wg<T, 32, MODE, SUMSQ>(a, wg, ntiles, st);
    case 64:
        return dispatch_wg<T, 64, MODE, SUMSQ>(a, wg, ntiles, st);
    default:
        return false;
    }
}

template <typename T, int VEC, int MODE, bool SUMSQ>
static void launch_cols(const S7Args &a, const ColShape &s, bool bc, hipStream_t st)
{
    if (bc)
        hipLaunchKernelGGL((k_stencil7_cols<T, VEC, MODE, SUMSQ, true>), s.wgs.dim(), dim3(kColWG), 0, st, a, s);
    else
        hipLaunchKernelGGL((k_stencil7_cols<T, VEC, MODE, SUMSQ, false>), s.wgs.dim(), dim3(kColWG), 0, st, a, s);
}

// The sizes the column kernel takes: gx groups of 256 cells per block, gy blocks
// of all components.
static int check_cols(const Geom &G, int ncomp, long long *gx, long long *gy)
{
    *gx = ((long long)G.n[0] * G.n[1] * G.n[2] + 255) / 256;
    *gy = (long long)G.nb[0] * G.nb[1] * G.nb[2] * ncomp;
    if (*gy > 65535 || *gx > 65535)
        return fail(CNV_ERR_UNSUPPORTED, "grid too large for the generic stencil kernel");
    return CNV_OK;
}

// The column kernel on blocks of any shape.
template <typename T, int MODE, bool SUMSQ>
static int run_cols(S7Args &a, int ncomp, hipStream_t st, bool finalize, int *nparts, long long cap)
{
    const int *n = a.G.n;
    long long gx = 0, gy = 0;
    const int rc = check_cols(a.G, ncomp, &gx, &gy);
    if (rc != CNV_OK)
        return rc;
    if (SUMSQ && cap > 0 && gx * gy > cap)
        return fail(CNV_ERR_SIZE, "grid needs more norm partials than the scratch array holds");
    const int vec = col_vec(n[0], sizeof(T));
    ColShape s;
    if (!col_shape(a.G, ncomp, vec, col_zchunk(a.G, ncomp, vec), s))
        return fail(CNV_ERR_UNSUPPORTED, "grid too large for the generic stencil kernel");
    bool bc = false;
    for (int c = 0; c < ncomp; ++c)
        bc = bc || a.has_bc[c];
    if (vec == 1)
        launch_cols<T, 1, MODE, SUMSQ>(a, s, bc, st);
    else if (vec == 2)
        launch_cols<T, 2, MODE, SUMSQ>(a, s, bc, st);
    else if constexpr (sizeof(T) == 4)
        launch_cols<T, 4, MODE, SUMSQ>(a, s, bc, st);
    CNV_HIP(hipGetLastError());
    if (nparts)
        *nparts = s.wgs.count;
    if (SUMSQ && finalize) {
        hipLaunchKernelGGL(k_finalize_sum, dim3(1), dim3(1024), 0, st, a.partials, s.wgs.count, a.sumsq);
        CNV_HIP(hipGetLastError());
    }
    return CNV_OK;
}

// Grids of 16, 32 or 64 cells per x/y edge run as columns up to 40 MB of
// input unless a tile is pinned: the marching tiles step through 8 or 16
// planes one after another, and on a small grid too few of them run at once
// to cover that chain's latency.  Per Euler step with its norm (marching
// tile / columns): 64^3 FP64 in 16^3 blocks 10.9 / 6.1 us, 128^3 FP64 in 32^3
// blocks 15.1 / 11.7, 64^3 FP32 in one 64^3 block 19.7 / 5.3, 192^3 FP32 (28
// MB) 17.6 / 16.9 in 32^3 and 23.7 / 17.3 in 64^3 blocks; 192^3 FP64 (57 MB)
// 28.6 / 26.1 in 16^3 but 24.2 / 25.3 in 32^3 blocks, and 256^3 FP64 49.9 /
// 59.2.
static bool cols_for_small(const Geom &G, int ncomp, size_t elem)
{
    const long long cells = (long long)G.nb[0] * G.nb[1] * G.nb[2] * ncomp * G.n[0] * G.n[1] * G.n[2];
    return cells * (long long)elem < 40ll * 1000 * 1000;
}

static bool march_edge(const int n[3]) { return n[0] == n[1] && (n[0] == 16 || n[0] == 32 || n[0] == 64); }

// cap: partials the buffer at a.partials holds (0: sized by the caller for
// the largest launch)
template <typename T, int MODE, bool SUMSQ>
static int run_t(S7Args &a, int ncomp, hipStream_t st, int force_generic, const S7Tune *over, bool finalize,
                 int *nparts, long long cap = 0)
{
    const int *n = a.G.n;
    const long long nbt = (long long)a.G.nb[0] * a.G.nb[1] * a.G.nb[2];
    if (!force_generic && march_edge(n)) {
        bool pinned = false;
        S7Tune tu = over ? *over : s7_default_tune(sizeof(T) == 8 ? CNV_F64 : CNV_F32, n[0], &pinned);
        if (!over && !pinned && cols_for_small(a.G, ncomp, sizeof(T)))
            return run_cols<T, MODE, SUMSQ>(a, ncomp, st, finalize, nparts, cap);
        a.zchunk = tu.zchunk < n[2] ? tu.zchunk : n[2];
        a.nzc = (n[2] + a.zchunk - 1) / a.zchunk;
        a.tiles_per_comp = (int)(nbt * a.nzc);
        const long long ntiles = (long long)a.tiles_per_comp * ncomp;
        if (SUMSQ && cap > 0 && ntiles > cap)
            return fail(CNV_ERR_SIZE, "grid needs more norm partials than the scratch array holds");
        if (ntiles < (1LL << 31)) {
            if (dispatch_spec<T, MODE, SUMSQ>(a, n[0], tu.wg, (int)ntiles, st)) {
                CNV_HIP(hipGetLastError());
                if (nparts)
                    *nparts = (int)ntiles;
                if (SUMSQ && finalize) {
                    hipLaunchKernelGGL(k_finalize_sum, dim3(1), dim3(1024), 0, st, a.partials, (int)ntiles, a.sumsq);
                    CNV_HIP(hipGetLastError());
                }
                return CNV_OK;
            }
            if (over)
                return fail(CNV_ERR_UNSUPPORTED, "tile shape not available for this block edge and dtype");
        }
    }
    return run_cols<T, MODE, SUMSQ>(a, ncomp, st, finalize, nparts, cap);
}

static int g_force_generic = -1;

static bool force_generic()
{
    if (g_force_generic < 0) {
        const char *e = getenv("CNV_STENCIL7_GENERIC");
        g_force_generic = (e && e[0] == '1') ? 1 : 0;
    }
    return g_force_generic == 1;
}

// Host check that every face the operator reads is written by the lab rules
// (the caller holds the grid's mutex).
static int check_faces(cnv_grid_s *g, int comp)
{
    const FaceInfo &f = face_info(g, comp);
    if (f.longest > 64)
        return fail(CNV_ERR_UNSUPPORTED, "BC list too long");
    if (f.unset)
        return fail(CNV_ERR_UNSUPPORTED, "BC list leaves ghost cells of a face unwritten for Stencil(-1,2)");
    return CNV_OK;
}

// What a single step refuses on a grid, before any launch.
static int check_components(const cnv_grid_s *u, int ncomp)
{
    if (ncomp > kMaxComp)
        return fail(CNV_ERR_UNSUPPORTED, "more than 8 components in one stencil call");
    for (int d = 0; d < 3; ++d)
        if (u->desc.block_cells[d] < 1)
            return fail(CNV_ERR_INVALID, "empty block");
    return CNV_OK;
}

static int check_step(cnv_grid_s *u)
{
    int rc = check_components(u, u->desc.ncomp);
    for (int c = 0; rc == CNV_OK && c < u->desc.ncomp; ++c) {
        std::lock_guard<std::mutex> lk(u->mtx);
        rc = check_faces(u, c);
    }
    long long gx, gy;
    if (rc == CNV_OK && (force_generic() || !march_edge(u->desc.block_cells)))
        rc = check_cols(geom_of(u), u->desc.ncomp, &gx, &gy);
    return rc;
}

// State of one launch inside a multi-step run (cnv_diffusion_run).
struct S7Run {
    double *partials;          // this launch's partial buffer
    const double *prev[2];     // the previous launch's partial sets, summed by workgroup 0
    int prev_n[2];
    double *prev_out[2];
    int *nparts;               // out: partials written per set by this launch
    size_t cap;                // capacity of each buffer half
};

// Partials of a launch that owns no grid scratch: `cap` doubles at `p`.
struct S7Scratch {
    double *p;
    long long cap;
};

static int launch_stencil7_t(cnv_grid_s *u, cnv_grid_s *out, cnv_grid_s *lap, int comp_in, int comp_out,
                             int ncomp, int mode, double nu_dt, double *sumsq, hipStream_t st,
                             const S7Tune *over, const S7Run *run = nullptr, const S7Scratch *scr = nullptr)
{
    const int bad = check_components(u, ncomp);
    if (bad != CNV_OK)
        return bad;
    S7Args a;
    a.u = static_cast<const char *>(u->data);
    a.out = static_cast<char *>(out->data);
    a.lap = lap ? static_cast<char *>(lap->data) : nullptr;
    a.G = geom_of(u);
    a.comp_in = comp_in;
    a.comp_out = comp_out;
    a.ncomp = ncomp;
    for (int c = 0; c < ncomp; ++c) {
        a.has_bc[c] = 0;
        a.heads[c] = nullptr;
    }
    if (!u->tables.empty()) { // a grid without tables is periodic on every face
        std::lock_guard<std::mutex> lk(u->mtx);
        for (int c = 0; c < ncomp; ++c) {
            int rc = ensure_bc_table(u, comp_in + c);
            if (rc != CNV_OK)
                return rc;
            rc = check_faces(u, comp_in + c);
            if (rc != CNV_OK)
                return rc;
            const BCTable &t = u->tables[comp_in + c];
            a.has_bc[c] = (t.any && t.heads) ? 1 : 0;
            a.heads[c] = t.heads;
        }
    }
    for (int c = ncomp; c < kMaxComp; ++c) {
        a.has_bc[c] = 0;
        a.heads[c] = nullptr;
    }
    for (int d = 0; d < 3; ++d)
        a.ih2[d] = 1. / (u->h[d] * u->h[d]);
    a.nudt = nu_dt;
    a.sumsq = sumsq;
    a.partials = nullptr;
    for (int k = 0; k < 2; ++k) {
        a.prev_p[k] = run ? run->prev[k] : nullptr;
        a.prev_n[k] = run ? run->prev_n[k] : 0;
        a.prev_out[k] = run ? run->prev_out[k] : nullptr;
    }
    a.zchunk = a.nzc = a.tiles_per_comp = 0;
    if (sumsq) {
        const long long nbt = u->nblocks_total;
        const long long cells = (long long)u->desc.block_cells[0] * u->desc.block_cells[1] * u->desc.block_cells[2];
        // upper bound on workgroups: generic kernel uses ceil(cells/256) per block
        const long long need = nbt * ncomp * ((cells + 255) / 256 + u->desc.block_cells[2]);
        if (run) { // fixed buffer halves: never reallocated inside a run
            if (need > (long long)run->cap)
                return fail(CNV_ERR_SIZE, "partial buffer too small for this run");
            a.partials = run->partials;
        } else if (scr) { // fixed scratch, checked against the launch's own tile count in run_t
            a.partials = scr->p;
        } else {
            int rc = ensure_partials(u, (size_t)need);
            if (rc != CNV_OK)
                return rc;
            a.partials = u->partials;
        }
    }
    const bool gen = over ? false : force_generic();
    const bool fin = run == nullptr;
    int *np = run ? run->nparts : nullptr;
    const bool dbl = u->desc.dtype == CNV_F64;
    if (scr) { // the one-step Euler update with its norm (the allocation-free entry point)
        if (mode != 1 || !sumsq)
            return fail(CNV_ERR_INVALID, "scratch partials serve the Euler step with a norm only");
        return dbl ? run_t<double, 1, true>(a, ncomp, st, gen, over, true, nullptr, scr->cap)
                   : run_t<float, 1, true>(a, ncomp, st, gen, over, true, nullptr, scr->cap);
    }
    if (mode == 0)
        return dbl ? run_t<double, 0, false>(a, ncomp, st, gen, over, fin, np)
                   : run_t<float, 0, false>(a, ncomp, st, gen, over, fin, np);
    if (mode == 1) {
        if (sumsq)
            return dbl ? run_t<double, 1, true>(a, ncomp, st, gen, over, fin, np)
                       : run_t<float, 1, true>(a, ncomp, st, gen, over, fin, np);
        return dbl ? run_t<double, 1, false>(a, ncomp, st, gen, over, fin, np)
                   : run_t<float, 1, false>(a, ncomp, st, gen, over, fin, np);
    }
    if (sumsq)
        return dbl ? run_t<double, 2, true>(a, ncomp, st, gen, over, fin, np)
                   : run_t<float, 2, true>(a, ncomp, st, gen, over, fin, np);
    return dbl ? run_t<double, 2, false>(a, ncomp, st, gen, over, fin, np)
               : run_t<float, 2, false>(a, ncomp, st, gen, over, fin, np);
}

int launch_stencil7(cnv_grid_s *u, cnv_grid_s *out, cnv_grid_s *lap, int comp_in, int comp_out,
                    int ncomp, int mode, double nu_dt, double *sumsq, hipStream_t st)
{
    return launch_stencil7_t(u, out, lap, comp_in, comp_out, ncomp, mode, nu_dt, sumsq, st, nullptr);
}

// ------------------------------------------------ allocation-free Euler step
//
// The per-tile FP64 partials of the norm of cnv_diffusion_step_noalloc live
// in `scratch`, a static device array (one copy per GPU, held until the
// process ends).  Host code never passes the array's name to a kernel: on
// the host it is a stand-in, not a device address.  The first call on a
// device looks up that device's address of the array with
// hipGetSymbolAddress, and every launch takes it from g_scratch_dev.  Each
// launch writes every partial it reads before the finalize kernel reads it,
// so nothing needs clearing between calls; calls that overlap on one GPU
// share the array and race.
constexpr long long kNoAllocPartials = 1LL << 17; // 1 MiB of doubles
static __device__ __align__(256) double scratch[kNoAllocPartials];
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mtx;
static double *g_scratch_dev[kMaxDevices] = {};

static int scratch_partials(double **out)
{
    int dev = -1;
    CNV_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return fail(CNV_ERR_UNSUPPORTED, "device index out of range for the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mtx);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return hip_fail(e, "hipGetSymbolAddress(scratch)");
        g_scratch_dev[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_dev[dev];
    return CNV_OK;
}

int launch_diffusion_noalloc(const cnv_grid_desc *desc, const void *u, void *u_new, double nu_dt, double *sumsq,
                             hipStream_t st)
{
    // grid objects on the stack over the caller's memory: layout fields
    // only, no BC lists or tables (every face periodic), no partials
    cnv_grid_s gu, go;
    int rc = grid_layout(desc, &gu);
    if (rc != CNV_OK)
        return rc;
    if (desc->entity != CNV_CELL)
        return fail(CNV_ERR_UNSUPPORTED, "the stencil operators take cell grids only");
    (void)grid_layout(desc, &go);
    gu.data = const_cast<void *>(u);
    go.data = u_new;
    gu.owns_data = go.owns_data = false;
    if (grids_overlap(&gu, &go))
        return fail(CNV_ERR_INVALID, "u and u_new must not overlap");
    if (!sumsq)
        return launch_stencil7_t(&gu, &go, nullptr, 0, 0, desc->ncomp, 1, nu_dt, nullptr, st, nullptr);
    S7Scratch scr{nullptr, kNoAllocPartials};
    rc = scratch_partials(&scr.p);
    if (rc != CNV_OK)
        return rc;
    return launch_stencil7_t(&gu, &go, nullptr, 0, 0, desc->ncomp, 1, nu_dt, sumsq, st, nullptr, nullptr, &scr);
}

// ---------------------------------------------------------------- autotuner

// Times every (workgroup size, z-planes per tile) candidate of the fused
// diffusion step (with the FP64 norm) on u -> out and keeps the fastest for
// (dtype, block edge).  Candidates that the block shape cannot take are
// skipped by the dispatcher's validity check.
int autotune_stencil7(cnv_grid_s *u, cnv_grid_s *out, int iters, int *best_wg, int *best_z, double *results,
                      int max_results, int *nresults)
{
    const int *n = u->desc.block_cells;
    if (!(n[0] == n[1] && (n[0] == 16 || n[0] == 32 || n[0] == 64)))
        return fail(CNV_ERR_UNSUPPORTED, "autotuning needs x/y block edges of 16, 32 or 64");
    if (iters < 1)
        return fail(CNV_ERR_INVALID, "iters must be >= 1");
    hipStream_t st;
    CNV_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    double *norm = nullptr;
    hipEvent_t e0, e1;
    CNV_HIP(hipMalloc((void **)&norm, sizeof(double)));
    CNV_HIP(hipEventCreate(&e0));
    CNV_HIP(hipEventCreate(&e1));
    const int wgs[4] = {64, 128, 256, 512};
    const int zcs[6] = {2, 4, 8, 16, 32, 64};
    float best = 1e30f;
    int bw = 0, bz = 0, cnt = 0;
    int rc = CNV_OK;
    for (int wi = 0; wi < 4 && rc == CNV_OK; ++wi)
        for (int zi = 0; zi < 6 && rc == CNV_OK; ++zi) {
            if (zcs[zi] > n[2])
                continue;
            S7Tune tu{wgs[wi], zcs[zi]};
            int r = launch_stencil7_t(u, out, nullptr, 0, 0, u->desc.ncomp, 1, 1e-9, norm, st, &tu);
            if (r == CNV_ERR_UNSUPPORTED)
                continue;
            if (r != CNV_OK) {
                rc = r;
                break;
            }
            (void)hipEventRecord(e0, st);
            for (int i = 0; i < iters; ++i)
                (void)launch_stencil7_t(u, out, nullptr, 0, 0, u->desc.ncomp, 1, 1e-9, norm, st, &tu);
            (void)hipEventRecord(e1, st);
            if (hipEventSynchronize(e1) != hipSuccess) {
                rc = fail(CNV_ERR_HIP, "autotune: kernel failed");
                break;
            }
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            const float us = ms * 1000.f / iters;
            if (results && cnt < max_results) {
                results[3 * cnt] = tu.wg;
                results[3 * cnt + 1] = tu.zchunk;
                results[3 * cnt + 2] = us;
            }
            ++cnt;
            if (us < best) {
                best = us;
                bw = tu.wg;
                bz = tu.zchunk;
            }
        }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(norm);
    (void)hipStreamDestroy(st);
    if (rc != CNV_OK)
        return rc;
    if (bw == 0)
        return fail(CNV_ERR_UNSUPPORTED, "no tile candidate ran");
    s7_set_tune(u->desc.dtype, n[0], bw, bz);
    if (best_wg)
        *best_wg = bw;
    if (best_z)
        *best_z = bz;
    if (nresults)
        *nresults = cnt < max_results ? cnt : max_results;
    return CNV_OK;
}

int get_tune_stencil7(int dtype, int edge, int *wg, int *zchunk)
{
    S7Tune t = s7_default_tune(dtype, edge);
    *wg = t.wg;
    *zchunk = t.zchunk;
    return CNV_OK;
}

// ---------------------------------------------------------------- sums
//
// Whole-component reductions run over chunks of 1024 16-byte vectors of a
// block (four per thread, loaded before they are added), so a grid of few
// large blocks fills the GPU like one of many small ones; the partials of all
// results are summed by one launch.  Bound by HBM: 16.8M FP32 cells in 64
// blocks of 64^3 cells take 18 us (sum and sum of squares), 416 us when a
// workgroup took whole blocks.

constexpr int kRedMaxWG = 2048; // workgroups at most: 3 * 2048 partials fit the scratch of any grid
constexpr int kRedVec = 1024;   // vectors per chunk

// Workgroup partials in a fixed wave tree and wave order; result valid in thread 0.
template <typename F>
__device__ inline double red_wg(double v, double *red, F &&f)
{
    for (int o = 32; o > 0; o >>= 1)
        v = f(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = v;
    __syncthreads();
    return f(f(f(red[0], red[1]), red[2]), red[3]);
}

// Result k of gridDim.x from its n partials at partials + k n: the maximum
// for k == kmax, the sum else.
__global__ __launch_bounds__(1024) void k_finalize_red(const double *__restrict__ partials, int n,
                                                       double *__restrict__ out, int kmax)
{
    __shared__ double red[16];
    const int tid = threadIdx.x, k = blockIdx.x;
    const bool mx = k == kmax;
    double s = 0.0;
    for (int i = tid; i < n; i += 1024) {
        const double v = partials[(size_t)k * n + i];
        s = mx ? fmax(s, v) : s + v;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double v = __shfl_xor(s, o, 64);
        s = mx ? fmax(s, v) : s + v;
    }
    if ((tid & 63) == 0)
        red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < 16; ++w)
            t = mx ? fmax(t, red[w]) : t + red[w];
        out[k] = t;
    }
}

// f(block, e) for every chunk of the workgroup: this thread's vectors start at
// elements e + j 256 VEC of the block, j = 0..3
template <int VEC, typename F>
__device__ inline void red_chunks(int cpb, long long nchunks, F &&f)
{
    for (long long ch = blockIdx.x; ch < nchunks; ch += gridDim.x) {
        const long long blk = ch / cpb;
        f(blk, ((ch - blk * cpb) * kRedVec + threadIdx.x) * VEC);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_sums(const T *p, long long bstride, long long cells, int cpb,
                                                long long nchunks, double *partials)
{
    constexpr int VEC = 16 / (int)sizeof(T);
    __shared__ double red[4];
    double s = 0.0, q = 0.0;
    red_chunks<VEC>(cpb, nchunks, [&](long long blk, long long e0) {
        const T *pb = p + blk * bstride;
        if (e0 + 3 * 256 * VEC + VEC <= cells) {
            VecT<T, VEC> v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = load_vec<T, VEC>(pb + e0 + j * 256 * VEC);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const double x = (double)v[j].v[k];
                    s += x;
                    q = __builtin_fma(x, x, q);
                }
        } else {
            for (int j = 0; j < 4; ++j)
                for (int k = 0; k < VEC; ++k)
                    if (e0 + j * 256 * VEC + k < cells) {
                        const double x = (double)pb[e0 + j * 256 * VEC + k];
                        s += x;
                        q = __builtin_fma(x, x, q);
                    }
        }
    });
    auto add = [](double a, double b) { return a + b; };
    s = red_wg(s, red, add);
    q = red_wg(q, red, add);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = s;
        partials[gridDim.x + blockIdx.x] = q;
    }
}

// Chunks per block, chunks and workgroups of a component of 16-byte vectors
// of `elem`-byte elements.
struct RedShape {
    long long cells, nchunks;
    int cpb, nwg;
};

static RedShape red_shape(const cnv_grid_s *g, size_t elem)
{
    RedShape r;
    r.cells = (long long)g->desc.block_cells[0] * g->desc.block_cells[1] * g->desc.block_cells[2];
    const long long per = kRedVec * (long long)(16 / elem);
    r.cpb = (int)((r.cells + per - 1) / per);
    r.nchunks = g->nblocks_total * r.cpb;
    r.nwg = (int)(r.nchunks < kRedMaxWG ? r.nchunks : kRedMaxWG);
    return r;
}

int launch_sums(cnv_grid_s *g, int comp, double *out, hipStream_t st)
{
    const RedShape r = red_shape(g, g->elem);
    {
        std::lock_guard<std::mutex> lk(g->mtx);
        int rc = ensure_partials(g, 2 * (size_t)r.nwg);
        if (rc != CNV_OK)
            return rc;
    }
    const Geom G = geom_of(g);
    if (g->desc.dtype == CNV_F64)
        hipLaunchKernelGGL(k_sums<double>, dim3(r.nwg), dim3(256), 0, st,
                           reinterpret_cast<const double *>((const char *)g->data + comp * g->component_bytes),
                           G.bstride, r.cells, r.cpb, r.nchunks, g->partials);
    else
        hipLaunchKernelGGL(k_sums<float>, dim3(r.nwg), dim3(256), 0, st,
                           reinterpret_cast<const float *>((const char *)g->data + comp * g->component_bytes),
                           G.bstride, r.cells, r.cpb, r.nchunks, g->partials);
    CNV_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_finalize_red, dim3(2), dim3(1024), 0, st, (const double *)g->partials, r.nwg, out, -1);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

// ---------------------------------------------------------------- compare

// Per-workgroup partials of sum (a-b)^2, sum b^2 and max |a-b| over one
// component of two grids of equal shape (any dtypes), evaluated in FP64.
template <typename TA, typename TB>
__global__ __launch_bounds__(256) void k_compare(const TA *pa, const TB *pb, long long bstride_a, long long bstride_b,
                                                   long long cells, int cpb, long long nchunks, double *partials)
{
    // vectors of the wider type's 16 bytes
    constexpr int VEC = 16 / (int)(sizeof(TA) > sizeof(TB) ? sizeof(TA) : sizeof(TB));
    __shared__ double red[4];
    double d2 = 0.0, b2 = 0.0, mx = 0.0;
    auto cell = [&](double x, double y) {
        const double d = x - y;
        d2 = __builtin_fma(d, d, d2);
        b2 = __builtin_fma(y, y, b2);
        mx = fmax(mx, fabs(d));
    };
    red_chunks<VEC>(cpb, nchunks, [&](long long blk, long long e0) {
        const TA *qa = pa + blk * bstride_a;
        const TB *qb = pb + blk * bstride_b;
        if (e0 + 3 * 256 * VEC + VEC <= cells) {
            VecT<TA, VEC> va[4];
            VecT<TB, VEC> vb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                va[j] = load_vec<TA, VEC>(qa + e0 + j * 256 * VEC);
                vb[j] = load_vec<TB, VEC>(qb + e0 + j * 256 * VEC);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int k = 0; k < VEC; ++k)
                    cell((double)va[j].v[k], (double)vb[j].v[k]);
        } else {
            for (int j = 0; j < 4; ++j)
                for (int k = 0; k < VEC; ++k) {
                    const long long e = e0 + j * 256 * VEC + k;
                    if (e < cells)
                        cell((double)qa[e], (double)qb[e]);
                }
        }
    });
    auto add = [](double a, double b) { return a + b; };
    auto most = [](double a, double b) { return fmax(a, b); };
    d2 = red_wg(d2, red, add);
    b2 = red_wg(b2, red, add);
    mx = red_wg(mx, red, most);
    if (threadIdx.x == 0) {
        const int n = gridDim.x;
        partials[blockIdx.x] = d2;
        partials[n + blockIdx.x] = b2;
        partials[2 * n + blockIdx.x] = mx;
    }
}

template <typename TA, typename TB>
static void compare_t(const cnv_grid_s *a, int ca, const cnv_grid_s *b, int cb, double *partials, double *out,
                      hipStream_t st)
{
    const TA *pa = reinterpret_cast<const TA *>((const char *)a->data + (size_t)ca * a->component_bytes);
    const TB *pb = reinterpret_cast<const TB *>((const char *)b->data + (size_t)cb * b->component_bytes);
    const RedShape r = red_shape(a, sizeof(TA) > sizeof(TB) ? sizeof(TA) : sizeof(TB));
    hipLaunchKernelGGL((k_compare<TA, TB>), dim3(r.nwg), dim3(256), 0, st, pa, pb,
                       (long long)(a->block_bytes / a->elem), (long long)(b->block_bytes / b->elem), r.cells, r.cpb,
                       r.nchunks, partials);
    hipLaunchKernelGGL(k_finalize_red, dim3(3), dim3(1024), 0, st, (const double *)partials, r.nwg, out, 2);
}

int launch_compare(const cnv_grid_s *a, int ca, const cnv_grid_s *b, int cb, double *out, hipStream_t st)
{
    // the reduction scratch of `a` holds two halves of at least 4096 doubles
    double *partials = a->partials;
    const bool da = a->desc.dtype == CNV_F64, db = b->desc.dtype == CNV_F64;
    if (da && db)
        compare_t<double, double>(a, ca, b, cb, partials, out, st);
    else if (da)
        compare_t<double, float>(a, ca, b, cb, partials, out, st);
    else if (db)
        compare_t<float, double>(a, ca, b, cb, partials, out, st);
    else
        compare_t<float, float>(a, ca, b, cb, partials, out, st);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

// ---------------------------------------------------------------- multi-step runs

// Steps per launch of a run: k at a time, then singles (k = 4: pairs too), in
// as many launches as has the parity of n, so that the field ends in u for even
// n and in tmp for odd.
std::vector<int> run_launches(int n, int k)
{
    int c4 = 0, c2 = 0;
    if (k == 2) {
        c2 = 2 * (n / 4);
    } else if (k == 4) {
        c4 = n / 4;
        const int rem = n % 4;
        // launches so far plus those of the rest: 0, 1 (single), 1 (pair), 2 (pair, single)
        if (rem < 2 && c4 % 2 != 0) {
            --c4;
            c2 = 2;
        } else if (rem >= 2 && c4 % 2 != 0) {
            c2 = 1;
        }
    }
    std::vector<int> l(c4, 4);
    l.insert(l.end(), c2, 2);
    l.insert(l.end(), n - 4 * c4 - 2 * c2, 1);
    return l;
}

// nsteps Euler steps alternating u -> tmp -> u ..., several per launch where
// the grid is periodic or has walls of one rule each: four or two by LDS tiles
// on small grids (tile_steps), two on larger ones by the kernels that march through
// z, on tiles of blocks of 16^3 and 32^3 cells or of the domain.  A pinned tile of
// the former keeps it.
// The norms of a launch are reduced by the next launch from the other half of
// u's partial buffer, those of the last launch by a launch of their own.
int launch_diffusion_run(cnv_grid_s *u, cnv_grid_s *tmp, int nsteps, double nu_dt, double *norms, hipStream_t st)
{
    double *P[2] = {u->partials, u->partials + u->partials_cap};
    const size_t cap = u->partials_cap;
    const int nc = u->desc.ncomp; // (tmp may have more)
    int xwg = 0, xz = 0, k = 1;
    bool tiles = false;
    int rz = 0, nt2 = 0;
    bool periodic = false, walls = false;
    if (nsteps >= 4 && !force_generic())
        periodic = run_periodic(u);
    // A run is refused before its first launch or not at all: it ends in single
    // steps unless all of them pair up, and the launches of several steps take
    // grids (components, blocks, list lengths) that a single step does not.
    // Periodic grids of 16^3 and 32^3 blocks step in pairs whatever a single
    // step takes.
    if (nsteps > 0 && !(periodic && run_periodic(tmp) && x2_shape_ok(u) && nsteps % 4 == 0)) {
        const int rc = check_step(u);
        if (rc != CNV_OK)
            return rc;
    }
    if (nsteps >= 4 && !force_generic())
        walls = !periodic && run_walls(u);
    if (periodic || walls) {
        const bool shape = x2_shape_ok(u), pinned = shape && x2_tile(u, &xwg, &xz);
        // the block-marching kernel, whose halo is the cheaper one, but for FP32 on
        // 16^3 blocks (us per step, block / domain tiles: 112^3 6.3 / 4.9, 256^3 21.8
        // / 17.2, with walls 27.1 / 22.9; 256^3 FP32 in 32^3 14.6 / 17.4, FP64 24.4 /
        // 34.9, in 16^3 FP64 30.3 / 34.1)
        const bool x2 = shape && (pinned || u->desc.dtype == CNV_F64 || u->desc.block_cells[0] == 32);
        const int kt = pinned ? 0 : tile_steps(u, x2, walls);
        tiles = kt > 0 && (size_t)kt * tile_count(u, kt, nc) <= cap && (size_t)2 * tile_count(u, 2, nc) <= cap;
        if (tiles) {
            k = kt;
        } else if (x2) {
            k = 2 * x2_tiles(u, xz) <= (long long)cap ? 2 : 1;
        } else {
            nt2 = run2_tiles(u, &rz);
            k = nt2 > 0 && (size_t)2 * nt2 <= cap ? 2 : 1;
        }
    }
    RunRules rules[2] = {}; // of u and of tmp
    for (int g = 0; walls && k > 1 && g < 2; ++g) {
        const int rc = run_rules(g == 0 ? u : tmp, nc, st, rules[g]);
        if (rc != CNV_OK)
            return rc;
    }
    const double *prev = nullptr; // nprev sets of prev_n partials, consecutive
    int nprev = 0, prev_n = 0;
    double *prev_out = nullptr;
    auto flush = [&]() -> int {
        if (nprev > 0) {
            hipLaunchKernelGGL(k_finalize_red, dim3(nprev), dim3(1024), 0, st, prev, prev_n, prev_out, -1);
            CNV_HIP(hipGetLastError());
        }
        nprev = 0;
        return CNV_OK;
    };
    int done = 0, L = 0; // steps and launches done
    for (const int kk : run_launches(nsteps, k)) {
        cnv_grid_s *a = L % 2 == 0 ? u : tmp, *b = L % 2 == 0 ? tmp : u;
        double *part = norms ? P[L % 2] : nullptr;
        const RunRules *wr = walls ? &rules[L % 2] : nullptr;
        int nt = 0, rc = CNV_OK;
        if (kk > 1 && tiles) {
            rc = launch_tile_euler(a, b, nc, kk, nu_dt, part, prev, nprev, prev_n, prev_out, wr, st);
            nt = tile_count(u, kk, nc);
        } else if (kk > 1 && nt2 > 0) {
            rc = launch_run2(a, b, nc, rz, nu_dt, part, prev, nprev, prev_n, prev_out, wr, st);
            nt = nt2;
        } else {
            if (nprev > 2)
                rc = flush();
            const double *pp[2] = {nprev > 0 ? prev : nullptr, nprev > 1 ? prev + prev_n : nullptr};
            const int pn[2] = {prev_n, prev_n};
            double *po[2] = {prev_out, prev_out + 1};
            if (rc == CNV_OK && kk > 1) {
                rc = launch_diffusion_x2(a, b, nc, nu_dt, part, part ? part + x2_tiles(u, xz) : nullptr, pp, pn, po,
                                         xwg, xz, &nt, st, wr);
            } else if (rc == CNV_OK) {
                S7Run run;
                run.partials = part;
                for (int s = 0; s < 2; ++s) {
                    run.prev[s] = pp[s];
                    run.prev_n[s] = pn[s];
                    run.prev_out[s] = po[s];
                }
                run.nparts = &nt;
                run.cap = cap;
                rc = launch_stencil7_t(a, b, nullptr, 0, 0, nc, 1, nu_dt, norms ? norms + done : nullptr, st,
                                       nullptr, &run);
            }
        }
        if (rc != CNV_OK)
            return rc;
        if (norms) {
            prev = part;
            nprev = kk;
            prev_n = nt;
            prev_out = norms + done;
        }
        done += kk;
        ++L;
    }
    return flush();
}

} // namespace cnv
