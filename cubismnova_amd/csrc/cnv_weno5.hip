// cnv_weno5.hip -- fifth-order WENO face states over the ghost-extended
// blocks of a grid (Jiang & Shu, J. Comput. Phys. 126:202-228, 1996).
//
// CubismNova advertises a WENO toolbox (README.rst:28-31) but ships none; the
// lab it would read is the FieldLab of Stencil(-3,4,false) with the blocks'
// BC lists, which this kernel assembles on the fly exactly as cnv_lab_load
// does.  For every cell i, direction d and component c it writes
//   u^-_{i+1/2} from cells i-2..i+2 with linear weights (1,6,3)/10, and
//   u^+_{i-1/2} from the mirrored stencils with weights (3,6,1)/10,
// sharing the three smoothness indicators between the two states.
// eps = 1e-6 * m2, m2 = mean of the five squared values + 1e-30, applied in
// the scale-free form  alpha_k = d_k / (1e-6 + beta_k / m2)^2, which keeps
// FP32 free of underflow for any data magnitude; the weights are evaluated
// multiplied by prod_j (1e-6 + beta_j / m2)^2 (three divisions per state
// pair instead of twelve).
//
// Work layout as in the 7-point kernel: a workgroup owns an x-y plane of one
// block of one component and marches through a z-chunk; the plane plus a
// two-cell x/y halo lives in LDS, the z neighbours in a register queue of
// planes loaded ahead.  FP64 grids are evaluated without contraction in the
// operation order of the CPU restatement (bit-identical); FP32 grids let the
// compiler fuse multiply-adds and use the hardware reciprocal.
#include "cnv_cols.h"
#include "cnv_march.h"

#include <algorithm>
#include <map>
#include <type_traits>
#include <utility>

namespace cnv
{

constexpr int kWMaxComp = 8;

struct W5Args {
    const char *in;
    char *out;
    Geom G;       // input geometry (cstride of the input grid)
    long long ocstride;
    int ncomp;
    int nzc, zchunk, tiles_per_comp;
    int has_bc[kWMaxComp];
    const DevBCHead *heads[kWMaxComp];
};

template <typename T, int NX, int NY, int WG>
__global__ __launch_bounds__(WG) void k_weno5(const W5Args a)
{
    using S = W5Shape<T, NX, NY, WG>;
    __shared__ alignas(16) T lds[2 * S::PLANE];

    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int comp = tile / a.tiles_per_comp;
    const int tt = tile - comp * a.tiles_per_comp;
    const long long blk = tt / a.nzc;
    const int zc = tt - (int)blk * a.nzc;
    const int NZ = a.G.n[2];
    const int z0 = zc * a.zchunk;
    const int z1 = min(NZ, z0 + a.zchunk);

    const T *cbase = reinterpret_cast<const T *>(a.in) + (long long)comp * a.G.cstride;
    const T *ub = cbase + blk * a.G.bstride;
    T *ob = reinterpret_cast<T *>(a.out) + (long long)(6 * comp) * a.ocstride + blk * a.G.bstride;

    FaceL<T> F[6];
    make_faces<T>(a.G, a.heads[comp], a.has_bc[comp], blk, cbase, F);
    w5_march<T, NX, NY, WG>(ub, ob, a.ocstride, F, NZ, z0, z1, lds);
}

// Blocks of any shape: a lane per VEC cells of a row and chunk of z planes
// (cnv_cols.h), the z stencil in a register queue of planes, the two rows and
// two cells on either side loaded per plane.  BC: some component's blocks
// carry BC lists.  Bound by the store stream (six values per value read) and,
// small, by load latency: 829k x 2 FP64 cells in 20x12x18 blocks 55 -> 29 us (3.2
// TB/s of one read and six writes), 864k x 5 FP32 cells in 24^3 blocks 68 us (3.5),
// 64 8^3 FP64 blocks 7.4; one thread per cell with 64-bit index divisions before.
template <typename T, int VEC, bool BC>
__global__ __launch_bounds__(kColWG) void k_weno5_cols(const W5Args a, const ColShape s)
{
    using V = VecT<T, VEC>;
    const ColLane c = col_lane<VEC>(s, a.G);
    if (!c.on)
        return;
    const int nx = a.G.n[0], ny = a.G.n[1], nz = a.G.n[2];
    const long long nxy = (long long)nx * ny;
    const long long row = (long long)nx * c.y; // within a plane
    const T *cb = reinterpret_cast<const T *>(a.in) + (long long)c.comp * a.G.cstride;
    const T *ub = cb + c.blk * a.G.bstride;
    const DevBCHead *h = nullptr;
    if (BC && a.has_bc[c.comp])
        h = a.heads[c.comp] + c.blk;
    auto nbr = [&](int f) { return cb + c.nbr[f] * a.G.bstride; };
    // cell x of this row / row y at this lane's cells / plane z of its column,
    // up to two past the block (its plane 0 where a plane is added later)
    auto cell = [&](int x) -> ColNb<T> {
        if (x < 0)
            return col_ghost<T, BC>(h, 0, nbr(0) + row + (nx + x), ub + row, ub + row + (-1 - x));
        if (x >= nx)
            return col_ghost<T, BC>(h, 1, nbr(1) + row + (x - nx), ub + row + (nx - 1), ub + row + (2 * nx - 1 - x));
        return {ub + row + x, (T)1, false};
    };
    auto line = [&](int y) -> ColNb<T> {
        const T *x0 = ub + c.x0;
        if (y < 0)
            return col_ghost<T, BC>(h, 2, nbr(2) + c.x0 + (long long)nx * (ny + y), x0, x0 + (long long)nx * (-1 - y));
        if (y >= ny)
            return col_ghost<T, BC>(h, 3, nbr(3) + c.x0 + (long long)nx * (y - ny), x0 + (long long)nx * (ny - 1),
                                    x0 + (long long)nx * (2 * ny - 1 - y));
        return {x0 + (long long)nx * y, (T)1, false};
    };
    const T *col = ub + row + c.x0;
    auto plane = [&](int z) -> V {
        if (z < 0)
            return col_load<T, VEC, BC>(col_ghost<T, BC>(h, 4, nbr(4) + row + c.x0 + nxy * (nz + z), col,
                                                         col + nxy * (-1 - z)), 0);
        if (z >= nz)
            return col_load<T, VEC, BC>(col_ghost<T, BC>(h, 5, nbr(5) + row + c.x0 + nxy * (z - nz),
                                                         col + nxy * (nz - 1), col + nxy * (2 * nz - 1 - z)), 0);
        return load_vec<T, VEC>(col + nxy * z);
    };
    const ColNb<T> xa = cell(c.x0 - 2), xb = cell(c.x0 - 1), xd = cell(c.x0 + VEC), xe = cell(c.x0 + VEC + 1);
    const ColNb<T> ya = line(c.y - 2), yb = line(c.y - 1), yd = line(c.y + 1), ye = line(c.y + 2);
    T *ob = reinterpret_cast<T *>(a.out) + (long long)(6 * c.comp) * a.ocstride + c.blk * a.G.bstride + row + c.x0;
    V q0 = plane(c.z0 - 2), q1 = plane(c.z0 - 1), q2 = plane(c.z0), q3 = plane(c.z0 + 1), q4 = plane(c.z0 + 2);
    for (int z = c.z0; z < c.z1; ++z) {
        const long long o = nxy * z;
        // x: the row's cells and two on either side
        T xs[VEC + 4];
        xs[0] = col_load1<T, BC>(xa, o);
        xs[1] = col_load1<T, BC>(xb, o);
        xs[VEC + 2] = col_load1<T, BC>(xd, o);
        xs[VEC + 3] = col_load1<T, BC>(xe, o);
        const V va = col_load<T, VEC, BC>(ya, o), vb = col_load<T, VEC, BC>(yb, o);
        const V vd = col_load<T, VEC, BC>(yd, o), ve = col_load<T, VEC, BC>(ye, o);
        V q5 = q4;
        if (z + 1 < c.z1)
            q5 = plane(z + 3);
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            xs[v + 2] = q2.v[v];
        V r[6];
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
            weno5<T>(q0.v[v], q1.v[v], q2.v[v], q3.v[v], q4.v[v], r[4].v[v], r[5].v[v]);
            weno5<T>(xs[v], xs[v + 1], xs[v + 2], xs[v + 3], xs[v + 4], r[0].v[v], r[1].v[v]);
            weno5<T>(va.v[v], vb.v[v], q2.v[v], vd.v[v], ve.v[v], r[2].v[v], r[3].v[v]);
        }
#pragma unroll
        for (int k = 0; k < 6; ++k)
            store_nt<T, VEC>(ob + k * a.ocstride + o, r[k]);
        q0 = q1;
        q1 = q2;
        q2 = q3;
        q3 = q4;
        q4 = q5;
    }
}

// ---------------------------------------------------------------- host side

struct W5Tune {
    int wg, zchunk;
};
static std::mutex g_w5_mtx;
static std::map<std::pair<int, int>, W5Tune> g_w5_tune; // (dtype, edge) -> choice

// built-in choices (measured at 512^3 for edge 32)
static W5Tune w5_default(int dtype, int edge)
{
    if (edge == 16)
        return dtype == CNV_F64 ? W5Tune{128, 16} : W5Tune{64, 16};
    if (edge == 32)
        return dtype == CNV_F64 ? W5Tune{256, 32} : W5Tune{256, 32};
    return W5Tune{256, 16};
}

// pinned: set to something else than the built-in tile
static W5Tune w5_tune(int dtype, int edge, bool *pinned = nullptr)
{
    std::lock_guard<std::mutex> lk(g_w5_mtx);
    auto it = g_w5_tune.find({dtype, edge});
    const W5Tune d = w5_default(dtype, edge), t = it == g_w5_tune.end() ? d : it->second;
    if (pinned)
        *pinned = t.wg != d.wg || t.zchunk != d.zchunk;
    return t;
}

// The tile of a launch over `nbc` blocks times components of nz planes: the
// pinned one, else the built-in one with the deepest z chunk (down to two
// planes) that gives enough tiles to fill the GPU.  A chunk's planes run one
// after another, about 2 us each, so on a grid of few tiles the chain is the
// launch.  Built-in depth / this rule: 128^3 FP32 in 32^3 blocks 68.8 / 18.8 us,
// in 64^3 blocks 107 / 20.7, 192^3 FP64 in 32^3 blocks 116 / 91, 256^3 FP32 in
// 64^3 blocks 124 / 103; twice or half as many tiles: 20.6 and 23.3, 31.9 (half),
// 99 and 116, 118 and 124.
static W5Tune w5_tile(int dtype, int edge, long long nbc, int nz)
{
    bool pinned = false;
    W5Tune t = w5_tune(dtype, edge, &pinned);
    if (pinned)
        return t;
    const long long enough =
        edge >= 64 ? (dtype == CNV_F64 ? 200 : 400) : edge == 32 ? 400 : dtype == CNV_F64 ? 800 : 1500;
    auto tiles = [&](int z) { return nbc * ((nz + z - 1) / z); };
    t.zchunk = std::min(t.zchunk, nz);
    while (t.zchunk > 2 && tiles(t.zchunk) < enough)
        t.zchunk = (t.zchunk + 1) / 2;
    return t;
}

// Grids of 16, 32 or 64 cells per x/y edge run as columns below 1.2M cells
// times components unless a tile is pinned: 32^3 FP32 69 -> 7.1 us, 64^3 FP64 in
// 32^3 blocks 93 -> 9.4, 96^3 FP64 in 16^3 blocks 32.5 -> 20.4.  At 2.1M cells the
// marching tile of the rule above is level or ahead (18.8 / 20.8 us FP32, 30.0 /
// 31.0 FP64 in 32^3 blocks).
static bool w5_cols_for_small(const Geom &G, int ncomp)
{
    return (long long)G.nb[0] * G.nb[1] * G.nb[2] * ncomp * G.n[0] * G.n[1] * G.n[2] < 1200000;
}

template <typename T, int NX, int WG>
constexpr bool w5_valid()
{
    return W5Shape<T, NX, NX, WG>::valid;
}

template <typename T, int NX, int WG>
static bool w5_launch(const W5Args &a, int ntiles, hipStream_t st)
{
    if constexpr (w5_valid<T, NX, WG>()) {
        hipLaunchKernelGGL((k_weno5<T, NX, NX, WG>), dim3(ntiles), dim3(WG), 0, st, a);
        return true;
    }
    return false;
}

template <typename T, int NX>
static bool w5_dispatch_wg(const W5Args &a, int wg, int ntiles, hipStream_t st)
{
    switch (wg) {
    case 64:
        return w5_launch<T, NX, 64>(a, ntiles, st);
    case 128:
        return w5_launch<T, NX, 128>(a, ntiles, st);
    case 256:
        return w5_launch<T, NX, 256>(a, ntiles, st);
    case 512:
        return w5_launch<T, NX, 512>(a, ntiles, st);
    default:
        return false;
    }
}

// The column kernel on blocks of any shape.
template <typename T>
static int w5_cols(const W5Args &a, hipStream_t st)
{
    const int *n = a.G.n;
    const long long gx = ((long long)n[0] * n[1] * n[2] + 255) / 256;
    const long long gy = (long long)a.G.nb[0] * a.G.nb[1] * a.G.nb[2] * a.ncomp;
    if (gx > 0x7fffffffLL || gy > 65535)
        return fail(CNV_ERR_UNSUPPORTED, "grid too large for the generic WENO5 kernel");
    const int vec = col_vec(n[0], sizeof(T));
    // planes per lane: FP64 as many as leave the two and a half waves per SIMD
    // that its registers allow at once, FP32 two and a half times as many lanes;
    // 16 at most.  24^3 x 5 FP32 68 us with 450k lanes, 78 with 180k; 48^3 x 2
    // FP32 60 with 500k, 70 with 166k; 20x12x18 x 2 FP64 29 with 184k, 32 with 276k
    // and 138k.
    const long long vectors = gy * ((long long)n[0] / vec * n[1] * n[2]);
    const int z = (int)std::min<long long>(16, std::max<long long>(1, vectors / (sizeof(T) == 4 ? 409600 : 163840)));
    ColShape s;
    if (!col_shape(a.G, a.ncomp, vec, std::min(z, n[2]), s))
        return fail(CNV_ERR_UNSUPPORTED, "grid too large for the generic WENO5 kernel");
    bool bc = false;
    for (int c = 0; c < a.ncomp; ++c)
        bc = bc || a.has_bc[c];
    auto go = [&](auto v) {
        constexpr int VEC = decltype(v)::value;
        if (bc)
            hipLaunchKernelGGL((k_weno5_cols<T, VEC, true>), s.wgs.dim(), dim3(kColWG), 0, st, a, s);
        else
            hipLaunchKernelGGL((k_weno5_cols<T, VEC, false>), s.wgs.dim(), dim3(kColWG), 0, st, a, s);
    };
    if (vec == 1)
        go(std::integral_constant<int, 1>());
    else if (vec == 2)
        go(std::integral_constant<int, 2>());
    else if constexpr (sizeof(T) == 4)
        go(std::integral_constant<int, 4>());
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

template <typename T>
static int w5_run(W5Args &a, hipStream_t st, const W5Tune *over)
{
    const int *n = a.G.n;
    const long long nbt = (long long)a.G.nb[0] * a.G.nb[1] * a.G.nb[2];
    if (n[0] == n[1] && (n[0] == 16 || n[0] == 32 || n[0] == 64)) {
        const int dtype = sizeof(T) == 8 ? CNV_F64 : CNV_F32;
        bool pinned = false;
        (void)w5_tune(dtype, n[0], &pinned);
        if (!over && !pinned && w5_cols_for_small(a.G, a.ncomp))
            return w5_cols<T>(a, st);
        const W5Tune tu = over ? *over : w5_tile(dtype, n[0], nbt * a.ncomp, n[2]);
        a.zchunk = tu.zchunk < n[2] ? tu.zchunk : n[2];
        a.nzc = (n[2] + a.zchunk - 1) / a.zchunk;
        a.tiles_per_comp = (int)(nbt * a.nzc);
        const long long ntiles = (long long)a.tiles_per_comp * a.ncomp;
        bool ok = false;
        if (ntiles < (1LL << 31)) {
            if (n[0] == 16)
                ok = w5_dispatch_wg<T, 16>(a, tu.wg, (int)ntiles, st);
            else if (n[0] == 32)
                ok = w5_dispatch_wg<T, 32>(a, tu.wg, (int)ntiles, st);
            else
                ok = w5_dispatch_wg<T, 64>(a, tu.wg, (int)ntiles, st);
        }
        if (ok) {
            CNV_HIP(hipGetLastError());
            return CNV_OK;
        }
        if (over)
            return fail(CNV_ERR_UNSUPPORTED, "tile shape not available for this block edge and dtype");
    }
    return w5_cols<T>(a, st);
}

int launch_weno5(cnv_grid_s *in, cnv_grid_s *out, hipStream_t st, const int *tile)
{
    const int nc = in->desc.ncomp;
    if (nc > kWMaxComp)
        return fail(CNV_ERR_UNSUPPORTED, "more than 8 components in one WENO5 call");
    for (int d = 0; d < 3; ++d)
        if (in->desc.block_cells[d] < 2)
            return fail(CNV_ERR_UNSUPPORTED, "WENO5 reads two ghost layers: block edges must be >= 2");
    W5Args a;
    a.in = static_cast<const char *>(in->data);
    a.out = static_cast<char *>(out->data);
    a.G = geom_of(in);
    a.ocstride = (long long)(out->component_bytes / out->elem);
    a.ncomp = nc;
    {
        std::lock_guard<std::mutex> lk(in->mtx);
        for (int c = 0; c < nc; ++c) {
            int rc = ensure_bc_table(in, c);
            if (rc != CNV_OK)
                return rc;
            if (face_info(in, c).unset)
                return fail(CNV_ERR_UNSUPPORTED,
                            "BC list leaves ghost cells of a face unwritten for Stencil(-3,4)");
            a.has_bc[c] = (in->tables[c].any && in->tables[c].heads) ? 1 : 0;
            a.heads[c] = in->tables[c].heads;
        }
    }
    for (int c = nc; c < kWMaxComp; ++c) {
        a.has_bc[c] = 0;
        a.heads[c] = nullptr;
    }
    a.nzc = a.zchunk = a.tiles_per_comp = 0;
    W5Tune over;
    if (tile) {
        over.wg = tile[0];
        over.zchunk = tile[1];
    }
    if (in->desc.dtype == CNV_F64)
        return w5_run<double>(a, st, tile ? &over : nullptr);
    return w5_run<float>(a, st, tile ? &over : nullptr);
}

template <typename T>
static bool w5_valid_rt(int edge, int wg)
{
    auto pick = [&](auto e) -> bool {
        constexpr int E = decltype(e)::value;
        return wg == 64    ? w5_valid<T, E, 64>()
               : wg == 128 ? w5_valid<T, E, 128>()
               : wg == 256 ? w5_valid<T, E, 256>()
               : wg == 512 ? w5_valid<T, E, 512>()
                           : false;
    };
    if (edge == 16)
        return pick(std::integral_constant<int, 16>());
    if (edge == 32)
        return pick(std::integral_constant<int, 32>());
    if (edge == 64)
        return pick(std::integral_constant<int, 64>());
    return false;
}

int weno5_set_tune(int dtype, int edge, int wg, int zchunk)
{
    if (edge != 16 && edge != 32 && edge != 64)
        return fail(CNV_ERR_INVALID, "WENO5 tiles exist for block edges 16, 32 and 64");
    if (zchunk < 1)
        return fail(CNV_ERR_INVALID, "zchunk must be >= 1");
    const bool ok = dtype == CNV_F64 ? w5_valid_rt<double>(edge, wg) : w5_valid_rt<float>(edge, wg);
    if (!ok)
        return fail(CNV_ERR_UNSUPPORTED, "WENO5 tile shape not available for this block edge and dtype");
    std::lock_guard<std::mutex> lk(g_w5_mtx);
    g_w5_tune[{dtype, edge}] = {wg, zchunk};
    return CNV_OK;
}

int weno5_get_tune(int dtype, int edge, int *wg, int *zchunk)
{
    const W5Tune t = w5_tune(dtype, edge);
    *wg = t.wg;
    *zchunk = t.zchunk;
    return CNV_OK;
}

// Times every (workgroup size, z-chunk) candidate on in -> out and keeps the
// fastest for the input's (dtype, block edge).
int autotune_weno5(cnv_grid_s *in, cnv_grid_s *out, int iters, int *best_wg, int *best_z, double *results,
                   int max_results, int *nresults)
{
    const int *n = in->desc.block_cells;
    if (!(n[0] == n[1] && (n[0] == 16 || n[0] == 32 || n[0] == 64)))
        return fail(CNV_ERR_UNSUPPORTED, "autotuning needs x/y block edges of 16, 32 or 64");
    if (iters < 1)
        return fail(CNV_ERR_INVALID, "iters must be >= 1");
    hipStream_t st;
    CNV_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    hipEvent_t e0, e1;
    CNV_HIP(hipEventCreate(&e0));
    CNV_HIP(hipEventCreate(&e1));
    const int wgs[4] = {64, 128, 256, 512};
    const int zcs[5] = {4, 8, 16, 32, 64};
    float best = 1e30f;
    int bw = 0, bz = 0, cnt = 0, rc = CNV_OK;
    for (int wi = 0; wi < 4 && rc == CNV_OK; ++wi)
        for (int zi = 0; zi < 5; ++zi) {
            if (zcs[zi] > n[2])
                continue;
            const int tile[2] = {wgs[wi], zcs[zi]};
            int r = launch_weno5(in, out, st, tile);
            if (r == CNV_ERR_UNSUPPORTED)
                continue;
            if (r != CNV_OK) {
                rc = r;
                break;
            }
            (void)hipEventRecord(e0, st);
            for (int i = 0; i < iters; ++i)
                (void)launch_weno5(in, out, st, tile);
            (void)hipEventRecord(e1, st);
            if (hipEventSynchronize(e1) != hipSuccess) {
                rc = fail(CNV_ERR_HIP, "autotune: kernel failed");
                break;
            }
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            const float us = ms * 1000.f / iters;
            if (results && cnt < max_results) {
                results[3 * cnt] = tile[0];
                results[3 * cnt + 1] = tile[1];
                results[3 * cnt + 2] = us;
            }
            ++cnt;
            if (us < best) {
                best = us;
                bw = tile[0];
                bz = tile[1];
            }
        }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(st);
    if (rc != CNV_OK)
        return rc;
    if (bw == 0)
        return fail(CNV_ERR_UNSUPPORTED, "no tile candidate ran");
    weno5_set_tune(in->desc.dtype, n[0], bw, bz);
    if (best_wg)
        *best_wg = bw;
    if (best_z)
        *best_z = bz;
    if (nresults)
        *nresults = cnt < max_results ? cnt : max_results;
    return CNV_OK;
}

} // namespace cnv
