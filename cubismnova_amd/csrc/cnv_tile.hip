// cnv_tile.hip -- K diffusion steps or Jacobi sweeps per launch on tiles of
// the domain held in LDS, for any block shape.
//
// On small grids a launch costs about 4.5 us whatever it does, and the
// plane-marching kernels add a serial chain of planes.  Here a workgroup loads a tile of
// CX x CY x CZ cells of the domain, wherever its blocks lie, plus K cells on
// every side into LDS, evaluates step j on the cells within K - j of the tile
// (so that step K covers exactly the tile), and writes the tile.  Block
// boundaries exist only in three offset tables (one entry per x, y and z of the
// loaded box); past a wall nothing is loaded or evaluated: a cell next to a
// wall reads the wall's constant or its own value times the wall's factor
// (layer 1 of Symmetry and Absorbing is that cell itself).  Every value is the
// single step's expression on the same operands, so results are bit-identical.
#include "cnv_cols.h"

#include <algorithm>
#include <type_traits>

namespace cnv
{

struct TileArgs {
    const char *u; // component slabs
    char *out;
    const char *f; // Jacobi: the source component
    long long cs_u, cs_o;
    long long bstride; // of all three grids
    int nb[3], n[3], ng[3], nt[3];
    FastDiv dn[3];
    int ntiles; // of all components
    RunRules rules;
    double ih2[3], nudt;
    const double *czm, *czp;
    double omega;
    double *part; // norms: part[j * ntiles + tile]
    // deferred sums of the previous launch: nprev sets of prev_n partials
    const double *prev_p;
    int nprev, prev_n;
    double *prev_out;
};

enum { TILE_EULER = 0, TILE_JACOBI = 1 };

template <typename T, int OP, int K, int CX, int CY, int CZ>
struct TileShape {
    static constexpr int VEC = 16 / (int)sizeof(T);
    static constexpr int PX = (K + VEC - 1) / VEC * VEC; // cells before the tile in an LDS row
    static constexpr int LX = CX + 2 * PX, LY = CY + 2 * K, LZ = CZ + 2 * K;
    static constexpr int SZ = LX * LY * LZ + 2 * VEC; // a row's end reads one cell past it
    static constexpr int NT = LX + LY + LZ;           // offset table entries
    static constexpr size_t lds = sizeof(T) * SZ * (OP == TILE_JACOBI ? 3 : 2) + 4 * NT + 3 * sizeof(T) * LZ + 512;
    static constexpr bool valid = CX % VEC == 0 && lds <= 160 * 1024;
};

// WALL: some domain face is no periodic neighbour
template <typename T, int OP, int K, int CX, int CY, int CZ, int WG, bool WALL, bool NORM>
__global__ __launch_bounds__(WG) void k_tile(const TileArgs a)
{
    using S = TileShape<T, OP, K, CX, CY, CZ>;
    static_assert(S::valid, "tile shape");
    constexpr int VEC = S::VEC, PX = S::PX, LX = S::LX, LY = S::LY, LZ = S::LZ, LXY = LX * LY;
    using V = VecT<T, VEC>;
    __shared__ alignas(16) T sA[S::SZ], sB[S::SZ];
    __shared__ alignas(16) T sF[OP == TILE_JACOBI ? S::SZ : 1];
    __shared__ int toff[S::NT];
    __shared__ T tz[OP == TILE_JACOBI ? 3 * LZ : 1]; // czm, czp, wd of the loaded planes
    __shared__ double red[K * (WG / 64)];

    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= a.ntiles) { // a workgroup for each deferred sum
        const int k = blockIdx.x - a.ntiles;
        wg_sum_partials<WG>(a.prev_p + (size_t)k * a.prev_n, a.prev_n, a.prev_out + k, red);
        return;
    }
    int t = xcd_remap(blockIdx.x, a.ntiles);
    const int tile = t;
    const int tx = t % a.nt[0];
    t /= a.nt[0];
    const int ty = t % a.nt[1];
    t /= a.nt[1];
    const int tzi = t % a.nt[2], comp = t / a.nt[2];
    const int X0 = tx * CX, Y0 = ty * CY, Z0 = tzi * CZ; // the tile's first cell in the domain
    const int NX = a.ng[0], NY = a.ng[1], NZ = a.ng[2];
    const T *ub = reinterpret_cast<const T *>(a.u) + (long long)comp * a.cs_u;
    T *ob = reinterpret_cast<T *>(a.out) + (long long)comp * a.cs_o;
    const DevRules rules = rules_of<OP == TILE_JACOBI>(a.rules, offsetof(TileArgs, rules), WALL ? comp : 0);
    // FM_* of the face 2 dir + side in four bits: the cell loop tests it at every
    // vector (a 64^3 refined solve 925 us, 980 with a load at each test)
    unsigned fm = 0u;
    for (int f = 0; WALL && f < 6; ++f)
        fm |= (unsigned)rules->fm[f] << (4 * f);
    auto rule = [&](int d, int side) { return (int)(fm >> (8 * d + 4 * side)) & 15; };
    auto value = [&](int d, int side) { return (T)rules->v[2 * d + side]; }; // constant or sign of a wall

    // element offset of every loaded x, y and z: periodic axes wrapped, walls
    // clamped (those cells are loaded and never used)
    if (tid < S::NT) {
        const int d = tid < LX ? 0 : tid < LX + LY ? 1 : 2;
        const int i = tid - (d == 0 ? 0 : d == 1 ? LX : LX + LY);
        int g = (d == 0 ? X0 - PX : (d == 1 ? Y0 : Z0) - K) + i;
        const int ngd = d == 0 ? NX : d == 1 ? NY : NZ;
        if (!WALL || rule(d, 0) == FM_PERIODIC) {
            g %= ngd;
            g = g < 0 ? g + ngd : g;
        } else {
            // (x: whole vectors where rows are whole vectors)
            g = min(max(g, 0), d == 0 && a.n[0] % VEC == 0 && i % VEC == 0 ? ngd - VEC : ngd - 1);
        }
        const int nd = d == 0 ? a.n[0] : d == 1 ? a.n[1] : a.n[2];
        const FastDiv fd = d == 0 ? a.dn[0] : d == 1 ? a.dn[1] : a.dn[2];
        const int b = fdiv(g, fd), l = g - b * nd;
        const long long bs = a.bstride * (d == 0 ? 1 : d == 1 ? a.nb[0] : (long long)a.nb[0] * a.nb[1]);
        const int ls = d == 0 ? 1 : d == 1 ? a.n[0] : a.n[0] * a.n[1];
        toff[tid] = (int)(b * bs) + l * ls; // (slabs hold fewer than 2^31 elements)
        if (OP == TILE_JACOBI && d == 2) {
            // past a wall the metric is not used
            const T ihx2 = (T)a.ih2[0], ihy2 = (T)a.ih2[1];
            const T cm = (T)a.czm[g], cp = (T)a.czp[g];
            const T diag = -(2 * ihx2 + 2 * ihy2 + cm + cp);
            tz[i] = cm;
            tz[LZ + i] = cp;
            tz[2 * LZ + i] = (T)a.omega / diag;
        }
    }
    __syncthreads();
    const int *ox = toff + PX, *oy = toff + LX, *oz = oy + LY; // x from -PX
    // cell (x, y, z) of the loaded box (y, z from 0, x from -PX) in LDS
    auto at = [&](int x, int y, int z) { return VEC + (x + PX) + LX * (y + LY * z); };

    // load the box, by vectors where the rows of a block are whole vectors (one
    // then lies in one block and is aligned), kLd loads per thread in flight
    const T *fb = OP == TILE_JACOBI ? reinterpret_cast<const T *>(a.f) : nullptr;
    auto load = [&](auto width) {
        constexpr int W = decltype(width)::value;
        constexpr int X = W == 1 ? K : PX, NXL = (CX + 2 * X) / W, N = NXL * LY * LZ;
        constexpr int kLd = (N + WG - 1) / WG < 6 ? (N + WG - 1) / WG : 6;
        using VW = VecT<T, W>;
        for (int l0 = tid; l0 < N; l0 += kLd * WG) {
            VW v[kLd], w[kLd];
#pragma unroll
            for (int k = 0; k < kLd; ++k) {
                const int l = min(l0 + k * WG, N - 1);
                const int r = l / NXL, x = (l - r * NXL) * W - X, z = r / LY, y = r - z * LY;
                const int o = ox[x] + oy[y] + oz[z];
                v[k] = load_vec<T, W>(ub + o);
                if (OP == TILE_JACOBI)
                    w[k] = load_vec<T, W>(fb + o);
            }
#pragma unroll
            for (int k = 0; k < kLd; ++k) {
                const int l = l0 + k * WG;
                const int r = l / NXL, x = (l - r * NXL) * W - X, z = r / LY, y = r - z * LY;
                if (l < N) {
                    store_vec<T, W>(sA + at(x, y, z), v[k]);
                    if (OP == TILE_JACOBI)
                        store_vec<T, W>(sF + at(x, y, z), w[k]);
                }
            }
        }
    };
    if (a.n[0] % VEC == 0)
        load(std::integral_constant<int, VEC>());
    else
        load(std::integral_constant<int, 1>());
    __syncthreads();

    const T ihx2 = (T)a.ih2[0], ihy2 = (T)a.ih2[1], ihz2 = (T)a.ih2[2], nudt = (T)a.nudt;
    double acc[K];
    T *A = sA, *B = sB;
#pragma unroll
    for (int j = 1; j <= K; ++j) {
        const int m = K - j;
        const int NV = m > 0 ? LX / VEC : CX / VEC; // vectors per row
        const int RY = CY + 2 * m, RZ = CZ + 2 * m;
        double s = 0.0;
        for (int q = tid; q < NV * RY * RZ; q += WG) {
            const int r = q / NV, z = j + r / RY, y = j + r % RY;
            const int x = (q - r * NV) * VEC - (m > 0 ? PX : 0); // relative to the tile
            const int p = at(x, y, z);
            const int gx = X0 + x, gy = Y0 - K + y, gz = Z0 - K + z;
            const V c = *reinterpret_cast<const V *>(A + p);
            V ym = *reinterpret_cast<const V *>(A + p - LX), yp = *reinterpret_cast<const V *>(A + p + LX);
            V zm = *reinterpret_cast<const V *>(A + p - LXY), zp = *reinterpret_cast<const V *>(A + p + LXY);
            T xl = A[p - 1], xr = A[p + VEC];
            int xe = -1; // the vector's element next to the upper x wall
            if constexpr (WALL) {
                auto wall = [&](int d, int side, T v) {
                    const int k = rule(d, side);
                    return k == FM_CONST ? value(d, side) : k == FM_MIRROR ? value(d, side) * v : v;
                };
                if (gx == 0 && rule(0, 0) != FM_PERIODIC)
                    xl = wall(0, 0, c.v[0]);
                if (rule(0, 1) != FM_PERIODIC)
                    xe = NX - 1 - gx;
                if (gy == 0 && rule(1, 0) != FM_PERIODIC)
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        ym.v[v] = wall(1, 0, c.v[v]);
                if (gy == NY - 1 && rule(1, 1) != FM_PERIODIC)
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        yp.v[v] = wall(1, 1, c.v[v]);
                if (gz == 0 && rule(2, 0) != FM_PERIODIC)
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        zm.v[v] = wall(2, 0, c.v[v]);
                if (gz == NZ - 1 && rule(2, 1) != FM_PERIODIC)
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        zp.v[v] = wall(2, 1, c.v[v]);
            }
            T cm = (T)0, cp = (T)0, wd = (T)0;
            V f;
            if constexpr (OP == TILE_JACOBI) {
                cm = tz[z];
                cp = tz[LZ + z];
                wd = tz[2 * LZ + z];
                f = *reinterpret_cast<const V *>(sF + p);
            }
            V res;
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                const T e = c.v[v];
                const T l = v == 0 ? xl : c.v[v - 1];
                T h = v == VEC - 1 ? xr : c.v[v + 1];
                if (WALL && xe == v)
                    h = rule(0, 1) == FM_CONST ? value(0, 1)
                        : rule(0, 1) == FM_MIRROR ? value(0, 1) * e : e;
                const T ddx = ihx2 * (fms2(e, h) + l);
                const T ddy = ihy2 * (fms2(e, yp.v[v]) + ym.v[v]);
                if constexpr (OP == TILE_EULER) {
                    const T ddz = ihz2 * (fms2(e, zp.v[v]) + zm.v[v]);
                    const T lap = ddx + ddy + ddz;
                    const T d = lap * nudt;
                    res.v[v] = e + d;
                } else {
                    const T az = cp * (zp.v[v] - e) - cm * (e - zm.v[v]);
                    const T au = ddx + ddy + az;
                    const T rr = f.v[v] - au;
                    res.v[v] = e + rr * wd;
                }
            }
            const bool core = x >= 0 && x < CX && y >= K && y < K + CY && z >= K && z < K + CZ && gy < NY && gz < NZ;
            if (NORM && core) {
#pragma unroll
                for (int v = 0; v < VEC; ++v) {
                    const double d = gx + v < NX ? (double)res.v[v] : 0.0;
                    s = __builtin_fma(d, d, s);
                }
            }
            if (j < K) {
                *reinterpret_cast<V *>(B + p) = res;
            } else if (core) {
                const int o = oy[y] + oz[z];
                // whole vectors of a row stay in one block, aligned, where its
                // edge is a multiple of the vector
                if (a.n[0] % VEC == 0) {
                    if (gx < NX)
                        store_vec<T, VEC>(ob + o + ox[x], res);
                } else {
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        if (gx + v < NX)
                            ob[o + ox[x + v]] = res.v[v];
                }
            }
        }
        acc[j - 1] = s;
        if (j < K)
            __syncthreads();
        T *const C = A;
        A = B;
        B = C;
    }

    if (NORM) { // per-tile partials of every step in a fixed wave tree and wave order
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int j = 0; j < K; ++j)
                acc[j] += __shfl_xor(acc[j], o, 64);
        if ((tid & 63) == 0)
#pragma unroll
            for (int j = 0; j < K; ++j)
                red[j * (WG / 64) + tid / 64] = acc[j];
        __syncthreads();
        if (tid < K) {
            double r = 0.0;
            for (int w = 0; w < WG / 64; ++w)
                r += red[tid * (WG / 64) + w];
            a.part[(size_t)tid * a.ntiles + tile] = r;
        }
    }
}

// ---------------------------------------------------------------- host side

// Tile of a launch of K steps: cells per axis and workgroup size.
template <int K>
struct TileOf;
template <>
struct TileOf<2> {
    static constexpr int CX = 16, CY = 16, CZ = 8, WG = 512;
};
template <>
struct TileOf<4> {
    static constexpr int CX = 16, CY = 8, CZ = 8, WG = 1024;
};

static bool tile_layout(const cnv_grid_s *u, TileArgs &a, int cx, int cy, int cz, int ncomp)
{
    const Geom G = geom_of(u);
    if (u->component_bytes / u->elem >= (1ull << 31))
        return false;
    a.bstride = G.bstride;
    const int c[3] = {cx, cy, cz};
    long long nt = ncomp;
    for (int d = 0; d < 3; ++d) {
        a.nb[d] = G.nb[d];
        a.n[d] = G.n[d];
        a.ng[d] = G.nb[d] * G.n[d];
        a.nt[d] = (a.ng[d] + c[d] - 1) / c[d];
        a.dn[d] = fast_div((unsigned)G.n[d]);
        nt *= a.nt[d];
    }
    if (nt >= (1LL << 32) / 1024 - 4) // (and the deferred sums: fewer than 2^32 threads)
        return false;
    a.ntiles = (int)nt;
    return true;
}

template <typename T, int OP, int K>
static void tile_launch(const TileArgs &a, bool wall, hipStream_t st)
{
    using C = TileOf<K>;
    const dim3 g((unsigned)(a.ntiles + a.nprev)), b(C::WG);
    if constexpr (OP == TILE_JACOBI) {
        if (wall)
            hipLaunchKernelGGL((k_tile<T, OP, K, C::CX, C::CY, C::CZ, C::WG, true, false>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((k_tile<T, OP, K, C::CX, C::CY, C::CZ, C::WG, false, false>), g, b, 0, st, a);
    } else if (wall) {
        if (a.part)
            hipLaunchKernelGGL((k_tile<T, OP, K, C::CX, C::CY, C::CZ, C::WG, true, true>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((k_tile<T, OP, K, C::CX, C::CY, C::CZ, C::WG, true, false>), g, b, 0, st, a);
    } else {
        if (a.part)
            hipLaunchKernelGGL((k_tile<T, OP, K, C::CX, C::CY, C::CZ, C::WG, false, true>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((k_tile<T, OP, K, C::CX, C::CY, C::CZ, C::WG, false, false>), g, b, 0, st, a);
    }
}

template <int K>
static bool tile_layout(const cnv_grid_s *u, TileArgs &a, int ncomp)
{
    using C = TileOf<K>;
    return tile_layout(u, a, C::CX, C::CY, C::CZ, ncomp);
}

// tiles of a launch of k steps on ncomp components of u; 0: not available
int tile_count(const cnv_grid_s *u, int k, int ncomp)
{
    TileArgs a;
    const bool ok = k == 2 ? tile_layout<2>(u, a, ncomp) : tile_layout<4>(u, a, ncomp);
    return ok ? a.ntiles : 0;
}

// Euler steps per tile launch on u; 0: the kernels that march through z take it,
// two steps per launch, on tiles of blocks (`block_tiles`) or of the domain.
// Figures are us per step of runs with norms, marching / tiles.  Four steps while
// there is at most one tile per CU, where the launch is its fixed 4.5 us plus one
// tile's 5 us (64^3 in 32^3 blocks 3.5 / 2.4 FP32, 4.0 / 3.1 FP64, with walls 4.5 /
// 2.9 and 4.6 / 3.5; 60^3 in 20^3 blocks, against single steps, 4.5 / 2.4 and 4.8
// / 3.1); with more, the 2.2 evaluations per cell of four steps cost more than
// the launches of two (80^3 FP32: 3.5 with four, 3.2 with two).  Two steps while
// the marching kernels have too few tiles.  In FP32, against domain tiles up to
// 500 tiles (72^3 3.6 / 3.2, 108^3 4.2 / 5.0), with walls, which cost those more, up
// to 700 (96^3 5.1 / 4.5, 108^3 6.3 / 5.7, 120^3 periodic 5.7 / 6.4); against block
// tiles up to 450 (96^3 in 32^3 blocks 4.1 / 3.9).  In FP64, against domain tiles
// up to 450 (72^3 3.85 / 3.85, 96^3 with walls 5.9 / 5.7, 120^3 6.1 / 8.9).
int tile_steps(const cnv_grid_s *u, bool block_tiles, bool walls)
{
    const int t4 = tile_count(u, 4, u->desc.ncomp), t2 = tile_count(u, 2, u->desc.ncomp);
    if (t4 == 0 || t2 == 0)
        return 0;
    if (t4 <= 256)
        return 4;
    const bool f32 = u->desc.dtype == CNV_F32;
    const int most = block_tiles ? (f32 ? 450 : 0) : f32 ? (walls ? 700 : 500) : 450;
    return t2 <= most ? 2 : 0;
}

int launch_tile_euler(cnv_grid_s *u, cnv_grid_s *out, int ncomp, int k, double nu_dt, double *part, const double *prev_p,
                      int nprev, int prev_n, double *prev_out, const RunRules *rules, hipStream_t st)
{
    TileArgs a{};
    if (!(k == 2 ? tile_layout<2>(u, a, ncomp) : tile_layout<4>(u, a, ncomp)))
        return fail(CNV_ERR_UNSUPPORTED, "grid too large for the tile kernel");
    a.u = static_cast<const char *>(u->data);
    a.out = static_cast<char *>(out->data);
    a.cs_u = (long long)(u->component_bytes / u->elem);
    a.cs_o = (long long)(out->component_bytes / out->elem);
    const bool wall = rules != nullptr;
    if (rules)
        a.rules = *rules;
    for (int d = 0; d < 3; ++d)
        a.ih2[d] = 1. / (u->h[d] * u->h[d]);
    a.nudt = nu_dt;
    a.part = part;
    a.prev_p = prev_p;
    a.nprev = nprev;
    a.prev_n = prev_n;
    a.prev_out = prev_out;
    if (u->desc.dtype == CNV_F64)
        k == 2 ? tile_launch<double, TILE_EULER, 2>(a, wall, st) : tile_launch<double, TILE_EULER, 4>(a, wall, st);
    else
        k == 2 ? tile_launch<float, TILE_EULER, 2>(a, wall, st) : tile_launch<float, TILE_EULER, 4>(a, wall, st);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

// k = 2 (FP32) or 4 sweeps u -> out on grids that take the two-sweep kernel; the
// caller has set up u's z metric.
int launch_tile_jacobi(cnv_grid_s *u, int cu, cnv_grid_s *f, int cf, cnv_grid_s *out, int co, int k, double omega,
                       hipStream_t st)
{
    TileArgs a{};
    if (!(k == 2 ? u->desc.dtype == CNV_F32 && tile_layout<2>(u, a, 1) : tile_layout<4>(u, a, 1)))
        return fail(CNV_ERR_UNSUPPORTED, "no tile launch of these sweeps on this grid");
    int fm[3][2];
    double fv[3][2];
    if (!jacobi2_faces(u, cu, fm, fv))
        return fail(CNV_ERR_UNSUPPORTED, "several sweeps per launch need one rule per domain face");
    bool wall = false;
    for (int f = 0; f < 6; ++f) {
        const int d = f >> 1, s = f & 1;
        wall = wall || fm[d][s] != FM_PERIODIC;
        a.rules.val[0].fm[f] = fm[d][s];
        a.rules.val[0].v[f] = fv[d][s];
    }
    a.u = static_cast<const char *>(u->data) + (size_t)cu * u->component_bytes;
    a.f = static_cast<const char *>(f->data) + (size_t)cf * f->component_bytes;
    a.out = static_cast<char *>(out->data) + (size_t)co * out->component_bytes;
    a.ih2[0] = 1. / (u->h[0] * u->h[0]);
    a.ih2[1] = 1. / (u->h[1] * u->h[1]);
    a.czm = u->czm_dev;
    a.czp = u->czp_dev;
    a.omega = omega;
    if (u->desc.dtype == CNV_F64)
        tile_launch<double, TILE_JACOBI, 4>(a, wall, st);
    else
        k == 2 ? tile_launch<float, TILE_JACOBI, 2>(a, wall, st) : tile_launch<float, TILE_JACOBI, 4>(a, wall, st);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

} // namespace cnv
