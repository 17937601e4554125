// cnv_run2.hip -- two Euler steps per launch on tiles of the domain that march
// through z, for any block shape.
//
// One step per launch moves the field through memory once per step (14.8 us for
// 144 x 96 x 120 x 3 FP32 cells in 24^3 blocks).  Here a workgroup of 16 rows of
// 16 lanes, 16 bytes of cells each, takes the planes of a domain tile one after
// another: a lane holds its cells of six planes (loaded three planes before their
// use), the row's x neighbours come from the next lanes by DPP, the y neighbours
// through LDS, and step 2 of the plane before runs behind step 1 of this one, so
// there is one barrier per plane.  The outer lane on each side and two rows on each
// side only feed their neighbours: 14 of 16 lanes and 12 of 16 rows give output.
// Block boundaries exist only in a lane's offset, computed once, and in the
// plane's offset (scalar).  Past a wall nothing is used: a cell next to a wall
// reads the wall's constant or its own value times the wall's factor.  Every
// value is the single step's expression on the same operands: bit-identical.
//
// Bound by VALU issue (about 115 instructions per lane and plane for eight FP32
// evaluations, 70 % of the issue slots at 256^3) and, on medium grids, by the last
// wave of workgroups.  us per step with norms, single steps / here: the field
// above 14.8 / 10.7, 128^3 FP64 in 8^3 blocks 8.9 / 6.9, 200^3 FP64 in 40^3 28.4 /
// 17.9, 256^3 in 64^3 blocks 26.3 / 17.9 FP32, 46.3 / 35.6 FP64.  512 or 1024
// threads (28 or 60 rows of output), two rows per thread, or 32 lanes per row
// evaluate less halo but leave fewer tiles: 11.5, 14.0, 12.6 and 11.8 us on
// the field above, 20.8, 24.1, 21.8 and 22.3 against 18.9 on 256^3 FP32.
#include "cnv_cols.h"

#include <algorithm>
#include <type_traits>

namespace cnv
{

struct Run2Args {
    const char *u; // component slabs
    char *out;
    long long cs_u, cs_o; // bytes per component
    unsigned bstride;     // bytes per block
    int nb[3], n[3], ng[3], nt[3];
    FastDiv dn[3];
    int zchunk, ntiles; // ntiles: of all components
    RunRules rules;
    double ih2[3], nudt;
    double *part; // norms: part[j * ntiles + tile]
    const double *prev_p;
    int nprev, prev_n;
    double *prev_out;
};

// the next (UP) or previous lane's value in a row of 16 lanes (at its ends the
// lane's own)
template <typename T, bool UP>
__device__ inline T lane_nbr(T v)
{
    constexpr int CTRL = UP ? 0x101 : 0x111; // row_shl / row_shr by one
    if constexpr (sizeof(T) == 4) {
        const int i = __builtin_bit_cast(int, v);
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(i, i, CTRL, 0xf, 0xf, false));
    } else {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        const int l = (int)(unsigned)b, h = (int)(unsigned)(b >> 32);
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(l, l, CTRL, 0xf, 0xf, false);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(h, h, CTRL, 0xf, 0xf, false);
        return __builtin_bit_cast(T, (unsigned long long)hi << 32 | lo);
    }
}

constexpr int kRun2WG = 256;

// VECL: the rows of a block
// are whole vectors.  WALL: some domain face is no periodic neighbour
template <typename T, bool VECL, bool WALL, bool NORM>
__global__ __launch_bounds__(kRun2WG) void k_run2(const Run2Args a)
{
    constexpr int WG = kRun2WG, LR = 16; // threads, lanes per row
    constexpr int VEC = 16 / (int)sizeof(T), ROWS = WG / LR, CX = (LR - 2) * VEC, CY = ROWS - 4;
    constexpr unsigned TS = sizeof(T);
    using V = VecT<T, VEC>;
    __shared__ alignas(16) T sU[2][(ROWS + 2) * LR * VEC], sV[2][(ROWS + 2) * LR * VEC];
    __shared__ double red[2 * (WG / 64)];

    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= a.ntiles) { // a workgroup for each deferred sum
        const int k = blockIdx.x - a.ntiles;
        wg_sum_partials<WG>(a.prev_p + (size_t)k * a.prev_n, a.prev_n, a.prev_out + k, red);
        return;
    }
    const int tile = xcd_remap(blockIdx.x, a.ntiles);
    int t = tile;
    const int tz = t % a.nt[2];
    t /= a.nt[2];
    const int tx = t % a.nt[0];
    t /= a.nt[0];
    const int ty = t % a.nt[1], comp = t / a.nt[1];
    const int NX = a.ng[0], NY = a.ng[1], NZ = a.ng[2];
    const int Z0 = tz * a.zchunk, nz = min(a.zchunk, NZ - Z0);
    const int q = tid % LR, r = tid / LR;
    const int gx = tx * CX + (q - 1) * VEC, gy = ty * CY + r - 2;
    const char *ub = a.u + (long long)comp * a.cs_u;
    char *ob = a.out + (long long)comp * a.cs_o;
    const DevRules rules = rules_of(a.rules, offsetof(Run2Args, rules), WALL ? comp : 0);

    // cell index inside the domain: periodic axes wrapped, walls clamped
    // (cells past a wall are loaded and never used)
    auto inside = [&](int g, int d, int n, int last) {
        if (!WALL || rules->fm[2 * d] == FM_PERIODIC) {
            g %= n;
            return g < 0 ? g + n : g;
        }
        return min(max(g, 0), last);
    };
    // byte offset of the lane's cells in a layer of blocks (fewer than 2^32
    // bytes, host-checked)
    unsigned off[VECL ? 1 : VEC];
    {
        const int y = inside(gy, 1, NY, NY - 1), by = fdiv(y, a.dn[1]);
        const unsigned oy = (unsigned)(by * a.nb[0]) * a.bstride + (unsigned)((y - by * a.n[1]) * a.n[0]) * TS;
#pragma unroll
        for (int v = 0; v < (VECL ? 1 : VEC); ++v) {
            const int x = inside(gx + v, 0, NX, NX - (VECL ? VEC : 1)), bx = fdiv(x, a.dn[0]);
            off[v] = oy + (unsigned)bx * a.bstride + (unsigned)(x - bx * a.n[0]) * TS;
        }
    }
    // the byte offset of a plane, advanced plane by plane (uniform)
    const unsigned pbytes = (unsigned)(a.n[0] * a.n[1]) * TS;
    const long long layer = (long long)(a.nb[0] * a.nb[1]) * a.bstride, skip = layer - (long long)pbytes * (a.n[2] - 1);
    struct Plane {
        long long off;
        int z, l; // in the domain and in its block
    };
    auto plane = [&](int z) {
        const int b = fdiv(z, a.dn[2]), l = z - b * a.n[2];
        return Plane{b * layer + (long long)pbytes * l, z, l};
    };
    auto next = [&](Plane p) {
        const bool end = p.l == a.n[2] - 1;
        p.off += end ? skip : (long long)pbytes;
        p.l = end ? 0 : p.l + 1;
        ++p.z;
        return p;
    };
    const bool pz = !WALL || rules->fm[4] == FM_PERIODIC;
    Plane in = plane(inside(Z0 - 2, 2, NZ, NZ - 1)), out = plane(Z0);
    int zin = Z0 - 2; // plane of the next load; `in` is it wrapped or clamped
    auto load = [&]() __attribute__((always_inline)) {
        const auto p = buf_rsrc(ub + in.off, ~0u);
        const bool go = pz || (zin >= 0 && zin < NZ - 1), wrap = in.z == NZ - 1;
        const Plane n = next(in);
        in.off = go ? (wrap ? 0 : n.off) : in.off;
        in.z = go ? (wrap ? 0 : n.z) : in.z;
        in.l = go ? (wrap ? 0 : n.l) : in.l;
        ++zin;
        V v;
        if constexpr (VECL) {
            v = buf_load<T, VEC>(p, off[0], 0);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e)
                v.v[e] = buf_load1<T>(p, off[e], 0);
        }
        return v;
    };

    const bool corex = q >= 1 && q <= LR - 2 && gx < NX;
    const bool core = corex && r >= 2 && r < ROWS - 2 && gy < NY;
    const bool wcore = __builtin_amdgcn_ballot_w64(core) != 0; // any in the wave
    const int lo = ((r + 1) * LR + q) * VEC;
    const T ihx2 = (T)a.ih2[0], ihy2 = (T)a.ih2[1], ihz2 = (T)a.ih2[2], nudt = (T)a.nudt;
    // walls next to the lane's cells; the w* flags are uniform in a wave
    const bool xlo = WALL && rules->fm[0] != FM_PERIODIC && gx == 0;
    const int xhi = WALL && rules->fm[1] != FM_PERIODIC ? NX - 1 - gx : -1; // element next to the upper wall
    const bool ylo = WALL && rules->fm[2] != FM_PERIODIC && gy == 0;
    const bool yhi = WALL && rules->fm[3] != FM_PERIODIC && gy == NY - 1;
    const bool wx = WALL && __builtin_amdgcn_ballot_w64(xlo || (xhi >= 0 && xhi < VEC)) != 0;
    const bool wy = WALL && __builtin_amdgcn_ballot_w64(ylo || yhi) != 0;
    auto wall = [&](int d, int side, T v) __attribute__((always_inline)) {
        const int k = rules->fm[2 * d + side];
        return k == FM_CONST ? (T)rules->v[2 * d + side] : k == FM_MIRROR ? (T)rules->v[2 * d + side] * v : v;
    };
    // one step of plane z from its own and the neighbouring planes, in the
    // single step's order
    auto step = [&](const V &c, V zm, V zp, const T *s, int z) __attribute__((always_inline)) {
        V ym = *reinterpret_cast<const V *>(s + lo - LR * VEC), yp = *reinterpret_cast<const V *>(s + lo + LR * VEC);
        V res;
        T xl = lane_nbr<T, false>(c.v[VEC - 1]);
        const T xr = lane_nbr<T, true>(c.v[0]);
        V xp;
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            xp.v[v] = v == VEC - 1 ? xr : c.v[v + 1];
        if constexpr (WALL) {
            if (wx) {
                xl = xlo ? wall(0, 0, c.v[0]) : xl;
#pragma unroll
                for (int v = VECL ? VEC - 1 : 0; v < VEC; ++v)
                    xp.v[v] = xhi == v ? wall(0, 1, c.v[v]) : xp.v[v];
            }
            if (wy) {
#pragma unroll
                for (int v = 0; v < VEC; ++v) {
                    ym.v[v] = ylo ? wall(1, 0, c.v[v]) : ym.v[v];
                    yp.v[v] = yhi ? wall(1, 1, c.v[v]) : yp.v[v];
                }
            }
            if (z == 0 && rules->fm[4] != FM_PERIODIC)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    zm.v[v] = wall(2, 0, c.v[v]);
            if (z == NZ - 1 && rules->fm[5] != FM_PERIODIC)
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    zp.v[v] = wall(2, 1, c.v[v]);
        }
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
            const T e = c.v[v], l = v == 0 ? xl : c.v[v - 1];
            const T ddx = ihx2 * (fms2(e, xp.v[v]) + l);
            const T ddy = ihy2 * (fms2(e, yp.v[v]) + ym.v[v]);
            const T ddz = ihz2 * (fms2(e, zp.v[v]) + zm.v[v]);
            const T lap = ddx + ddy + ddz;
            const T d = lap * nudt;
            res.v[v] = e + d;
        }
        return res;
    };

    // Plane i (z = Z0 - 2 + i) of the input is in slot i % 6 of a register ring,
    // loaded four planes ahead, of the first step in slot i % 3; the current
    // planes' y neighbours in LDS, two planes each
    V u[6], w[3];
    double s1 = 0.0, s2 = 0.0;
    auto put = [&](T *s, const V &v) __attribute__((always_inline)) { *reinterpret_cast<V *>(s + lo) = v; };
#pragma unroll
    for (int i = 0; i < 5; ++i)
        u[i] = load();
    put(sU[1], u[1]);
    __syncthreads();
    // step 1 of plane i, in slots k = i mod 6
    auto first = [&](auto kk, int i) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        u[(k + 4) % 6] = load();
        w[k % 3] = step(u[k], u[(k + 5) % 6], u[(k + 1) % 6], sU[k % 2], Z0 - 2 + i);
    };
    auto share = [&](auto kk) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        put(sU[(k + 1) % 2], u[(k + 1) % 6]);
        put(sV[k % 2], w[k % 3]);
        __syncthreads();
    };
    // step 2 of plane i - 1
    auto second = [&](auto kk, int i) __attribute__((always_inline)) {
        constexpr int k = decltype(kk)::value;
        const auto p = buf_rsrc(ob + out.off, ~0u);
        out = next(out);
        if (!wcore)
            return;
        const V c = w[(k + 2) % 3];
        const V o = step(c, w[(k + 1) % 3], w[k % 3], sV[(k + 1) % 2], Z0 - 3 + i);
        if (core) {
            if (NORM) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const bool have = VECL || gx + e < NX;
                    const double d1 = have ? (double)c.v[e] : 0.0, d2 = have ? (double)o.v[e] : 0.0;
                    s1 = __builtin_fma(d1, d1, s1);
                    s2 = __builtin_fma(d2, d2, s2);
                }
            }
            if constexpr (VECL) {
                buf_store<T, VEC>(p, off[0], 0, o);
            } else {
#pragma unroll
                for (int e = 0; e < VEC; ++e)
                    if (gx + e < NX)
                        buf_store1<T>(p, off[e], 0, o.v[e]);
            }
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    using I5 = std::integral_constant<int, 5>;
    first(I1(), 1);
    share(I1());
    first(I2(), 2);
    share(I2());
    int i = 3;
    const int last = nz + 2;
    auto both = [&](auto kk) __attribute__((always_inline)) {
        first(kk, i);
        second(kk, i);
        share(kk);
        return ++i > last;
    };
    for (;;)
        if (both(I3()) || both(I4()) || both(I5()) || both(I0()) || both(I1()) || both(I2()))
            break;

    if (NORM) { // per-tile partials of both steps in a fixed wave tree and wave order
        double acc[2] = {s1, s2};
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j] += __shfl_xor(acc[j], o, 64);
        if ((tid & 63) == 0)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                red[j * (WG / 64) + tid / 64] = acc[j];
        __syncthreads();
        if (tid < 2) {
            double s = 0.0;
            for (int k = 0; k < WG / 64; ++k)
                s += red[tid * (WG / 64) + k];
            a.part[(size_t)tid * a.ntiles + tile] = s;
        }
    }
}

// ---------------------------------------------------------------- host side

template <typename T>
static bool run2_layout(const cnv_grid_s *u, Run2Args &a, int ncomp, int zchunk)
{
    constexpr int VEC = 16 / (int)sizeof(T), CX = 14 * VEC, CY = kRun2WG / 16 - 4;
    const Geom G = geom_of(u);
    const unsigned long long layer = (unsigned long long)u->block_bytes * G.nb[0] * G.nb[1];
    if (layer >= (1ull << 32))
        return false;
    a.bstride = (unsigned)u->block_bytes;
    const int c[3] = {CX, CY, zchunk};
    long long nt = ncomp;
    for (int d = 0; d < 3; ++d) {
        a.nb[d] = G.nb[d];
        a.n[d] = G.n[d];
        a.ng[d] = G.nb[d] * G.n[d];
        a.nt[d] = (a.ng[d] + c[d] - 1) / c[d];
        a.dn[d] = fast_div((unsigned)G.n[d]);
        nt *= a.nt[d];
    }
    a.zchunk = zchunk;
    if (nt >= (1LL << 32) / kRun2WG - 4) // (and the deferred sums: fewer than 2^32 threads)
        return false;
    a.ntiles = (int)nt;
    return true;
}

template <typename T, bool VECL>
static void run2_launch(const Run2Args &a, bool wall, hipStream_t st)
{
    const dim3 g((unsigned)(a.ntiles + a.nprev)), b(kRun2WG);
    if (wall) {
        if (a.part)
            hipLaunchKernelGGL((k_run2<T, VECL, true, true>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((k_run2<T, VECL, true, false>), g, b, 0, st, a);
    } else {
        if (a.part)
            hipLaunchKernelGGL((k_run2<T, VECL, false, true>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((k_run2<T, VECL, false, false>), g, b, 0, st, a);
    }
}

// tiles of a launch with z chunks of zchunk planes; 0: not available
static int run2_count(const cnv_grid_s *u, int zchunk)
{
    Run2Args a;
    const bool ok = u->desc.dtype == CNV_F64 ? run2_layout<double>(u, a, u->desc.ncomp, zchunk)
                                             : run2_layout<float>(u, a, u->desc.ncomp, zchunk);
    return ok ? a.ntiles : 0;
}

// The tiles of a launch and their z chunk.  A chunk of z planes evaluates z + 2
// and loads z + 4, so deep chunks do less work until the tiles no longer fill the
// GPU: about 900 tiles, between 4 and 32 planes (us per step at 4 / 8 / 12 / 16 /
// 32 planes: 128^3 FP64 in 55 columns of tiles 6.9 / 7.0 / 7.0 / 6.9 / 8.6, the
// field above in 72 columns 11.4 / 10.7 / 10.6 / 12.1 / 17.1, 256^3 FP32 in 110
// columns 23.8 / 22.5 / 21.8 / 19.6 / 18.9, FP64 in 220 41.7 / 47.6 / 42.8 / 38.4 /
// 35.8).
int run2_tiles(const cnv_grid_s *u, int *zchunk)
{
    const int nz = u->desc.nblocks[2] * u->desc.block_cells[2];
    const int xy = run2_count(u, nz);
    if (xy == 0)
        return 0;
    const int chunks = (900 + xy - 1) / xy;
    *zchunk = std::min(std::max((nz + chunks - 1) / chunks, 4), 32);
    return run2_count(u, *zchunk);
}

int launch_run2(cnv_grid_s *u, cnv_grid_s *out, int ncomp, int zchunk, double nu_dt, double *part, const double *prev_p,
                int nprev, int prev_n, double *prev_out, const RunRules *rules, hipStream_t st)
{
    Run2Args a{};
    const bool f64 = u->desc.dtype == CNV_F64;
    if (!(f64 ? run2_layout<double>(u, a, ncomp, zchunk) : run2_layout<float>(u, a, ncomp, zchunk)))
        return fail(CNV_ERR_UNSUPPORTED, "grid too large for two steps per launch");
    a.u = static_cast<const char *>(u->data);
    a.out = static_cast<char *>(out->data);
    a.cs_u = (long long)u->component_bytes;
    a.cs_o = (long long)out->component_bytes;
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
    const bool wall = rules != nullptr, vec = u->desc.block_cells[0] % (f64 ? 2 : 4) == 0;
    if (f64)
        vec ? run2_launch<double, true>(a, wall, st) : run2_launch<double, false>(a, wall, st);
    else
        vec ? run2_launch<float, true>(a, wall, st) : run2_launch<float, false>(a, wall, st);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

} // namespace cnv
