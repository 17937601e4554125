// cnv_cols.h -- lanes over block columns, for blocks of any shape.
//
// The z-marching tiles of cnv_march.h need square x-y planes of 16, 32 or 64
// cells.  Every other block shape runs as columns: a lane owns VEC
// consecutive cells of one row of one block and steps through a chunk of z
// planes with the z neighbours in registers; x and y neighbours are loads of
// their own that hit the lines the wave and its neighbours fetch anyway.
// Lanes are numbered through (component, block, z chunk, row, vector) without
// gaps, so a wave holds lanes of several small blocks (8^3 blocks of FP64
// have 32 lanes per plane) and no lane is lost to a plane that is no multiple
// of the wave.
#pragma once

#include "cnv_device.h"

namespace cnv
{

// n / d for 0 <= n < 2^31 by one multiplication: m = floor(2^(31+l) / d) + 1,
// l = ceil(log2 d), so m d - 2^(31+l) <= d <= 2^l and the quotient is exact;
// d > 2^(l-1) keeps m within 32 bits.
struct FastDiv {
    unsigned m;
    int s; // shift of the high word; -1: d = 1
};

inline FastDiv fast_div(unsigned d)
{
    if (d == 1)
        return {0u, -1};
    int l = 1;
    while ((1ull << l) < d)
        ++l;
    return {(unsigned)((1ull << (31 + l)) / d + 1), l - 1};
}

__device__ inline int fdiv(int n, FastDiv d)
{
    return d.s < 0 ? n : (int)(__umulhi((unsigned)n, d.m) >> d.s);
}

constexpr int kColWG = 256;

// The lane numbering of a launch (host-filled).
struct ColShape {
    int lanes;       // per tile: vectors of one x-y plane
    int vx;          // vectors per row
    int nzc, zchunk; // z chunks per block, planes per chunk
    int nbt;         // blocks
    int ntiles;      // components * blocks * z chunks
    WgGrid wgs;
    FastDiv dlanes, dvx, dnzc, dnbt, dnbx, dnby;
};

// Cells per lane: 16-byte rows where nx allows it, else 8-byte, else one.
// (Blocks start at multiples of 32 bytes, so a row of nx % VEC == 0 cells
// starts at a multiple of the vector.)
inline int col_vec(int nx, size_t elem)
{
    const int most = (int)(16 / elem);
    return nx % most == 0 ? most : nx % 2 == 0 ? 2 : 1;
}

// Planes per lane: as many as leave two and a half waves per SIMD (256 CUs x 4
// SIMDs x 64 lanes), since a chunk re-reads its two end planes and pays its
// start-up once.  Measured per Euler step around that line: 24^3 FP32 blocks
// 14.2 us with 311k lanes, 16.3 with 155k and 16.4 with 622k; 48^3 FP64 15.5
// with 187k, 17.5 with 373k, 20.2 with 93k; 40^3 FP64 38.6 with 173k, 42.2
// with 864k; 64 8^3 FP32 blocks 5.7 with one plane per lane, 10.0 with eight.
inline int col_zchunk(const Geom &G, int ncomp, int vec)
{
    const long long vectors = (long long)G.nb[0] * G.nb[1] * G.nb[2] * ncomp * (G.n[0] / vec) * G.n[1] * G.n[2];
    const long long z = vectors / 163840;
    return (int)(z < 1 ? 1 : z > G.n[2] ? G.n[2] : z);
}

// zchunk planes per lane; false when the launch does not fit 32-bit tiles or
// lanes of a plane
inline bool col_shape(const Geom &G, int ncomp, int vec, int zchunk, ColShape &s)
{
    s.vx = G.n[0] / vec;
    if ((long long)s.vx * G.n[1] >= (1LL << 31) - kColWG)
        return false;
    s.lanes = s.vx * G.n[1];
    const long long nbt = (long long)G.nb[0] * G.nb[1] * G.nb[2];
    s.nzc = (G.n[2] + zchunk - 1) / zchunk;
    s.zchunk = (G.n[2] + s.nzc - 1) / s.nzc; // even chunks
    s.nzc = (G.n[2] + s.zchunk - 1) / s.zchunk;
    const long long ntiles = nbt * ncomp * s.nzc;
    const long long nwg = (ntiles * s.lanes + kColWG - 1) / kColWG;
    if (ntiles >= (1LL << 31) - kColWG || nwg >= (1LL << 31) - kColWG)
        return false;
    s.wgs = wg_grid(nwg);
    s.nbt = (int)nbt;
    s.ntiles = (int)ntiles;
    s.dlanes = fast_div((unsigned)s.lanes);
    s.dvx = fast_div((unsigned)s.vx);
    s.dnzc = fast_div((unsigned)s.nzc);
    s.dnbt = fast_div((unsigned)s.nbt);
    s.dnbx = fast_div((unsigned)G.nb[0]);
    s.dnby = fast_div((unsigned)G.nb[1]);
    return true;
}

struct ColLane {
    bool on; // false past the last tile
    int comp, blk, x0, y, z0, z1;
    int nbr[6]; // face-neighbour blocks (periodic)
};

template <int VEC>
__device__ inline ColLane col_lane(const ColShape &s, const Geom &G)
{
    ColLane c;
    // the workgroup's first lane by scalar arithmetic, then 32 bits per lane
    const long long base = (long long)xcd_remap(wg_index(s.wgs), s.wgs.count) * kColWG;
    const int t0 = base < (1LL << 31) ? fdiv((int)base, s.dlanes) : (int)(base / s.lanes);
    const int r = (int)(base - (long long)t0 * s.lanes) + (int)threadIdx.x;
    const int dt = fdiv(r, s.dlanes);
    const int i = r - dt * s.lanes;
    const int tile = t0 + dt;
    c.on = tile < s.ntiles;
    const int q = fdiv(tile, s.dnzc);
    c.z0 = (tile - q * s.nzc) * s.zchunk;
    c.z1 = min(G.n[2], c.z0 + s.zchunk);
    c.comp = fdiv(q, s.dnbt);
    c.blk = q - c.comp * s.nbt;
    c.y = fdiv(i, s.dvx);
    c.x0 = (i - c.y * s.vx) * VEC;
    const int nbx = G.nb[0], nby = G.nb[1], nbz = G.nb[2];
    const int by_ = fdiv(c.blk, s.dnbx), bx = c.blk - by_ * nbx;
    const int bz = fdiv(by_, s.dnby), by = by_ - bz * nby;
    const int lx = nbx, ly = nbx * nby;
    c.nbr[0] = bx > 0 ? c.blk - 1 : c.blk + (nbx - 1);
    c.nbr[1] = bx < nbx - 1 ? c.blk + 1 : c.blk - (nbx - 1);
    c.nbr[2] = by > 0 ? c.blk - lx : c.blk + lx * (nby - 1);
    c.nbr[3] = by < nby - 1 ? c.blk + lx : c.blk - lx * (nby - 1);
    c.nbr[4] = bz > 0 ? c.blk - ly : c.blk + ly * (nbz - 1);
    c.nbr[5] = bz < nbz - 1 ? c.blk + ly : c.blk - ly * (nbz - 1);
    return c;
}

// Where a lane reads one neighbour: cells at p, times s (mirror sign, 1 for
// a copy), or the constant s.
template <typename T>
struct ColNb {
    const T *p;
    T s;
    bool cst;
};

template <typename T, int VEC, bool BC>
__device__ inline VecT<T, VEC> col_load(const ColNb<T> &b, long long o)
{
    VecT<T, VEC> v = load_vec<T, VEC>(b.p + o);
    if (BC)
#pragma unroll
        for (int k = 0; k < VEC; ++k)
            v.v[k] = b.cst ? b.s : b.s * v.v[k];
    return v;
}

template <typename T, bool BC>
__device__ inline T col_load1(const ColNb<T> &b, long long o)
{
    const T v = b.p[o];
    return BC ? (b.cst ? b.s : b.s * v) : v;
}

// Ghost of block face f: from `nbr` in the neighbour block, or by the block's
// rule from its own cells: `edge` (Absorbing) or `mirror` (Symmetry).
template <typename T, bool BC>
__device__ inline ColNb<T> col_ghost(const DevBCHead *h, int f, const T *nbr, const T *edge, const T *mirror)
{
    ColNb<T> r{nbr, (T)1, false};
    if (BC && h) {
        const int k = h->kind[f];
        const T v = (T)h->val[f];
        if (k == FACE_ABSORB) {
            r.p = edge;
        } else if (k == FACE_SYMMETRY) {
            r.p = mirror;
            r.s = v;
        } else if (k == FACE_DIRICHLET) {
            r.p = edge; // a valid address; the value is not used
            r.s = v;
            r.cst = true;
        }
    }
    return r;
}

} // namespace cnv
