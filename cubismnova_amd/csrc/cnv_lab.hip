// cnv_lab.hip -- FieldLab assembly on the GPU, several lab cells per thread.
//
// Instead of the reference's sequence "inner copy, 26 neighbour copies, then
// each BC in list order" (Block/FieldLab.h:180-224), every region of the lab
// is resolved to one rule: walking the block's BC list backwards, the last BC
// whose slab holds the region decides it; Dirichlet ends the walk, Absorbing
// and Symmetry move it to its source (mirror) and continue with the BCs before
// them.  Cells no BC touches are the block's own values, a periodic
// neighbour's values, or unwritten (edges/corners of non-tensorial labs; sides
// skipped by a non-periodic BC).  That is the same result as the sequential
// passes because every BC pass reads only cells it does not write
// (BC/Absorbing.h:94-102, BC/Symmetry.h:107-113).
//
// Node and face slabs: a block at the upper end of a "plus" dimension holds
// one more element there, so each block's extent (and its lab range) is its
// own, and ghosts below a block count back from the neighbour's own end
// (FieldLabLoader.h:217-219, 236-241).  The all-blocks launch lays every lab
// out in the largest block's geometry, the block's lab in the low corner.
#include "cnv_device.h"

namespace cnv
{

constexpr int kMaxBC = 16;

template <typename T>
struct LabArgs {
    const T *base; // component slab
    Geom G;
    int sb[3], se[3];
    int tens;
    int apply_bc;
    int plus;       // bit d: upper-end blocks one element larger along d
    int L[3];       // lab slot extent (the largest block's lab)
    long long lcells; // L0*L1*L2
    // workgroups per block and per lab plane, planes per workgroup, planes per z chunk
    int wgslot, wgxy, gz, zchunk;
    T *out;
    // single-block mode: block index and the list by value
    int single;
    int block[3];
    int nlist;
    DevBC list[kMaxBC];
    // all-blocks mode: per-block tables (null when no block carries a BC)
    int has_tab;
    const DevBCHead *heads;
    const DevBC *entries;
};

// extent of block B along d (node / face slabs: one more at the upper end)
template <typename T>
__device__ inline int blk_extent(const LabArgs<T> &a, const int *B, int d)
{
    return a.G.n[d] + (((a.plus >> d) & 1) && B[d] == a.G.nb[d] - 1 ? 1 : 0);
}

// The lab falls into 27 regions (below, inside, above the block along each
// axis), and the walk over the BC list takes the same turns for every cell of
// a region: a BC slab is a union of regions, and a cell a BC moved is inside
// the block along that axis (ghost widths are at most the block extent), so no
// later slab holds it along that axis again.  A region is therefore one rule:
// the source element of lab cell (q0, q1, q2) is base + cx q0 + cy q1 +
// cz q2, scaled by up to three mirror signs in order; or a constant; or the
// region is never written.
enum { LAB_NONE = 0, LAB_COPY = 1, LAB_CONST = 2 };
template <typename T>
struct LabRegion {
    long long base, cz;
    int cx, cy; // a row has fewer than 2^31 elements
    int mode, nsign;
    T s[3]; // signs in the order they apply; s[0] the constant
};

template <typename T>
__device__ inline void lab_region(const LabArgs<T> &a, const int B[3], const int N[3], const DevBC *list, int n,
                                  const int r0[3], LabRegion<T> &R)
{
    // position along axis e: coordinate al[e] q[e] + be[e], region reg[e]
    int reg[3] = {r0[0], r0[1], r0[2]};
    int al[3] = {1, 1, 1};
    long long be[3] = {0, 0, 0};
    bool periodic[3] = {true, true, true};
    int skip[3] = {1, 1, 1};
    for (int k = 0; k < n; ++k)
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (list[k].dir == e) {
                periodic[e] = list[k].kind == CNV_BC_BASE;
                skip[e] = list[k].side == 0 ? -1 : 1;
            }
    T cval = (T)0;
    R.mode = LAB_COPY;
    R.nsign = 0;
    R.s[0] = R.s[1] = R.s[2] = (T)1;
    // the last BC whose slab holds the cell decides it; a mirror or edge rule
    // moves it and the BCs before that one follow
    for (int k = a.apply_bc ? n - 1 : -1; k >= 0; --k) {
        const DevBC b = list[k];
        if (b.kind == CNV_BC_BASE)
            continue;
        bool in = true;
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            if (e == b.dir)
                in = in && a.sb[e] != 0 && a.se[e] != 1 // BC::Base::isValidStencil_ (BC/Base.h:73-78)
                     && reg[e] == (b.side == 0 ? -1 : 1);
            else if (!a.tens)
                in = in && reg[e] == 0;
        }
        if (!in)
            continue;
        if (b.kind == CNV_BC_DIRICHLET) {
            R.mode = LAB_CONST;
            cval = (T)b.value;
            break;
        }
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (e == b.dir) {
                reg[e] = 0;
                if (b.kind == CNV_BC_ABSORBING) {
                    al[e] = 0;
                    be[e] = b.side == 0 ? 0 : N[e] - 1;
                } else {
                    al[e] = -al[e];
                    be[e] = (b.side == 0 ? -1 : 2LL * N[e] - 1) - be[e];
                }
            }
        if (b.kind == CNV_BC_SYMMETRY) { // the last sign found applies first
            R.s[2] = R.s[1];
            R.s[1] = R.s[0];
            R.s[0] = (T)b.value;
            ++R.nsign;
        }
    }
    if (R.mode == LAB_CONST) {
        T v = cval;
        if (R.nsign > 0)
            v = R.s[0] * v;
        if (R.nsign > 1)
            v = R.s[1] * v;
        if (R.nsign > 2)
            v = R.s[2] * v;
        R.s[0] = v;
        R.base = 0;
        R.cx = R.cy = 0;
        R.cz = 0;
        return;
    }
    int nb[3], out = 0;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        out += reg[e] != 0;
        if (!periodic[e] && reg[e] == skip[e])
            R.mode = LAB_NONE; // neighbour skipped, never written
        nb[e] = B[e] + reg[e];
        nb[e] = nb[e] < 0 ? a.G.nb[e] - 1 : nb[e] == a.G.nb[e] ? 0 : nb[e];
    }
    if (!a.tens && out > 1)
        R.mode = LAB_NONE; // edge/corner of a non-tensorial lab
    // source in the neighbour's own extent NE; below the block it counts back
    // from the neighbour's end (shift NE - N)
    R.base = (nb[0] + (long long)a.G.nb[0] * (nb[1] + (long long)a.G.nb[1] * nb[2])) * a.G.bstride;
    long long stride = 1;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        const int NE = blk_extent(a, nb, e);
        const long long shift = -(long long)reg[e] * N[e] + (reg[e] < 0 ? NE - N[e] : 0);
        if (e == 0)
            R.cx = al[e];
        else if (e == 1)
            R.cy = al[e] * (int)stride;
        else
            R.cz = al[e] * stride;
        R.base += stride * (be[e] + shift);
        stride *= NE;
    }
}

// A lane owns one (x, y) column of a block's lab, or every gz-th plane of it
// where a workgroup holds several copies of a small lab plane, and steps
// through a chunk of z: the 27 rules of the block go to LDS, a lane keeps the
// three of its column, and each cell is then one load, one store and a handful
// of index instructions (the kernel before ran the BC walk and 64-bit index
// divisions per cell).  kLabPer loads are in flight per lane.  Labs of 512 16^3
// FP64 blocks with 3 ghosts 82 -> 17 us (3.6 TB/s of blocks read and labs
// written), of 512 32^3 FP32 blocks 216 -> 40 us (4.5 TB/s; 60 us when the
// workgroups of neighbouring blocks ran on different XCDs, each re-reading the
// shared lines), of 27 8^3 FP64 blocks 18 -> 7 us.  Bound by the caches' lines
// for the x ghosts (three cells of a 128-byte line) and, small, by the rules.
constexpr int kLabPer = 4;

// ROWS: a row of workgroups per block, where one dimension does not hold them all.
template <typename T, bool ROWS>
__global__ __launch_bounds__(256) void k_lab(const LabArgs<T> a)
{
    __shared__ LabRegion<T> reg[27];
    __shared__ DevBC s_list[kMaxBC];
    const int tid = threadIdx.x;
    int B[3], n = 0;
    // the workgroups of a block, and of neighbouring blocks, on one XCD
    const int wg = xcd_remap(blockIdx.x, gridDim.x);
    const int slot = ROWS ? blockIdx.y : wg / a.wgslot, wl = ROWS ? blockIdx.x : wg - slot * a.wgslot;
    if (a.single) {
        B[0] = a.block[0];
        B[1] = a.block[1];
        B[2] = a.block[2];
        n = a.nlist;
        if (tid < n)
            s_list[tid] = a.list[tid];
    } else {
        const int by_ = slot / a.G.nb[0];
        B[0] = slot - by_ * a.G.nb[0];
        B[2] = by_ / a.G.nb[1];
        B[1] = by_ - B[2] * a.G.nb[1];
        if (a.has_tab) {
            const int off = a.heads[slot].offset;
            n = min(a.heads[slot].count, kMaxBC);
            if (tid < n)
                s_list[tid] = a.entries[off + tid];
        }
    }
    const int N[3] = {blk_extent(a, B, 0), blk_extent(a, B, 1), blk_extent(a, B, 2)};
    if (n > 0)
        __syncthreads();
    if (tid < 27) {
        const int rz = tid / 9, ry = (tid - 9 * rz) / 3;
        const int r[3] = {tid - 9 * rz - 3 * ry - 1, ry - 1, rz - 1};
        LabRegion<T> R;
        lab_region(a, B, N, s_list, n, r, R);
        reg[tid] = R;
    }
    __syncthreads();
    // this lane's column and planes
    const int LX = a.L[0];
    const int zc = wl / a.wgxy;
    const long long lxy = (long long)LX * a.L[1];
    long long i = (long long)(wl - zc * a.wgxy) * 256 + tid;
    int zg = 0;
    if (a.gz > 1) { // lab planes of at most 128 cells: gz of them per workgroup
        zg = tid / (int)lxy;
        i = tid - zg * (int)lxy;
    }
    // the block's own lab extent (smaller blocks fill the low corner of the slot)
    const int ex = N[0] + a.se[0] - 1 - a.sb[0], ey = N[1] + a.se[1] - 1 - a.sb[1],
              ez = N[2] + a.se[2] - 1 - a.sb[2];
    const int y = i < (1LL << 31) ? (int)i / LX : (int)(i / LX);
    const int x = (int)(i - (long long)y * LX);
    if (zg >= a.gz || i >= lxy || x >= ex || y >= ey)
        return;
    const int q0 = x + a.sb[0], q1 = y + a.sb[1];
    const int rxy = (q0 < 0 ? 0 : q0 < N[0] ? 1 : 2) + 3 * (q1 < 0 ? 0 : q1 < N[1] ? 1 : 2);
    long long base[3], cz[3];
    int mode[3];
    bool signs = false;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const LabRegion<T> &R = reg[rxy + 9 * r];
        base[r] = R.base + ((long long)R.cy * q1 + R.cx * q0);
        cz[r] = R.cz;
        mode[r] = R.mode;
        signs = signs || R.mode == LAB_CONST || R.nsign > 0;
    }
    T *out = a.out + slot * a.lcells + i;
    const int z1 = min(ez, (zc + 1) * a.zchunk);
    for (int z0 = zc * a.zchunk + zg; z0 < z1; z0 += kLabPer * a.gz) {
        T v[kLabPer];
#pragma unroll
        for (int k = 0; k < kLabPer; ++k) {
            const int z = z0 + k * a.gz, q2 = z + a.sb[2];
            const bool lo = q2 < 0, hi = q2 >= N[2];
            const int m = lo ? mode[0] : hi ? mode[2] : mode[1];
            const long long b = lo ? base[0] : hi ? base[2] : base[1], c = lo ? cz[0] : hi ? cz[2] : cz[1];
            // a load without a branch: element 0 where nothing is copied
            v[k] = a.base[z < z1 && m == LAB_COPY ? b + c * q2 : 0];
        }
        if (signs)
#pragma unroll
            for (int k = 0; k < kLabPer; ++k) {
                const int q2 = z0 + k * a.gz + a.sb[2];
                const LabRegion<T> &R = reg[rxy + (q2 < 0 ? 0 : q2 < N[2] ? 9 : 18)];
                if (R.mode == LAB_CONST) {
                    v[k] = R.s[0];
                } else {
                    if (R.nsign > 0)
                        v[k] = R.s[0] * v[k];
                    if (R.nsign > 1)
                        v[k] = R.s[1] * v[k];
                    if (R.nsign > 2)
                        v[k] = R.s[2] * v[k];
                }
            }
#pragma unroll
        for (int k = 0; k < kLabPer; ++k) {
            const int z = z0 + k * a.gz, q2 = z + a.sb[2];
            const int m = q2 < 0 ? mode[0] : q2 >= N[2] ? mode[2] : mode[1];
            if (z < z1 && m != LAB_NONE)
                out[lxy * z] = v[k];
        }
    }
}

template <typename T>
static int launch_lab_t(const cnv_grid_s *g, int comp, const cnv_stencil &s, bool apply_bc,
                        bool single, const DevBC *list, int nlist, const int *block, void *out,
                        hipStream_t st)
{
    LabArgs<T> a;
    a.G = geom_of(g);
    a.base = reinterpret_cast<const T *>((const char *)g->data + (size_t)comp * g->component_bytes);
    a.plus = plus_mask(g, comp);
    for (int d = 0; d < 3; ++d) {
        a.sb[d] = s.begin[d];
        a.se[d] = s.end[d];
        // one block: its own lab extent; all blocks: the largest block's
        const int wide = ((a.plus >> d) & 1) && (!single || block[d] == a.G.nb[d] - 1);
        a.L[d] = a.G.n[d] + wide + s.end[d] - 1 - s.begin[d];
    }
    a.tens = s.tensorial ? 1 : 0;
    a.apply_bc = apply_bc ? 1 : 0;
    a.lcells = (long long)a.L[0] * a.L[1] * a.L[2];
    a.out = static_cast<T *>(out);
    a.single = single ? 1 : 0;
    a.nlist = 0;
    a.has_tab = 0;
    a.heads = nullptr;
    a.entries = nullptr;
    long long nslots = 1;
    if (single) {
        for (int d = 0; d < 3; ++d)
            a.block[d] = block[d];
        a.nlist = nlist;
        for (int k = 0; k < nlist; ++k)
            a.list[k] = list[k];
    } else {
        const BCTable &t = g->tables[comp];
        a.has_tab = (t.any && t.heads && t.entries) ? 1 : 0;
        a.heads = t.heads;
        a.entries = t.entries;
        nslots = g->nblocks_total;
        for (int d = 0; d < 3; ++d)
            a.block[d] = 0;
        // per-block lists are read into LDS; longer lists are not supported
        for (const auto &l : g->bcs[comp])
            if (l.size() > (size_t)kMaxBC)
                return fail(CNV_ERR_UNSUPPORTED, "more than 16 BCs on one block");
    }
    if (nslots > 65535)
        return fail(CNV_ERR_UNSUPPORTED, "too many blocks for one lab launch");
    if ((a.lcells + 255) / 256 > 0x7fffffffLL)
        return fail(CNV_ERR_UNSUPPORTED, "lab too large");
    // workgroups per lab plane, or planes per workgroup; z chunks of whole
    // passes until there is one workgroup per SIMD (each builds the block's
    // rules, about 2 us, so more of them cost: the 16^3 labs above take 16.7 us
    // with 1024 and 19.4 with 3072)
    const long long lxy = (long long)a.L[0] * a.L[1];
    a.gz = lxy <= 128 ? (int)(256 / lxy) : 1;
    const long long wgxy = (lxy + 255) / 256;
    if (wgxy > 0x7fffffffLL)
        return fail(CNV_ERR_UNSUPPORTED, "lab too large");
    a.wgxy = (int)wgxy;
    const int per = kLabPer * a.gz; // planes of one pass
    int nzc = 1;
    const int passes = (a.L[2] + per - 1) / per;
    while (wgxy * nslots * nzc < 1024 && nzc < passes)
        ++nzc;
    a.zchunk = (passes + nzc - 1) / nzc * per;
    nzc = (a.L[2] + a.zchunk - 1) / a.zchunk;
    const long long gx = wgxy * nzc;
    const long long most = (1LL << 24) - 1; // a dimension of 2^32 threads or more is cut off without an error
    if (gx > most)
        return fail(CNV_ERR_UNSUPPORTED, "lab too large");
    a.wgslot = (int)gx;
    if (gx * nslots <= most)
        hipLaunchKernelGGL((k_lab<T, false>), dim3((unsigned)(gx * nslots)), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((k_lab<T, true>), dim3((unsigned)gx, (unsigned)nslots), dim3(256), 0, st, a);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

int launch_lab(const cnv_grid_s *g, int comp, const cnv_stencil &s, bool apply_bc, bool single,
               const DevBC *list, int nlist, const int *block, void *out, hipStream_t st)
{
    if (g->desc.dtype == CNV_F64)
        return launch_lab_t<double>(g, comp, s, apply_bc, single, list, nlist, block, out, st);
    return launch_lab_t<float>(g, comp, s, apply_bc, single, list, nlist, block, out, st);
}

// ---------------------------------------------------------------- fill

template <typename T>
__global__ __launch_bounds__(256) void k_fill(T *dst, T v, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        dst[i] = v;
}

int launch_fill(void *dst, int dtype, double value, size_t count, hipStream_t st)
{
    if (count == 0)
        return CNV_OK;
    size_t blocks = (count + 255) / 256;
    if (blocks > 65536)
        blocks = 65536;
    if (dtype == CNV_F64)
        hipLaunchKernelGGL(k_fill<double>, dim3((unsigned)blocks), dim3(256), 0, st, (double *)dst,
                           value, count);
    else
        hipLaunchKernelGGL(k_fill<float>, dim3((unsigned)blocks), dim3(256), 0, st, (float *)dst,
                           (float)value, count);
    CNV_HIP(hipGetLastError());
    return CNV_OK;
}

} // namespace cnv
