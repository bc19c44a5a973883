// Adding the sweeps' increment blocks (SweepParts) to the state: a cell takes
// its entry of every block that holds one, the directions in the order x, y,
// z and the blocks of a direction in a fixed order, so the sum does not
// depend on which workgroup wrote first.  Bound by memory: a block's planes
// are read once, in runs along x, with one lane per cell and no branch between
// a direction's loads.  With L planes per segment, TA pencils and CI cells a
// direction holds (L + 2) / L x (TA + 2) / TA x (CI + 1) / CI times q, and more
// where the grid does not fill its last blocks: the three directions 3.9 to
// 4.5 times q on large grids, 6 on 64 x 64 x 48, 10 to 16 on grids of 10 to 20
// cells.  The source pass's conversion with this in it takes 0.97 ms on the full
// domain (250 x 200 x 300, FP64): it moves 6.2 GB, 6.4 TB/s, some of it still in
// the last-level cache (a copy of 6 GB runs at 4.9 TB/s); 0.30 ms in FP32 on 181
// x 160 x 243.  With the parts in the tiles' lane order and a branch per
// neighbour it took 1.59 and 0.48.
#pragma once
#include "bc_src.h"
#include "magic_dev.h"

namespace magic {

// The three directions of one step, and the components of q
template <typename T>
struct StepParts {
    SweepParts<T> d[3];
    int nc;
};

// One coordinate of a cell against the blocks along its axis: up to three
// (block, offset) candidates.  Along a and b a block of W = 2**lg holds
// offsets 0 (the last one of the block before) .. W + 1.
struct Cand {
    int blk, off;
    bool has;
};
// candidate q (0: the cell's own block, 1: the one before, 2: the one after)
__device__ __forceinline__ Cand cand_ab(int q, int x, int lg, int nblk, int last)
{
    const int W = 1 << lg;
    if (q == 0) return {x >> lg, (x & (W - 1)) + 1, x >= 0 && (x >> lg) < nblk};
    if (q == 1) return {(x - 1) >> lg, W + 1, x >= 1 && (x & (W - 1)) == 0};
    return {(x + 1) >> lg, 0, x + 1 <= last && ((x + 1) & (W - 1)) == 0};
}

// acc[m] += direction DIR's increments of cell (i, j, k); j and k are the
// wave's own (scalar), i the lane's.  Lanes without an entry read the nearest
// column's, which a slab that holds them has too.  Along x a lane takes its own block's
// entry and, at an edge, one neighbour's, both loaded without a branch (a
// lane that is at no edge loads its own entry again and drops it), so that
// all loads of a direction are in flight together; the blocks along the other
// axes are the same for the wave.
template <int DIR, typename T>
__device__ __forceinline__ void add_parts(const SweepParts<T> &p, int nc, int i, int j, int k, T (&acc)[10])
{
    const int TA = 1 << p.lgTA, L = 1 << p.lgL;
    const int ncell = p.CI + 1, trow = TA + 2, npos = ncell * trow;
    const int bs = (L + 2) * nc * npos;   // elements of a block
    const int b = DIR == 2 ? j : k;
    if (!p.base || b < -1 || b > p.nB + 2) return;
    // the other scalar axis: a = j (x-sweep), n = j (y), n = k (z)
    const int n = DIR == 1 ? j : k;
    int k0 = 0, r = 0;
    if (DIR == 0) {
        if (j < -1 || j > p.nA + 2) return;
    } else {
        if (n < 1 || n > p.n) return;
        k0 = (int)__umulhi((unsigned)(n - 1), p.iCI);
        r = n - 1 - k0 * p.CI;
    }
    // the lane's axis: own block and offset, and the edge neighbour's
    int lb, lo, eb, eo;
    bool own, edge;
    if (DIR == 0) {
        own = i >= 1 && i <= p.n;
        const int x = min(max(i - 1, 0), p.n - 1);
        lb = (int)__umulhi((unsigned)x, p.iCI);
        lo = x - lb * p.CI + 1;
        edge = own && lo == p.CI;
        eb = lb + 1;
        eo = 0;
    } else {
        const bool in = i >= -1 && i <= p.nA + 2;
        const int x = min(max(i, -1), p.nA + 2);
        lb = x >> p.lgTA;
        lo = (x & (TA - 1)) + 1;
        own = in && x >= 0 && lb < p.nt;
        const bool before = x >= 1 && lo == 1, after = x + 1 <= p.nA + 1 && lo == TA;
        edge = in && (before || after);
        eb = before ? lb - 1 : lb + 1;
        eo = before ? TA + 1 : 0;
        if (lb < 0 || lb >= p.nt) { lb = eb; lo = eo; }   // before the first tile or past the last
    }
    if (!edge) { eb = lb; eo = lo; }
    // blocks run fastest along x: the lanes' blocks are neighbours
    const long long oown = (long long)lb * bs + lo, oedge = (long long)eb * bs + eo;
    const int slow = DIR == 0 ? ncell : trow;      // positions run along x, then along the other in-plane axis
    // the blocks that hold an entry, in a fixed order: usually one, so that
    // only those are gone through (looking at all nine in turn took 30 us on
    // 64 x 64 x 48, 26 now; 24 FP32 grids of 40 x 36 x 60 124 and 95 us)
    int hb = 0, hs = 0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        hb |= cand_ab(q, b, p.lgL, p.ns, p.nB + 1).has ? 1 << q : 0;
        if (DIR == 0) hs |= cand_ab(q, j, p.lgTA, p.nt, p.nA + 1).has ? 1 << q : 0;
    }
    if (DIR != 0) hs = r == p.CI - 1 ? 3 : 1;
    for (int left = (hb & 1 ? hs : 0) | (hb & 2 ? hs << 3 : 0) | (hb & 4 ? hs << 6 : 0); left; left &= left - 1) {
            const int q = __builtin_ctz(left), qb = q >= 6 ? 2 : q >= 3 ? 1 : 0, qs = q - 3 * qb;
            const Cand cb = cand_ab(qb, b, p.lgL, p.ns, p.nB + 1);
            Cand cs;
            if (DIR == 0) cs = cand_ab(qs, j, p.lgTA, p.nt, p.nA + 1);
            else cs = {k0 + qs, qs == 0 ? r + 1 : 0, true};
            const T *src = p.base + (long long)(cb.blk * p.sS + cs.blk * (DIR == 0 ? p.sT : p.sK)) * bs +
                           cb.off * nc * npos + cs.off * slow;
            T v[10], e[10];
#pragma unroll
            for (int m = 0; m < 10; m++)
                if (m < 5 || m < nc) {
                    // plane component of q(m+1)
                    const int tm = DIR == 0 || m == 0 || m > 3 ? m
                                   : DIR == 1 ? (m == 1 ? 2 : m == 2 ? 1 : 3)    // y: a = x, b = z
                                              : (m == 1 ? 2 : m == 2 ? 3 : 1);   // z: a = x, b = y
                    v[m] = src[oown + tm * npos];
                    e[m] = src[oedge + tm * npos];
                }
#pragma unroll
            for (int m = 0; m < 10; m++)
                if (m < 5 || m < nc) {
                    acc[m] += own ? v[m] : T(0.0);
                    acc[m] += edge ? e[m] : T(0.0);
                }
        }
}

// The step's increments of padded cell (ip, jp, kk) (launch: cell_block, a
// wave along x)
template <typename T>
__device__ __forceinline__ void step_parts(const StepParts<T> &sp, int ip, int jp, int kk, int mbc, T (&acc)[10])
{
#pragma unroll
    for (int m = 0; m < 10; m++) acc[m] = T(0.0);
    const int i = ip + 1 - mbc;
    const int j = __builtin_amdgcn_readfirstlane(jp) + 1 - mbc, k = __builtin_amdgcn_readfirstlane(kk) + 1 - mbc;
    add_parts<0>(sp.d[0], sp.nc, i, j, k, acc);
    add_parts<1>(sp.d[1], sp.nc, i, j, k, acc);
    add_parts<2>(sp.d[2], sp.nc, i, j, k, acc);
}

// q += the step's increments, columns ip0 .. ip1-1 of the padded grid (launch:
// slab_cells); on: the control flag of a batch's scenario, or nullptr
template <typename T>
__global__ void k_add_parts(Dims d, T *q, StepParts<T> sp, int ip0, int ip1, const int *on)
{
    if (on && *on == 0) return;
    const int ip = ip0 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int jp = (int)(blockIdx.y * blockDim.y + threadIdx.y);
    if (ip >= ip1 || jp >= d.NY) return;
    const int kk = (int)blockIdx.z;
    const long long c = ((long long)kk * d.NY + jp) * d.NX + ip;
    T acc[10];
    step_parts(sp, ip, jp, kk, d.mbc, acc);
#pragma unroll
    for (int m = 0; m < 10; m++)
        if (m < sp.nc) q[m * d.P + c] = q[m * d.P + c] + acc[m];
}

}  // namespace magic
