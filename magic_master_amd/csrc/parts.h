// Adding the sweeps' increment blocks (SweepParts) to the state: a cell takes
// its entry of every block that holds one, the directions in the order x, y,
// z and the blocks of a direction in a fixed order, so the sum does not
// depend on which workgroup wrote first.  Bound by memory: a block's planes
// are read once (plus the neighbours' edge entries, up to 36 % at 16 planes
// per segment), in runs of a tile's row.
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

// acc[m] += direction DIR's increments of the cell at (n, a, b) (Fortran
// indices along the pencils, the tile axis and the marching axis)
template <int DIR, typename T>
__device__ __forceinline__ void add_parts(const SweepParts<T> &p, int nc, int n, int a, int b, T (&acc)[10])
{
    if (!p.base || n < 1 || n > p.n || a < -1 || a > p.nA + 2 || b < -1 || b > p.nB + 2) return;
    const int TA = 1 << p.lgTA, L = 1 << p.lgL;
    const int ncell = p.CI + 1, trow = TA + 2, npos = ncell * trow;
    const int k0 = (int)__umulhi((unsigned)(n - 1), p.iCI), r = n - 1 - k0 * p.CI;
    // along each axis: the block before (its upper edge), the cell's own, the
    // one after (its lower edge)
#pragma unroll
    for (int ib = 0; ib < 3; ib++) {
        int s, pl;
        if (ib == 0) { s = (b - 1) >> p.lgL; pl = L + 1; if ((b & (L - 1)) != 0 || b < 1) continue; }
        else if (ib == 1) { s = b >> p.lgL; pl = (b & (L - 1)) + 1; if (b < 0 || s >= p.ns) continue; }
        else { s = (b + 1) >> p.lgL; pl = 0; if (((b + 1) & (L - 1)) != 0 || b > p.nB) continue; }
#pragma unroll
        for (int ia = 0; ia < 3; ia++) {
            int t, ai;
            if (ia == 0) { t = (a - 1) >> p.lgTA; ai = TA + 1; if ((a & (TA - 1)) != 0 || a < 1) continue; }
            else if (ia == 1) { t = a >> p.lgTA; ai = (a & (TA - 1)) + 1; if (a < 0 || t >= p.nt) continue; }
            else { t = (a + 1) >> p.lgTA; ai = 0; if (((a + 1) & (TA - 1)) != 0 || a > p.nA) continue; }
#pragma unroll
            for (int in = 0; in < 2; in++) {
                if (in == 1 && r != p.CI - 1) continue;
                const int k = k0 + in, ci = in == 0 ? r + 1 : 0;
                const T *src = p.base + ((long long)((s * p.nk + k) * p.nt + t) * (L + 2) + pl) * nc * npos +
                               (p.pm ? ai * ncell + ci : ci * trow + ai);
#pragma unroll
                for (int m = 0; m < 10; m++) {
                    // plane component of q(m+1)
                    const int tm = DIR == 0 || m == 0 || m > 3 ? m
                                   : DIR == 1 ? (m == 1 ? 2 : m == 2 ? 1 : 3)    // y: a = x, b = z
                                              : (m == 1 ? 2 : m == 2 ? 3 : 1);   // z: a = x, b = y
                    if (m < 5 || m < nc) acc[m] += src[tm * npos];
                }
            }
        }
    }
}

// The step's increments of padded cell (ip, jp, kk)
template <typename T>
__device__ __forceinline__ void step_parts(const StepParts<T> &sp, int ip, int jp, int kk, int mbc, T (&acc)[10])
{
#pragma unroll
    for (int m = 0; m < 10; m++) acc[m] = T(0.0);
    const int i = ip + 1 - mbc, j = jp + 1 - mbc, k = kk + 1 - mbc;
    add_parts<0>(sp.d[0], sp.nc, i, j, k, acc);
    add_parts<1>(sp.d[1], sp.nc, j, i, k, acc);
    add_parts<2>(sp.d[2], sp.nc, k, i, j, acc);
}

// q += the step's increments, every cell (launch: padded_cells)
template <typename T, class G>
__device__ __forceinline__ void b_add_parts(const uint3 BI, Dims d, T *q, const StepParts<T> &sp, const G &gate)
{
    if (!gate.on()) return;
    const int ip = (int)(BI.x * blockDim.x + threadIdx.x);
    const int jp = (int)(BI.y * blockDim.y + threadIdx.y);
    if (ip >= d.NX || jp >= d.NY) return;
    const int kk = (int)BI.z;
    const long long c = ((long long)kk * d.NY + jp) * d.NX + ip;
    T acc[10];
    step_parts(sp, ip, jp, kk, d.mbc, acc);
#pragma unroll
    for (int m = 0; m < 10; m++)
        if (m < sp.nc) q[m * d.P + c] = q[m * d.P + c] + acc[m];
}

template <typename T, class G>
__global__ void k_add_parts(Dims d, T *q, StepParts<T> sp, G gate)
{
    b_add_parts(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, q, sp, gate);
}

}  // namespace magic
