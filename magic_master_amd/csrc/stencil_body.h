// Boundary, pre-step and diffusion/conduction stencil kernels shared by the
// FP64 form (T = double, coefficients as 3-D planes) and the FP32
// perturbation form (T = float, coefficients as background columns, COLC).
// bc_src.hip and bc_src32.hip instantiate them under their own
// floating-point contraction settings.
//
// Index convention: a cell with Fortran indices (i, j, k) in
// [1-mbc, mx+mbc] x [1-mbc, my+mbc] x [1-mbc, mz+mbc] lives at
// ((k+mbc-1)*NY + (j+mbc-1))*NX + (i+mbc-1) of every plane.
#pragma once
#include "bc_src.h"

// Every kernel below takes a gate G: GridGate (factors as passed) for one grid; the batched driver passes a gate that reads its scenario's
// step-control block on the device (skip when the scenario is idle in this
// stage, factors that depend on the scenario's dt).

namespace magic {

__device__ __forceinline__ long long cid(const Dims &d, int i, int j, int k)
{
    return ((long long)(k + d.mbc - 1) * d.NY + (j + d.mbc - 1)) * d.NX + (i + d.mbc - 1);
}

// The cell whose value bc3's x and y passes (bc3_mpi.f:97-312, 320-536) leave
// at (i, j, k): its column, whether the x or y momentum changes sign on the
// way, and whether any face writes the cell at all (else it is the cell
// itself).  The y pass comes after the x pass, so a row beyond y takes its
// source row's value with that row's x ghosts; periodic faces copy interior
// layers only, in x interior rows only.
struct GhostSrc {
    int i, j;
    bool fx, fy, def;
};
__device__ __forceinline__ GhostSrc xy_source(const Dims &d, const Faces &f, int i, int j, int k)
{
    GhostSrc s = {i, j, false, false, false};
    const bool kin = k >= 1 && k <= d.mz;
    while (s.j < 1 || s.j > d.my) {   // once, or more often where my < mbc
        const bool lo = s.j < 1;
        const int m = lo ? f.m[2] : f.m[3];
        if (m == 1) s.j = lo ? 1 : d.my;
        else if (m == 3) { s.j = (lo ? 1 : 2 * d.my + 1) - s.j; s.fy = !s.fy; }
        else if (m == 2 && kin) s.j += lo ? d.my : -d.my;
        else break;
        s.def = true;
    }
    while (s.i < 1 || s.i > d.mx) {
        const bool lo = s.i < 1;
        const int m = lo ? f.m[0] : f.m[1];
        if (m == 1) s.i = lo ? 1 : d.mx;
        else if (m == 3) { s.i = (lo ? 1 : 2 * d.mx + 1) - s.i; s.fx = !s.fx; }
        else if (m == 2 && kin && s.j >= 1 && s.j <= d.my) s.i += lo ? d.mx : -d.mx;
        else break;
        s.def = true;
    }
    return s;
}

// bc3 (bc3_mpi.f:5-812) in one pass: a lane per ghost cell writes what the
// reference's x, y and z passes leave there, taken straight from the interior
// cell that it comes from, all components; no lane reads a cell that another
// writes.  The three passes as kernels of their own took 30 us on small
// grids, most of it three launches of a few waves with a chain of loads each.
// f.m: the faces (0: skipped).  zf(m, side, kbc, v, cg, cb, col): the z
// pass's scaling of component m (stencil for faces 1 and 3; z faces need mz >=
// mbc, the host runs them apart otherwise).  CLAMP_BC: b4step3 (b4step3.f:35-45,
// tracers clamped to [0, 1] on every cell) with it.  UVW_BC: diffuse's own z
// ghosts of q(2:4) (diffuse.f:48-54) after the x and y faces.
template <typename T, class ZF, class G>
__device__ __forceinline__ void b_bc(const uint3 BI, Dims d, T *q, int nc, const Faces &f, int mode, const ZF &zf,
                                     const G &gate)
{
    if (!gate.on()) return;
    unsigned e = BI.x * 256u + (unsigned)(threadIdx.y * blockDim.x + threadIdx.x);
    const bool clamp = (mode & CLAMP_BC) != 0 && nc > 5;
    int part = 0;
    while (part < 4 && e >= bc_lanes(d, part)) e -= bc_lanes(d, part++);
    if (part == 4 || (part == 3 && !clamp)) return;
    const unsigned g = 2u * d.mbc;
    auto ghost = [&](unsigned x, int n) { return (int)x < d.mbc ? (int)x + 1 - d.mbc : n + 1 + (int)x - d.mbc; };
    int i, j, k;
    if (part == 0) {
        const unsigned r = e / d.NX;
        i = (int)(e - r * d.NX) + 1 - d.mbc;
        const unsigned l = r / d.NY;
        j = (int)(r - l * d.NY) + 1 - d.mbc;
        k = ghost(l, d.mz);
    } else if (part == 1) {
        const unsigned r = e / d.NX;
        i = (int)(e - r * d.NX) + 1 - d.mbc;
        const unsigned l = r / g;
        j = ghost(r - l * g, d.my);
        k = (int)l + 1;
    } else if (part == 2) {
        const unsigned r = e / g;
        i = ghost(e - r * g, d.mx);
        const unsigned l = r / d.my;
        j = (int)(r - l * d.my) + 1;
        k = (int)l + 1;
    } else {
        const unsigned r = e / d.mx;
        i = (int)(e - r * d.mx) + 1;
        const unsigned l = r / d.my;
        j = (int)(r - l * d.my) + 1;
        k = (int)l + 1;
    }
    const long long cg = cid(d, i, j, k);
    const int side = k < 1 ? 0 : 1, kbc = k < 1 ? 1 - k : k - d.mz;
    const int mz = part == 0 ? f.m[4 + side] : 0;
    const int kb = part == 0 && (mz == 1 || mz == 3) ? (side == 0 ? 1 : d.mz) : mz == 2 ? (side == 0 ? k + d.mz : k - d.mz) : k;
    const GhostSrc s = xy_source(d, f, i, j, kb);
    const long long cb = cid(d, s.i, s.j, kb);
    const bool def = s.def || mz != 0;
    const long long col = (long long)(j + d.mbc - 1) * d.NX + (i + d.mbc - 1);
    // the boundary cell of the cell's own column: the z pass's background
    const long long cc = cid(d, i, j, kb);
    // diffuse's z ghosts: the column's first or last interior layer
    const bool uvw = (mode & UVW_BC) != 0 && part == 0;
    GhostSrc s2 = s;
    long long cu = cb;
    if (uvw || mz == 3) {   // the mirrored layer of a wall, or the edge layer
        const int kl = uvw ? (side == 0 ? 1 : d.mz) : (side == 0 ? kbc : d.mz + 1 - kbc);
        s2 = xy_source(d, f, i, j, kl);
        cu = cid(d, s2.i, s2.j, kl);
    }
#pragma unroll
    for (int m = 0; m < 10; m++) {
        if (m >= 5 && m >= nc) break;
        const T *p = q + (long long)m * d.P;
        const bool edge = (uvw && m >= 1 && m <= 3) || (mz == 3 && m == 3);
        T v = p[edge ? cu : cb];
        if (m == 1 && (edge ? s2.fx : s.fx)) v = -v;
        if (m == 2 && (edge ? s2.fy : s.fy)) v = -v;
        if (mz == 3 && m == 3) v = -v;
        else if (mz == 1 || mz == 3) v = zf(m, side, kbc, v, cg, cc, col);
        const bool cl = clamp && m >= 5;
        const T raw = v;
        if (cl) v = fmaxD(T(0.0), fminD(v, T(1.0)));
        // an interior tracer already within its range is only read
        if (part == 3 ? cl && !(v == raw) : (def || edge || cl)) q[(long long)m * d.P + cg] = v;
    }
}
template <typename T, class ZF, class G>
__global__ __launch_bounds__(256) void k_bc(Dims d, T *q, int nc, Faces f, int mode, ZF zf, G gate)
{
    b_bc(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, q, nc, f, mode, zf, gate);
}

// b4step3.f:35-45: clamp tracers to [0, 1] on every cell.
template <typename T, class G>
__device__ __forceinline__ void b_clamp(const uint3 BI, T *q, long long P, int nc, const G &gate)
{
    if (!gate.on()) return;
    const long long c = (long long)BI.x * blockDim.x + threadIdx.x;
    if (c >= P) return;
    for (int m = 5; m < nc; m++) {
        const T v = q[m * P + c];
        q[m * P + c] = fmaxD(T(0.0), fminD(v, T(1.0)));
    }
}
template <typename T, class G>
__global__ void k_clamp(T *q, long long P, int nc, G gate)
{
    b_clamp(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, q, P, nc, gate);
}

// Interior thread mapping: x fastest.
#define INTERIOR_IJK                                                          \
    const int i = (int)(BI.x * blockDim.x + threadIdx.x) + 1;                \
    const int j = (int)(BI.y * blockDim.y + threadIdx.y) + 1;                \
    const int k = (int)BI.z + 1;                                             \
    if (i > d.mx || j > d.my) return;                                         \
    const long long c = cid(d, i, j, k);

// All-cells thread mapping over the padded grid: x fastest; kk is the
// padded layer index (k + mbc - 1).
#define PADDED_IJK                                                            \
    const int ip = (int)(BI.x * blockDim.x + threadIdx.x);                   \
    const int jp = (int)(BI.y * blockDim.y + threadIdx.y);                   \
    if (ip >= d.NX || jp >= d.NY) return;                                     \
    const int kk = (int)BI.z;                                                \
    const long long c = ((long long)kk * d.NY + jp) * d.NX + ip;

// diffuse.f:70-118: cross-derivative terms of q(2:4) (after the z-ghost
// fill), written to the interior of the three planes of u; q is not
// changed (its planes keep the values the reference's copy holds, whose
// ghost layers the directional passes read).  A workgroup covers 64 x-cells
// by 4 y-rows and marches over kb layers, holding q(2:4) of three
// consecutive layers with a one-cell halo in x and y in LDS, so each value
// is read from memory once per workgroup.  Launch: block (64, 4), grid
// (ceil(mx/64), ceil(my/4), ceil(mz/kb)).
template <typename T, bool COLC, class G>
__device__ __forceinline__ void b_diff_cross(const uint3 BI, Dims d, T *u, const T *q, const T *coef, T dxy, T dxz, T dyz, int kb, const G &gate)
{
    if (!gate.on()) return;
    dxy = gate.f(dxy, 0);
    dxz = gate.f(dxz, 1);
    dyz = gate.f(dyz, 2);
    constexpr int TX = 66, TL = TX * 6;     // (64 + 2) x (4 + 2) cells per layer
    __shared__ T s[3][3][TL];               // [layer k mod 3][component][cell]
    const int tx = (int)threadIdx.x, ty = (int)threadIdx.y, t = ty * 64 + tx;
    const int i0 = (int)BI.x * 64 + 1, j0 = (int)BI.y * 4 + 1;
    const int k0 = (int)BI.z * kb + 1;
    const int k1 = k0 + kb - 1 < d.mz ? k0 + kb - 1 : d.mz;
    const int i = i0 + tx, j = j0 + ty;
    const bool own = i <= d.mx && j <= d.my;
    const T *u1 = q + d.P, *u2 = q + 2 * d.P, *u3 = q + 3 * d.P;
    // layer kk (0 <= kk <= mz + 1) of the tile and its halo; cells past
    // mx + 1 or my + 1 are not read by any interior cell
    auto load = [&](int kk) {
        const int sl = kk % 3;
        for (int e = t; e < TL; e += 256) {
            const int ii = i0 - 1 + e % TX, jj = j0 - 1 + e / TX;
            if (ii <= d.mx + 1 && jj <= d.my + 1) {
                const long long c = cid(d, ii, jj, kk);
                s[sl][0][e] = u1[c];
                s[sl][1][e] = u2[c];
                s[sl][2][e] = u3[c];
            }
        }
    };
    load(k0 - 1);
    load(k0);
    const int e = (ty + 1) * TX + tx + 1;   // this lane's cell in the tile
    for (int k = k0; k <= k1; k++) {
        load(k + 1);   // into the slot of layer k - 2, whose readers passed the barrier below
        __syncthreads();
        if (own) {
            const int lm = (k - 1) % 3, l0 = k % 3, lp = (k + 1) % 3;
            // f[c+a+b] - f[c-a+b] + f[c-a-b] - f[c+a-b] for the pairs of axes
            auto Xxy = [&](int m) {
                const T *f = s[l0][m];
                return f[e + 1 + TX] - f[e - 1 + TX] + f[e - 1 - TX] - f[e + 1 - TX];
            };
            auto Xxz = [&](int m) {
                return s[lp][m][e + 1] - s[lp][m][e - 1] + s[lm][m][e - 1] - s[lm][m][e + 1];
            };
            auto Xyz = [&](int m) {
                return s[lp][m][e + TX] - s[lp][m][e - TX] + s[lm][m][e - TX] - s[lm][m][e + TX];
            };
            const T ctxxy = Xxy(1), ctxxz = Xxz(2);
            const T ctyxy = Xxy(0), ctyyz = Xyz(2);
            const T ctzxz = Xxz(0), ctzyz = Xyz(1);
            const long long c = cid(d, i, j, k);
            const T co = coef[COLC ? (long long)(k + d.mbc - 1) : c];
            u[c] = s[l0][0][e] + co * (dxy * ctxxy + dxz * ctxxz);
            u[d.P + c] = s[l0][1][e] + co * (dxy * ctyxy + dyz * ctyyz);
            u[2 * d.P + c] = s[l0][2][e] + co * (dxz * ctzxz + dyz * ctzyz);
        }
        __syncthreads();
    }
}
template <typename T, bool COLC, class G>
__global__ __launch_bounds__(256) void k_diff_cross(Dims d, T *u, const T *q, const T *coef, T dxy, T dxz, T dyz,
                                                    int kb, G gate)
{
    b_diff_cross<T, COLC>(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, u, q, coef, dxy, dxz, dyz, kb, gate);
}

// One component's x, y and z passes (diffuse.f:153-208 after the cross terms;
// conduct.f:262-323), fused, each with the reference's operand order and
// roundings:
//   x: X = U + fx*co*((U[i+1]-U)-U+U[i-1])   on the interior rows
//   y: Y = X + fy*co*((X[j+1]-X)-X+X[j-1])
//   z: q = Y + fz*co*((Y[k-1]-Y)-Y+Y[k+1])
// u holds the interior before the passes, gh the ghost layers, which the
// reference copies once and never refreshes between passes; except in
// conduct (COND), where conduct.f:86-91 fills the z ghosts before the z pass:
// for i in [1-mbc, mz+mbc], bounded by mz, not mx.  When mx > mz the columns
// i > mz+mbc keep their stale z ghosts.  When mz > mx an out-of-row i
// addresses the array linearly: within a layer the writes land on later rows
// with those rows' own values, and S = mz-mx of them cross into the next
// layer: at in-layer offsets r < S, layers 0 and 1 end up with layer 2's
// values, whose columns then see no z difference in layer 1 and layer 2's
// own value below layer 2; the ghost columns among them keep layer 2's
// ghosts in layer 1 for later substeps (late).  (Writes past the last
// layers change ghosts that nothing reads.)
// A workgroup covers 64 x-cells by 4 y-rows and kb layers: per layer it forms
// X on 6 rows (its rows and one on either side) in LDS, Y on its 4 rows, and
// keeps Y of three consecutive layers in registers for the z pass (the layer
// below its first is recomputed).
template <typename T, bool COLC, bool COND>
__device__ __forceinline__ void diff_passes(const uint3 BI, const Dims &d, T *out, const T *u, const T *gh, const T *coef, T fx,
                                            T fy, T fz, int kb, int S, bool late, T (&sx)[6][64])
{
    const int tx = (int)threadIdx.x, ty = (int)threadIdx.y;
    const int i = (int)BI.x * 64 + tx + 1;
    const int j0 = (int)BI.y * 4 + 1;
    const int j = j0 + ty;
    const int k0 = (int)BI.z * kb + 1;
    const int k1 = k0 + kb - 1 < d.mz ? k0 + kb - 1 : d.mz;
    const bool own = i <= d.mx && j <= d.my;
    const long long sy = d.NX, sz = (long long)d.NX * d.NY;
    auto co_at = [&](long long c, int k) { return coef[COLC ? (long long)(k + d.mbc - 1) : c]; };
    auto spilt = [&](int ii, int jj) { return COND && (jj + d.mbc - 1) * d.NX + (ii + d.mbc - 1) < S; };
    // ghost column (ii, jj) of layer kk at cell c
    auto ghost = [&](long long c, int ii, int jj, int kk) {
        return gh[COND && late && kk == 1 && spilt(ii, jj) ? c + sz : c];
    };
    // Y at (i, j, kk) for an interior layer kk; every lane of the block calls it
    auto yres = [&](int kk) {
        __syncthreads();   // the previous layer's readers of sx are done
        for (int r = ty; r < 6; r += 4) {
            const int jr = j0 - 1 + r;
            if (i <= d.mx && jr >= 1 && jr <= d.my) {
                const long long c = cid(d, i, jr, kk);
                const T aq = u[c];
                const T am = i > 1 ? u[c - 1] : ghost(c - 1, 0, jr, kk);
                const T ap = i < d.mx ? u[c + 1] : ghost(c + 1, d.mx + 1, jr, kk);
                const T qt = ap - aq - aq + am;
                sx[r][tx] = aq + fx * co_at(c, kk) * qt;
            }
        }
        __syncthreads();
        T y = T(0.0);
        if (own) {
            const long long c = cid(d, i, j, kk);
            const T aq = sx[ty + 1][tx];
            const T am = j > 1 ? sx[ty][tx] : ghost(c - sy, i, 0, kk);
            const T ap = j < d.my ? sx[ty + 2][tx] : ghost(c + sy, i, d.my + 1, kk);
            const T qt = ap - aq - aq + am;
            y = aq + fy * co_at(c, kk) * qt;
        }
        return y;
    };
    const long long cb = own ? cid(d, i, j, k0) : 0;
    const bool fill = COND && i <= d.mz + d.mbc;   // conduct refreshes this column's z ghosts
    const bool spill = spilt(i, j);
    T ym = k0 > 1 ? yres(k0 - 1) : (own ? gh[cb - sz] : T(0.0));
    T y0 = yres(k0);
    if (k0 == 1 && fill) ym = y0;
    for (int k = k0; k <= k1; k++) {
        const long long c = own ? cid(d, i, j, k) : 0;
        const T yp = k < d.mz ? yres(k + 1) : (fill ? y0 : own ? gh[c + sz] : T(0.0));
        if (COND && spill && k <= 2) {
            if (k == 1) y0 = yp;
            ym = y0;
        }
        if (own) {
            const T qt = ym - y0 - y0 + yp;
            out[c] = y0 + fz * co_at(c, k) * qt;
        }
        ym = y0;
        y0 = yp;
    }
}

// The diffusion passes of the three velocities and conduct's first substep
// in one launch (components 0-3 side by side in the grid's z), or with only4
// conduct's substep kk >= 2.  fac(3*cc + n): the factor of component cc along
// axis n, from wherever the caller keeps them (an indexed copy of them would
// live in scratch).  Launch: block (64, 4), grid (ceil(mx/64), ceil(my/4),
// ncomp * ceil(mz/kb)).
template <typename T, bool COLC, class G, class FAC>
__device__ __forceinline__ void b_diff(const uint3 BI, Dims d, const DiffArgs<T> &a, const FAC &fac, int kk, const G &gate)
{
    if (!gate.on()) return;
    __shared__ T sx[6][64];
    const int nz = (d.mz + a.kb - 1) / a.kb;
    const int cc = kk > 1 ? 3 : __builtin_amdgcn_readfirstlane((int)BI.z / nz);
    const uint3 bi = {BI.x, BI.y, kk > 1 ? BI.z : BI.z - cc * nz};
    const T fx = fac(3 * cc), fy = fac(3 * cc + 1), fz = fac(3 * cc + 2);
    if (cc < 3) {
        T *p = a.q + (cc + 1) * d.P;
        diff_passes<T, COLC, false>(bi, d, p, a.u + cc * d.P, p, a.nu, fx, fy, fz, a.kb, 0, false, sx);
    } else if (gate.conducts(kk)) {
        const T *q5 = a.q + 4 * d.P;
        const T *src = kk == 1 ? q5 : (kk & 1) ? a.qt : a.ut;
        diff_passes<T, COLC, true>(bi, d, (kk & 1) ? a.ut : a.qt, src, q5, a.kap, fx, fy, fz, a.kb, a.S, kk > 1, sx);
    }
}
template <typename T, bool COLC, class G>
__global__ __launch_bounds__(256) void k_diff(Dims d, DiffArgs<T> a, int kk, G gate)
{
    b_diff<T, COLC>(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, a, [&](int n) { return a.f[n]; }, kk, gate);
}

// interior copy of planes src -> dst (n planes with stride P)
template <typename T, class G>
__device__ __forceinline__ void b_copy_interior(const uint3 BI, Dims d, T *dst, const T *src, int nplanes, const G &gate)
{
    if (!gate.on()) return;
    INTERIOR_IJK
    for (int m = 0; m < nplanes; m++) dst[m * d.P + c] = src[m * d.P + c];
}
template <typename T, class G>
__global__ void k_copy_interior(Dims d, T *dst, const T *src, int nplanes, G gate)
{
    b_copy_interior(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, d, dst, src, nplanes, gate);
}

// plain copy of n elements (copyq3 and the working copies of the source pass)
template <typename T, class G>
__device__ __forceinline__ void b_copy(const uint3 BI, unsigned nblk, T *dst, const T *src, long long n, const G &gate)
{
    if (!gate.on()) return;
    for (long long e = (long long)BI.x * blockDim.x + threadIdx.x; e < n;
         e += (long long)nblk * blockDim.x)
        dst[e] = src[e];
}
template <typename T, class G>
__global__ void k_copy(T *dst, const T *src, long long n, G gate)
{
    b_copy(uint3{blockIdx.x, blockIdx.y, blockIdx.z}, gridDim.x, dst, src, n, gate);
}

}  // namespace magic
