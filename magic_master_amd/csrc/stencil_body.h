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

// Every kernel below takes a gate G: GridGate (factors as passed) for one
// grid; the batched driver passes a gate that reads its scenario's
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
        k = (int)l * CLAMP_LAYERS + 1;
        const long long sz = (long long)d.NX * d.NY;
        for (int m = 5; m < nc; m++) {
            T *p = q + (long long)m * d.P + cid(d, i, j, k), v[CLAMP_LAYERS];
#pragma unroll
            for (int n = 0; n < CLAMP_LAYERS; n++)
                if (k + n <= d.mz) v[n] = p[n * sz];
#pragma unroll
            for (int n = 0; n < CLAMP_LAYERS; n++) {
                const T cl = fmaxD(T(0.0), fminD(v[n], T(1.0)));
                if (k + n <= d.mz && !(cl == v[n])) p[n * sz] = cl;   // only read where in its range already
            }
        }
        return;
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
        if (cl) v = fmaxD(T(0.0), fminD(v, T(1.0)));
        if (def || edge || cl) q[(long long)m * d.P + cg] = v;
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
// A wave covers 64 x-cells by DIFF_ROWS y-rows and marches over kb layers,
// every lane holding its column of rows in registers: per layer it forms X on
// its rows and one on either side, Y on its rows, and keeps Y of three
// consecutive layers for the z pass (the layers around its first and last are
// formed twice).  The next layer's values are loaded before the current one's
// are used; nothing is shared between lanes, so no wave waits for another.
// Bound by memory.  Against rows in LDS with two barriers per layer: 250 x 200
// x 300 FP64 558 -> 412 us, FP32 batch of 8 grids of 200 x 200 x 300 1.60 ->
// 0.78 ms (4 reads, 4 writes of 384 MB: 3.9 TB/s).
template <typename T, bool COLC, bool COND>
__device__ __forceinline__ void diff_passes(const uint3 BI, const Dims &d, T *out, const T *u, const T *gh, const T *coef, T fx,
                                            T fy, T fz, int kb, int S, bool late)
{
    constexpr int R = DIFF_ROWS;
    const int tx = (int)threadIdx.x, ty = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int il = (int)BI.x * 64 + tx + 1, i = il < d.mx ? il : d.mx;   // lanes past the end repeat the last column
    const int j0 = ((int)BI.y * 4 + ty) * R + 1;
    const int k0 = (int)BI.z * kb + 1;
    const int k1 = k0 + kb - 1 < d.mz ? k0 + kb - 1 : d.mz;
    if (j0 > d.my || k0 > d.mz) return;
    const long long sz = (long long)d.NX * d.NY;
    auto co_at = [&](long long c, int k) { return coef[COLC ? (long long)(k + d.mbc - 1) : c]; };
    auto spilt = [&](int ii, int jj) { return COND && (jj + d.mbc - 1) * d.NX + (ii + d.mbc - 1) < S; };
    // ghost column (ii, jj) of layer kk at cell c
    auto ghost = [&](long long c, int ii, int jj, int kk) {
        return gh[COND && late && kk == 1 && spilt(ii, jj) ? c + sz : c];
    };
    const bool first = i == 1, last = i == d.mx;
    // rows j0-1 .. j0+R of the layer loaded last: the cell and its x neighbours
    constexpr int NCO = COLC ? 1 : R + 2;
    T wa[R + 2], wm[R + 2], wp[R + 2], wc[NCO];
#pragma unroll
    for (int r = 0; r < R + 2; r++) wa[r] = wm[r] = wp[r] = T(0.0);
#pragma unroll
    for (int r = 0; r < NCO; r++) wc[r] = T(0.0);
    auto load = [&](int kk) __attribute__((always_inline)) {
        if (COLC) wc[0] = co_at(0, kk);
#pragma unroll
        for (int r = 0; r < R + 2; r++) {
            const int j = j0 - 1 + r;
            const long long c = cid(d, i, j, kk);
            T a = T(0.0), m = T(0.0), p = T(0.0), cc = T(0.0);
            if (j >= 1 && j <= d.my) {
                a = u[c];
                m = first ? ghost(c - 1, 0, j, kk) : u[c - 1];
                p = last ? ghost(c + 1, d.mx + 1, j, kk) : u[c + 1];
                if (!COLC) cc = co_at(c, kk);
            } else if (j <= d.my + 1) {
                a = ghost(c, i, j, kk);
            }
            wa[r] = a;
            wm[r] = m;
            wp[r] = p;
            if (!COLC) wc[COLC ? 0 : r] = cc;
        }
    };
    // X, then Y of the loaded layer, whose coefficients go to co; layer kn is
    // loaded (0: none) once X is formed
    auto yres = [&](T (&y)[R], T (&co)[COLC ? 1 : R], int kn) __attribute__((always_inline)) {
        T x[R + 2];
#pragma unroll
        for (int r = 0; r < R + 2; r++) {
            const int j = j0 - 1 + r;
            x[r] = wa[r];
            if (j >= 1 && j <= d.my) {
                const T qt = wp[r] - wa[r] - wa[r] + wm[r];
                x[r] = wa[r] + fx * wc[COLC ? 0 : r] * qt;
            }
        }
#pragma unroll
        for (int r = 0; r < (COLC ? 1 : R); r++) co[r] = wc[COLC ? 0 : r + 1];
        if (kn > 0) load(kn);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const T qt = x[r + 2] - x[r + 1] - x[r + 1] + x[r];
            y[r] = x[r + 1] + fy * co[COLC ? 0 : r] * qt;
        }
    };
    const bool fill = COND && i <= d.mz + d.mbc;   // conduct refreshes this column's z ghosts
    T ym[R], y0[R], yp[R], co0[COLC ? 1 : R], con[COLC ? 1 : R];
    const int kl = k1 < d.mz ? k1 + 1 : d.mz;   // last layer formed
    if (k0 > 1) {
        load(k0 - 1);
        yres(ym, co0, k0);
    } else {
        load(k0);
    }
    yres(y0, co0, k0 < kl ? k0 + 1 : 0);
    if (k0 == 1) {
#pragma unroll
        for (int r = 0; r < R; r++) ym[r] = fill || j0 + r > d.my ? y0[r] : gh[cid(d, i, j0 + r, 0)];
    }
    for (int k = k0; k <= k1; k++) {
        if (k < d.mz) yres(yp, con, k + 2 <= kl ? k + 2 : 0);
        else
#pragma unroll
            for (int r = 0; r < R; r++) yp[r] = fill || j0 + r > d.my ? y0[r] : gh[cid(d, i, j0 + r, d.mz + 1)];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int j = j0 + r;
            if (COND && k <= 2 && spilt(i, j)) {
                if (k == 1) y0[r] = yp[r];
                ym[r] = y0[r];
            }
            const T qt = ym[r] - y0[r] - y0[r] + yp[r];
            if (il <= d.mx && j <= d.my) out[cid(d, i, j, k)] = y0[r] + fz * co0[COLC ? 0 : r] * qt;
            ym[r] = y0[r];
            y0[r] = yp[r];
        }
#pragma unroll
        for (int r = 0; r < (COLC ? 1 : R); r++) co0[r] = con[r];
    }
}

// The diffusion passes of the three velocities and conduct's first substep
// in one launch (components 0-3 side by side in the grid's z), or with only4
// conduct's substep kk >= 2.  fac(3*cc + n): the factor of component cc along
// axis n, from wherever the caller keeps them (an indexed copy of them would
// live in scratch).  Launch: block (64, 4), grid (ceil(mx/64), ceil(my /
// (4 DIFF_ROWS)), ncomp * ceil(mz/kb)).
template <typename T, bool COLC, class G, class FAC>
__device__ __forceinline__ void b_diff(const uint3 BI, Dims d, const DiffArgs<T> &a, const FAC &fac, int kk, const G &gate)
{
    if (!gate.on()) return;
    const int nz = (d.mz + a.kb - 1) / a.kb;
    const int cc = kk > 1 ? 3 : __builtin_amdgcn_readfirstlane((int)BI.z / nz);
    const uint3 bi = {BI.x, BI.y, kk > 1 ? BI.z : BI.z - cc * nz};
    const T fx = fac(3 * cc), fy = fac(3 * cc + 1), fz = fac(3 * cc + 2);
    if (cc < 3) {
        T *p = a.q + (cc + 1) * d.P;
        diff_passes<T, COLC, false>(bi, d, p, a.u + cc * d.P, p, a.nu, fx, fy, fz, a.kb, 0, false);
    } else if (gate.conducts(kk)) {
        const T *q5 = a.q + 4 * d.P;
        const T *src = kk == 1 ? q5 : (kk & 1) ? a.qt : a.ut;
        diff_passes<T, COLC, true>(bi, d, (kk & 1) ? a.ut : a.qt, src, q5, a.kap, fx, fy, fz, a.kb, a.S, kk > 1);
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

}  // namespace magic
