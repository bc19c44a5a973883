// Tiled directional sweep of the MAGIC unsplit f-wave step, for a float
// type T and two state forms:
//   T = double, PERT = false: q is the conserved state (the FP64 form);
//   T = float,  PERT = true : q is the perturbation q - q_bar from a
//     background column at rest (the FP32 form); the f-wave jumps are formed
//     from perturbation pressures, so the hydrostatic balance cancels
//     analytically, and the Courant number is reduced in FP64.
// This header holds the kernel; sweep_tile.hip and sweep_tile32.hip
// instantiate it under their own floating-point contraction settings.
//
// Same per-interface algebra as sweep.hip (rpn3euX.f, rpt3euX.f, rptt3euX.f,
// flux3fw.f, step3.f); different data movement:
//   * a workgroup takes one block of pencils and interfaces: TA pencils that
//     are neighbours along the tile axis "a" (x-sweep: a = y; y- and z-sweeps:
//     a = x, so that tile-axis-major lanes read rows of x) by CH interfaces
//     along the pencils (chunks overlap by 2: the limiter's upwind
//     neighbours), and marches over a segment of L planes along the other
//     transverse axis b; TA, CH and the lane order form the tile shape;
//   * the 3x3 increments of each interface (its cells i-1 and i into the
//     pencil and its 8 transverse neighbours, step3.f:189-226) are summed in a
//     ring of three planes in LDS, LT[plane][component][position], in
//     sub-steps (one per phase and a offset, so no two lanes add to the same
//     entry at once; separated by the wave's program order or by barriers,
//     see the sub-step loop).  A plane is complete once the planes on both
//     sides have been swept; it is then written, contiguous and once, to the
//     block's own part of the increment buffer (SweepParts);
//   * the parts of all blocks of the three directions are added to q
//     afterwards (parts.h), each cell's in a fixed order: no two workgroups
//     write the same memory, so the blocks need no colouring, no atomics and
//     no order, and one launch covers the whole step.
// The result is deterministic.  Against the earlier tile, which marched along
// the pencils and added each chunk's three planes to q with FP64 atomics in
// six colour launches per direction, q moves once instead of three times per
// direction.
#pragma once
#include "magic_dev.h"
#include "magic_solver.h"

namespace magic {

// Tile shapes: TA pencils x CH interfaces per chunk (TA*CH = 256 lanes),
// lanes either tile-axis-major (consecutive lanes on neighbouring pencils)
// or pencil-major (consecutive lanes along one pencil).  The host picks one
// per sweep direction (a fixed table or the autotuner); every shape computes
// the same increments, only the grouping of their sums differs.
template <int SH>
struct TileShape;
template <>
struct TileShape<0> { static constexpr int TA = 16; static constexpr bool PM = false; };
template <>
struct TileShape<1> { static constexpr int TA = 8; static constexpr bool PM = false; };
template <>
struct TileShape<2> { static constexpr int TA = 8; static constexpr bool PM = true; };
template <>
struct TileShape<3> { static constexpr int TA = 4; static constexpr bool PM = true; };
static_assert(TileShape<TILE_NSHAPE - 1>::TA > 0, "one TileShape per shape index");

// Pointer into global memory.  The kernel reads its state pointers
// from an argument block in memory, where the compiler cannot tell their
// address space and would use flat loads and stores; flat accesses count on
// the LDS counter too, so every LDS wait would also wait for them.
template <typename T>
using gptr = __attribute__((address_space(1))) T *;
template <typename T>
__device__ __forceinline__ gptr<T> to_global(T *p) { return (gptr<T>)p; }

// A value that nothing depends on: what an idle lane holds where the others
// have computed one (a zero there would cost a move per value and plane).
template <typename X>
__device__ __forceinline__ X idle_value()
{
    X x;
    asm volatile("" : "=v"(x));
    return x;
}

template <typename AT>
__device__ __forceinline__ void report_t(const AT &A, int code, int i, int pg, int ph)
{
    if (atomicCAS(A.status, 0, code) == 0) {
        int fi, fj, fk;
        if (A.sweep == 1) { fi = i; fj = pg; fk = ph; }
        else if (A.sweep == 2) { fi = ph; fj = i; fk = pg; }
        else { fi = pg; fj = ph; fk = i; }
        A.status[1] = A.sweep; A.status[2] = fi; A.status[3] = fj; A.status[4] = fk;
    }
}

// x += v in LDS.  FP64: the hardware's add, which reads nothing back (13
// cycles per wave; the sweeps of 250 x 200 x 300 5.3 -> 4.6 ms).  FP32 adds in
// registers: ds_add_f32 takes 190 cycles per wave.
__device__ __forceinline__ void lds_add(double &x, double v)
{
    __hip_atomic_fetch_add(&x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_add(float &x, float v) { x += v; }

// One block (tile bt along the tile axis, chunk bk along the pencils, segment
// bs along b) of direction A; called by every lane of a 256-lane workgroup.
template <typename T, bool PERT, int NTR, int SH>
__device__ __forceinline__ void tile_sweep_body(const SweepArgsT<T> &A, int bt, int bk, int bs)
{
    constexpr int NC = 5 + NTR;
    constexpr int NT = 256, TA = TileShape<SH>::TA, CH = NT / TA;
    constexpr bool PM = TileShape<SH>::PM;
    constexpr int NCELL = CH - 1;               // cells S .. S+CH-2 of a chunk
    constexpr int TROW = TA + 2;                // a offsets A0-1 .. A0+TA
    constexpr int NPOS = TROW * NCELL;          // positions of a plane
    constexpr T beta = T(0.666666666666666);
    static_assert(TA * CH == NT && TA == tile_ta(SH) && NPOS == part_npos(SH), "tile is 256 lanes");

    // What the limiters read of the neighbouring interfaces: the jumps (FP64 in
    // both forms) and the tracer waves.  With four tracers or more in FP64 they
    // lie in the ring's third plane, which takes increments only afterwards
    // (and is cleared in between), so that two workgroups fit a compute unit.
    constexpr bool OVERLAY = sizeof(T) == 8 && NTR >= 4;
    constexpr int NSV = OVERLAY ? 1 : NT;
    __shared__ double s_delv[5 * NSV];
    __shared__ T s_trwv[(NTR > 0 ? NTR : 1) * NSV];
    __shared__ T s_s2[NT];
    __shared__ T s_cfo[NT];
    __shared__ int s_flag[NT];
    __shared__ T s_cprev[TA];
    __shared__ int s_found[TA];
    __shared__ int s_need;
    __shared__ T LT[3 * NC * NPOS];
    static_assert(!OVERLAY || (5 + NTR) * NT <= NC * NPOS, "the jumps and tracer waves fit a plane");

    const int t0 = threadIdx.x;
    int t = t0;
    int pa = PM ? (t / CH) : (t % TA);    // pencil within the tile
    int c = PM ? (t % CH) : (t / TA);     // interface offset within the chunk
    const int nb = PM ? 1 : TA;                 // lane distance between neighbouring interfaces
    const int n = A.n, a_is_g = A.a_is_g;
    const int A0 = bt * TA, B0 = bs << A.lgL;
    const int nplane = min(1 << A.lgL, A.nB + 2 - B0);   // planes B0 .. B0 + nplane - 1
    int a = A0 + pa;                            // tile-axis coordinate of this lane's pencil
    bool pen = a <= A.nA + 1;
    const T dtdn = T(A.dtdn);
    const T d = dtdn;
    const T ca = T(a_is_g ? A.fg : A.fh), cb2 = T(a_is_g ? A.fh : A.fg);   // dt/da, dt/db
    const gptr<const T> qold = to_global(A.qold);
    const gptr<const double> gam = to_global(A.gam), vgrav = to_global(A.vgrav);
    const gptr<const double> crho = to_global(A.crho), cE = to_global(A.cE), cgam = to_global(A.cgam),
                             cvg = to_global(A.cvg), cres = to_global(A.cres);

    // position within a plane: fastest along x, as the part's (the x-sweep's
    // odd row length also keeps lanes on neighbouring pencils in different banks)
    const int pA = A.sweep == 1 ? NCELL : 1, pN = A.sweep == 1 ? 1 : TROW;
    auto pix = [&](int ai, int ci) { return ai * pA + ci * pN; };
    for (int e = t; e < 3 * NC * NPOS; e += NT) LT[e] = T(0.0);
    if (t < TA) s_cprev[t] = T(0.0);
    if (t == 0) s_need = 0;
    __syncthreads();
    double cflmax = 0.0;            // Courant number, reduced in FP64

    // cell I-1 of interface I on plane b; the states of a lane's interface
    long long cell0 = (long long)(a + A.mbc - 1) * A.sA + (long long)(c - 1 + A.mbc - 1) * A.sN;
    T pqa[NC], pqb[NC], pga = T(0.0), pgb = T(0.0), pvg = T(0.0);
    auto fetch = [&](int Iq, int b) {
        if (pen && Iq <= n + 2) {
            const long long x = cell0 + (long long)(Iq - c) * A.sN + (long long)(b + A.mbc - 1) * A.sB;
            const long long y = x + A.sN;
#pragma unroll
            for (int m = 0; m < NC; m++) {
                pqa[m] = (qold + A.cofs[m])[x];
                pqb[m] = (qold + A.cofs[m])[y];
            }
            if constexpr (!PERT) {
                pga = gam[x];
                pgb = gam[y];
                if (A.gravity) pvg = vgrav[y];
            }
        }
    };
    // The next plane's states are loaded ahead: in the FP32 form while the
    // current plane's transverse terms are computed, which hides the latency
    // whole; in FP64, where they would not fit beside part 3, while the plane
    // that is complete is flushed.
    constexpr bool EARLY = sizeof(T) == 4;
    int I0 = bk * (CH - 2) + c;
    // In FP64 the registers are full: what a lane can form again from its
    // index is formed again for every flush and, with two tracers or more, for
    // every plane (the asm hides that it is the same each time), or the compiler
    // keeps it all through the loop and spills, and each reload from scratch
    // then waits for the flush's stores as well (28.4k -> 21.7k cycles per wave
    // and plane with the hardware's LDS adds).
    constexpr bool RELOAD = sizeof(T) == 8;

    // one plane of the ring to the block's part, as it lies in LDS: whole
    // contiguous lines, nothing read back
    gptr<T> part = to_global(A.parts) + (long long)(bs * A.sS + bk * A.sK + bt * A.sT) * (((1 << A.lgL) + 2) * NC * NPOS);
    auto flush = [&](int p, int slot) {
        int tf = t;
        if constexpr (RELOAD) asm volatile("" : "+v"(tf));
        T *src = LT + slot * (NC * NPOS);
        const gptr<T> dst = part + p * (NC * NPOS);
        // all read before the first is written: one wait
        constexpr int NF = NC * NPOS / NT, REM = NC * NPOS % NT;
        T v[NF + 1], zero = T(0.0);
        if constexpr (RELOAD) asm volatile("" : "+v"(zero));
#pragma unroll
        for (int k = 0; k < NF; k++) v[k] = src[tf + k * NT];
        if (REM && tf < REM) v[NF] = src[tf + NF * NT];
#pragma unroll
        for (int k = 0; k < NF; k++) {
            dst[tf + k * NT] = v[k];
            if constexpr (!OVERLAY) src[tf + k * NT] = zero;
        }
        if (REM && tf < REM) {
            dst[tf + NF * NT] = v[NF];
            if constexpr (!OVERLAY) src[tf + NF * NT] = zero;
        }
    };
    fetch(I0, B0);

    for (int plane = 0; plane < nplane; plane++) {
        if constexpr (RELOAD && NTR >= 2) {
            t = t0;
            asm volatile("" : "+v"(t));
            pa = PM ? (t / CH) : (t % TA);
            c = PM ? (t % CH) : (t / TA);
            a = A0 + pa;
            pen = a <= A.nA + 1;
            cell0 = (long long)(a + A.mbc - 1) * A.sA + (long long)(c - 1 + A.mbc - 1) * A.sN;
            I0 = bk * (CH - 2) + c;
        }
        const int b = B0 + plane;               // other transverse coordinate
        const int pg = a_is_g ? a : b, ph = a_is_g ? b : a;   // (g, h) coordinates
        // the ring's planes of b-1, b and b+1
        const int r0 = plane % 3, r1 = r0 == 2 ? 0 : r0 + 1, r2 = r1 == 2 ? 0 : r1 + 1;
        double *const s_del = OVERLAY ? (double *)(LT + r2 * (NC * NPOS)) : s_delv;   // [5][NT]
        T *const s_trw = OVERLAY ? LT + r2 * (NC * NPOS) + 5 * NT : s_trwv;           // [NTR][NT]
        // No barrier here without the overlay: the previous plane's last
        // readers of the s_* arrays (part 2) are behind its phase barriers, and
        // its flush's accesses of the ring are behind this plane's barrier
        // after part 1.  With it, the flush has to have read the plane.
        if (OVERLAY && plane > 0) __syncthreads();
        int kk = bk;                            // chunk being solved (an earlier one while looking for CFLup)
        int looked = 0;
        asm volatile("" : "+s"(looked));        // one copy of the solve in the loop below
        RoeT<double> R;
        double b1, b2, b3, b4, b5, al1, al5, s1, s2, s3;
        bool lf, act1, act2;
        T trw[NTR > 0 ? NTR : 1];   // unlimited tracer waves
        T c1, c2, c3;
        int I;
        for (;;) {
        I = kk * (CH - 2) + c;                  // Fortran interface index
        act1 = pen && I <= n + 2;
        act2 = act1 && c >= 1 && c <= CH - 2 && I >= 1 && I <= n + 1;
        if (looked) fetch(I, b);

        // ---------------- part 1: Roe solve of interface I (rpn3euX.f:138-421)
        // The waves stay in their strengths (b1, b5 acoustic, b4 entropy, b2
        // and b3 shear; W: the same as the solve's FP64 values); the f-wave
        // vectors of rpn3euX.f:217-271 are never formed.  al1, al5 and lf:
        // the left-going parts of waves 1, 3 and 2 (rpn3euX.f:311-399).
        // The solve runs in FP64 in both forms (see rcp1 in magic_solver.h).
        for (double *v : {&R.u, &R.v, &R.w, &R.enth, &R.a, &R.u2v2w2, &R.g1a2, &R.euv, &R.i2a, &b1, &b2, &b3, &b4, &b5,
                          &al1, &al5, &s1, &s2, &s3})
            *v = idle_value<double>();
        c1 = idle_value<T>(); c2 = idle_value<T>(); c3 = idle_value<T>();
        lf = false;
#pragma unroll
        for (int k = 0; k < NTR; k++) trw[k] = idle_value<T>();
        if (act1) {
            constexpr bool RF = sizeof(T) == 4;
            double qa[NC], qb[NC], vgc = 0.0;
            double ga, gb;
#pragma unroll
            for (int m = 0; m < NC; m++) {
                qa[m] = pqa[m];
                qb[m] = pqb[m];
            }
            ga = pga;
            gb = pgb;
            vgc = pvg;
            // perturbation form: q holds q - background; the background is a
            // column at rest (rho_bar(k), E_bar(k), gamma(k)), so the full
            // states differ from q only in rho and E
            double rpa = 0, rpb = 0, ppa = 0, ppb = 0;
            int kib = 0;
            if constexpr (PERT) {
                const int ka = A.sweep == 3 ? I - 1 : b, kb = A.sweep == 3 ? I : b;
                const int kia = ka + A.mbc - 1;
                kib = kb + A.mbc - 1;
                ga = cgam[kia];
                gb = cgam[kib];
                rpa = qa[0];
                rpb = qb[0];
                const double epa = qa[4], epb = qb[4];
                qa[0] = crho[kia] + rpa;
                qb[0] = crho[kib] + rpb;
                qa[4] = cE[kia] + epa;
                qb[4] = cE[kib] + epb;
                ppa = epa;
                ppb = epb;
            }
            if (!(qa[0] > 0.0) || !(qb[0] > 0.0)) report_t(A, 1, I, pg, ph);
            // square root, its reciprocal and the reciprocal of both densities
            double rhsqrtl, il, iqa, rhsqrtr, ir, iqb;
            root_rcp<RF>(qa[0], rhsqrtl, il);
            root_rcp<RF>(qb[0], rhsqrtr, ir);
            iqa = rcp1<RF>(qa[0]);
            iqb = rcp1<RF>(qb[0]);
            const double i2 = rcp1<RF>(rhsqrtl + rhsqrtr);
            const double gamma = (rhsqrtr * gb + rhsqrtl * ga) * i2;
            const double gamma1 = gamma - 1.0;
            if constexpr (PERT) {
                // p - p_bar = (gamma-1) (E' - kinetic energy), p_bar = (gamma-1) E_bar
                ppa = (ga - 1.0) * (ppa - 0.5 * quot(qa[1] * qa[1] + qa[2] * qa[2] + qa[3] * qa[3], qa[0], iqa));
                ppb = (gb - 1.0) * (ppb - 0.5 * quot(qb[1] * qb[1] + qb[2] * qb[2] + qb[3] * qb[3], qb[0], iqb));
            }
            const double pl = pressure_nc(ga, qa[4], qa[1], qa[2], qa[3], iqa);
            const double pr = pressure_nc(gb, qb[4], qb[1], qb[2], qb[3], iqb);
            R.u = (qa[1] * il + qb[1] * ir) * i2;
            R.v = (qa[2] * il + qb[2] * ir) * i2;
            R.w = (qa[3] * il + qb[3] * ir) * i2;
            R.enth = ((qa[4] + pl) * il + (qb[4] + pr) * ir) * i2;
            R.u2v2w2 = R.u * R.u + R.v * R.v + R.w * R.w;
            const double a2 = gamma1 * (R.enth - 0.5 * R.u2v2w2);
            if (!(a2 > 0.0)) report_t(A, 2, I, pg, ph);
            double ia;
            root_rcp<RF>(a2, R.a, ia);
            R.i2a = 0.5 * ia;
            R.g1a2 = quot(gamma1, a2, ia * ia);
            R.euv = R.enth - R.u2v2w2;
            const double ur = qb[1] * iqb, ul = qa[1] * iqa;
            const double d1 = qb[1] - qa[1];
            double d2;
            if constexpr (PERT) d2 = (qb[1] * ur + ppb) - (qa[1] * ul + ppa);   // background part below
            else d2 = flux_jump_nc(qb[1], ur, pr, qa[1], ul, pl);
            const double d3 = ur * qb[2] - ul * qa[2];
            const double d4 = ur * qb[3] - ul * qa[3];
            double d5 = (qb[4] + pr) * ur - (qa[4] + pl) * ul;
            if (A.gravity) {
                if constexpr (PERT) {
                    // the background's own jump p_bar_b - p_bar_a - .5 (rho_bar_a +
                    // rho_bar_b) aux17 is the column residual (zero to FP64 rounding)
                    const double vg = cvg[kib];
                    d2 = d2 - 0.5 * (rpb + rpa) * vg + cres[kib];
                    d5 = d5 - 0.5 * (qb[1] + qa[1]) * vg;
                } else {
                    d2 = gravity_jump_nc(d2, qa[0], qb[0], vgc);
                    d5 = d5 - 0.5 * (qb[1] + qa[1]) * vgc;
                }
            }
            b4 = R.g1a2 * (R.euv * d1 + R.u * d2 + R.v * d3 + R.w * d4 - d5);
            b2 = d3 - R.v * d1;
            b3 = d4 - R.w * d1;
            b5 = (d2 + (R.a - R.u) * d1 - R.a * b4) * R.i2a;
            b1 = d1 - b4 - b5;
            s1 = R.u - R.a;
            s2 = R.u;
            s3 = R.u + R.a;
#pragma unroll
            for (int k = 0; k < NTR; k++)
                trw[k] = (T)((k + 1 <= A.nspecadv) ? s2 * (qb[5 + k] - qa[5 + k]) : ur * qb[5 + k] - ul * qa[5 + k]);
            // Entropy fix (rpn3euX.f:316-398).  The signs of the speeds it
            // compares, u -+ c of a state with c**2 = gamma p/rho, are taken
            // from u**2 against c**2 with the intermediate states scaled by
            // the wave speed, without their square roots and reciprocals;
            // those are formed only in a transonic wave.
            {
                const double cca = ga * pl * qa[0];   // (rho c)**2
                const bool super = pl >= 0.0 && qa[1] >= 0.0 && qa[1] * qa[1] >= cca && s1 > 0.0;
                // state behind wave 1, times s1
                const double r1 = qa[0] * s1 + b1, m1 = qa[1] * s1 + b1 * s1;
                const double m2 = qa[2] * s1 + b1 * R.v, m3 = qa[3] * s1 + b1 * R.w;
                const double e1 = qa[4] * s1 + b1 * (R.enth - R.u * R.a);
                const double cc1 = ga * (ga - 1.0) * (e1 * r1 - 0.5 * (m1 * m1 + m2 * m2 + m3 * m3));
                al1 = s1 < 0.0 ? b1 : 0.0;
                if (m1 * s1 > 0.0 && m1 * m1 > cc1 && !(qa[1] >= 0.0 && qa[1] * qa[1] >= cca)) {
                    const double s0 = ul - sqrt1<RF>(ga * pl * iqa);
                    const double sa = m1 / r1 - sqrt1<RF>(cc1) / fabs(r1);
                    if (s0 < 0.0 && sa > 0.0) al1 = s0 * (sa - s1) / (sa - s0) / s1 * b1;
                }
                if (super) al1 = 0.0;
                lf = s2 < 0.0 && !super;
                al5 = 0.0;
                if (lf) {
                    const double ccb = gb * pr * qb[0];
                    // state ahead of wave 3, times s3
                    const double r2 = qb[0] * s3 - b5, n1 = qb[1] * s3 - b5 * s3;
                    const double n2 = qb[2] * s3 - b5 * R.v, n3 = qb[3] * s3 - b5 * R.w;
                    const double e2 = qb[4] * s3 - b5 * (R.enth + R.u * R.a);
                    const double cc2 = gb * (gb - 1.0) * (e2 * r2 - 0.5 * (n1 * n1 + n2 * n2 + n3 * n3));
                    al5 = s3 < 0.0 ? b5 : 0.0;
                    if (n1 * s3 < 0.0 && n1 * n1 > cc2 && !(qb[1] <= 0.0 && qb[1] * qb[1] >= ccb)) {
                        const double sr = ur + sqrt1<RF>(gb * pr * iqb);
                        const double sb = n1 / r2 + sqrt1<RF>(cc2) / fabs(r2);
                        if (sb < 0.0 && sr > 0.0) al5 = sb * (sr - s3) / (sr - sb) / s3 * b5;
                    }
                }
            }
            c1 = fabs((T)s1 * dtdn); c2 = fabs((T)s2 * dtdn); c3 = fabs((T)s3 * dtdn);
            s_del[t] = d1; s_del[NT + t] = d2; s_del[2 * NT + t] = d3; s_del[3 * NT + t] = d4; s_del[4 * NT + t] = d5;
            s_s2[t] = (T)s2;
#pragma unroll
            for (int k = 0; k < NTR; k++) s_trw[k * NT + t] = trw[k];
            // the limiters need the Courant number an earlier interface left
            if (act2 && b1 == 0.0 && b2 == 0.0 && (b3 != 0.0 || b4 != 0.0)) s_need = 1;
        }
        __syncthreads();
        // CFLup (rpn3euX.f:563-619) is the Courant number last assigned along
        // the pencil.  It is needed from an earlier interface only where waves
        // 1 and 2 vanish exactly and wave 3 or 4 does not (pure shear or
        // contact): then every interface says what it assigned; and the
        // earlier chunks are solved again, from the nearest back, until every
        // pencil of the tile has met an assignment, and this chunk once more.
        // A block that marched along the pencil would carry the value for
        // nothing; here a sheared sheet across 250 x 200 x 300 cells (FP64, 4
        // interfaces) costs 10 % of the three sweeps (3.25 -> 3.57 ms), shear at
        // every interface of the x-sweep without any assignment, the worst case,
        // 7.5 ms.
        if (s_need == 0) break;
        s_flag[t] = (act1 && c <= CH - 2 && I >= 1 && I <= n + 1 && (b1 != 0.0 || b2 != 0.0 || b5 != 0.0)) ? 1 : 0;
        s_cfo[t] = b5 != 0.0 ? c3 : (b2 != 0.0 ? c2 : c1);
        __syncthreads();
        if (bk == 0 || (looked && kk == bk)) break;
        if (!looked) {
            looked = 1;
            if (t < TA) { s_cprev[t] = T(0.0); s_found[t] = 0; }
        } else if (t < TA && !s_found[t]) {
            for (int j = CH - 2; j >= 0; j--) {
                const int tt = PM ? t * CH + j : j * TA + t;
                if (s_flag[tt]) { s_cprev[t] = s_cfo[tt]; s_found[t] = 1; break; }
            }
        }
        kk = __syncthreads_and(t >= TA || (kk < bk && s_found[t])) ? -1 : kk - 1;
        if (kk < 0) kk = bk;
        }

        // ---------------- part 2: limiters (rpn3euX.f:434-676) and the strengths
        // of the second-order correction (flux3fw.f:270-284).  From here on the
        // transverse directions are the tile axis a and the marching axis b.
        const T un = (T)R.u, ua = (T)R.v, ub = (T)R.w, snd = (T)R.a, isnd = (T)(2.0 * R.i2a);
        const T kin = (T)(0.5 * R.u2v2w2), hk = (T)(R.enth - 0.5 * R.u2v2w2);   // |u|^2/2 and H - |u|^2/2
        const T x1 = (T)b1, x4 = (T)b4, xa = (T)b2, xb = (T)b3, x5 = (T)b5;     // strengths
        T l1 = (T)al1, l5 = (T)al5;                                            // left-going acoustic parts
        T q1 = idle_value<T>(), q4 = idle_value<T>(), qsa = idle_value<T>(), qsb = idle_value<T>(),
          q5 = idle_value<T>();   // strengths of cqxx
        T trq[NTR > 0 ? NTR : 1];
        T nrm[2][5];   // FP32 form: the cell's own normal update
#pragma unroll
        for (int k = 0; k < NTR; k++) trq[k] = idle_value<T>();
        if constexpr (PERT) {
#pragma unroll
            for (int m = 0; m < 10; m++) nrm[m / 5][m % 5] = idle_value<T>();
        }
        if (act2) {
            const T ts1 = (T)s1, ts2 = (T)s2, ts3 = (T)s3;
            // sign(s) / 2 * (1 - |s| dt/dn)
            const T k1 = copysign(T(0.5), ts1) * (T(1.0) - c1), k2 = copysign(T(0.5), ts2) * (T(1.0) - c2),
                    k3 = copysign(T(0.5), ts3) * (T(1.0) - c3);
            const int up1 = signbit(s1) ? t + nb : t - nb, up2 = signbit(s2) ? t + nb : t - nb,
                      up3 = signbit(s3) ? t + nb : t - nb;
            const LimT<T> lim2(c2);
#pragma unroll
            for (int k = 0; k < NTR; k++) {
                const T fc = trw[k];
                T wl = T(0.0);
                if (fc != T(0.0)) {
                    const T r = s_trw[k * NT + (s2 > 0.0 ? t - nb : t + nb)] / fc;
                    if (k + 1 <= A.nspecadv) wl = lim2.bee(T(0.5), beta, r, lim2.weight(fabs(s_s2[up2] * dtdn)));
                    else wl = fmaxF(T(0.0), fminF(T(1.0), r));
                }
                trq[k] = k2 * (wl * fc);
            }
            // the upwind interfaces' strengths in this interface's waves: those
            // of wave 2 come from one of the two acoustic waves' sides
            auto b4of = [&](int e) {
                return R.g1a2 * (R.euv * s_del[e] + R.u * s_del[NT + e] + R.v * s_del[2 * NT + e] + R.w * s_del[3 * NT + e] -
                                 s_del[4 * NT + e]);
            };
            auto b5of = [&](int e, double b4e) {
                return (s_del[NT + e] + (R.a - R.u) * s_del[e] - R.a * b4e) * R.i2a;
            };
            const double b4l = b4of(up1), b4r = b4of(up3);
            const double g1 = s_del[up1] - b4l - b5of(up1, b4l), g5 = b5of(up3, b4r), g4 = up2 == up1 ? b4l : b4r;
            const double g2 = s_del[2 * NT + up2] - R.v * s_del[up2], g3 = s_del[3 * NT + up2] - R.w * s_del[up2];
            T wt = T(1.0);   // the upwind Courant number's weight: 1 where it is c2 itself
            if (b2 == 0.0 && (b3 != 0.0 || b4 != 0.0)) {
                T cflup;
                if (b1 != 0.0) cflup = c1;
                else {
                    cflup = s_cprev[pa];
                    for (int j = c - 1; j >= 0; j--)
                        if (s_flag[t - (c - j) * nb]) { cflup = s_cfo[t - (c - j) * nb]; break; }
                }
                wt = lim2.weight(cflup);
            }
            // Whether a shear strength vanishes is asked of the strength itself;
            // the reference asks what is left of it in the wave's momentum,
            // (b2 + v b4) - v b4, which rounding can make zero or not.
            // A vanishing wave needs no case of its own: the limiters are
            // finite for any ratio, NaN among them, and multiply a strength
            // of zero.
            constexpr bool RF = sizeof(T) == 4;
            const T wl1 = suppow1((T)ratio<RF>(g1, b1), c1), wl5 = suppow1((T)ratio<RF>(g5, b5), c3);
            const T wl2 = lim2.bee(T(1.0), beta, (T)ratio<RF>(g2, b2), T(1.0)), wl3 = lim2.bee(T(1.0), beta, (T)ratio<RF>(g3, b3), wt),
                    wl4 = lim2.bee(T(1.0), beta, (T)ratio<RF>(g4, b4), wt);
            // strengths of cqxx, in FP64 up to here
            const double w1 = (double)(k1 * wl1) * b1, w2 = (double)(k2 * wl2) * b2, w3 = (double)(k2 * wl3) * b3,
                         w4 = (double)(k2 * wl4) * b4, w5 = (double)(k3 * wl5) * b5;
            if constexpr (PERT) {
                // The FP32 form forms the cell's own normal update in FP64 with
                // the unrounded dt/dn and rounds it once: the second-order
                // correction nearly cancels the fluctuation in smooth flow, and
                // rounding the two products apart (with dt/dn in FP32) grew,
                // over some 300 steps, into an error of T' of 1e-4 of its peak
                // in the thin upper layers of weak plumes.
#pragma unroll
                for (int ph2 = 0; ph2 < 2; ph2++) {
                    const double dD = -A.dtdn, sg = ph2 == 0 ? 1.0 : -1.0;
                    const bool has = (ph2 == 0) == lf;
                    const double n1 = dD * ((ph2 == 0 ? al1 : b1 - al1) + sg * w1);
                    const double n5 = dD * ((ph2 == 0 ? al5 : b5 - al5) + sg * w5);
                    const double n4 = dD * ((has ? b4 : 0.0) + sg * w4);
                    const double nv = dD * ((has ? b2 : 0.0) + sg * w2), nw = dD * ((has ? b3 : 0.0) + sg * w3);
                    const double pp = n1 + n5, nn = R.a * (n5 - n1), rho = pp + n4, kk = 0.5 * R.u2v2w2;
                    const double mv = R.v * rho + nv, mw = R.w * rho + nw;
                    nrm[ph2][0] = (T)rho;
                    nrm[ph2][1] = (T)(R.u * rho + nn);
                    nrm[ph2][2] = (T)mv;
                    nrm[ph2][3] = (T)mw;
                    nrm[ph2][4] = (T)((R.enth - kk) * pp + kk * rho + R.u * nn + R.v * nv + R.w * nw);
                }
                cflmax = fmaxF(cflmax, fmaxF(fabs((double)ts1), fabs((double)ts3)) * A.dtdn);   // |u| is between them
            } else {
                cflmax = fmaxF(cflmax, fmaxF(c1, c3));
            }
            q1 = (T)w1; q4 = (T)w4; q5 = (T)w5;
            qsa = (T)w2;
            qsb = (T)w3;
        }
        if constexpr (OVERLAY) {
            // clear the third plane: a lane its own pencil's entries (and the
            // tile's edge entries) of the cell that phase 0 adds to, so that
            // with tile-axis-major lanes the wave's order is enough
            __syncthreads();
            T *cl = LT + r2 * (NC * NPOS);
            if (c >= 1) {
#pragma unroll
                for (int m = 0; m < NC; m++) cl[m * NPOS + pix(pa, c - 1)] = T(0.0);
                if (pa < 2)
#pragma unroll
                    for (int m = 0; m < NC; m++) cl[m * NPOS + pix(pa + TA, c - 1)] = T(0.0);
            }
            if constexpr (PM) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        if (EARLY && plane + 1 < nplane) fetch(I0, b + 1);

        // ---------------- part 3: transverse terms (flux3fw.f:297-625), two phases
        // The transverse splits by the interface's Roe eigensystem
        // (rpt3euX.f:106-214, rptt3euX.f:108-214) run in variables relative to
        // the Roe velocity (WaveT: entropy s, pressure p/a^2, momenta n, a, b),
        // in which a split is a few products and nested splits need no change
        // of variables.  A split along a with weights w (of the speeds u_a - c,
        // u_a, u_a + c) is S_a[w].  With w_j = -min(speed, 0), -|speed|,
        // max(speed, 0) for the target offsets j = -1, 0, +1, the reference's
        // 9-point increments of one interface (step3.f:189-226) are
        //   D[r][j] = S_a[w_r] y_j + S_b[w_j] z_r,
        //   y_j = S_b[w_j] F - (d c_a / 2) E [j = 0],
        //   z_r = S_a[w_r] F - (d c_b / 2) E [r = 0],
        // E = asdq +- 2 cqxx, F = -(d c_a c_b / 6)(asdq +- 3 cqxx), plus the
        // cell's own normal update in the centre.  Each D is carried to the
        // conserved components once, when it is added to the tile, in three
        // sub-steps (one per a offset, so no two lanes add to one entry at
        // once): deterministic.  Against splitting conserved vectors and
        // summing a 3 x 3 x NC register accumulator this halves the sweep's
        // arithmetic, and nothing wider than the y and z vectors stays live.
        const T kf = -(T(1.0) / T(6.0)) * d * ca * cb2, kea = -T(0.5) * d * ca, keb = -T(0.5) * d * cb2;
        const SpeedT<T> va(ua, snd), vb(ub, snd);
        T hm = lf ? T(1.0) : T(0.0);   // 1 where the contact waves belong to the phase
#pragma unroll 1
        for (int phase = 0; phase < 2; phase++) {
            // phase 0 (L): interface I -> cell I-1; phase 1 (R): -> cell I
            const bool on = act2 && (phase == 0 ? I >= 2 : I <= n);
            const int ci = phase == 0 ? c - 1 : c;  // cell index within the chunk's tile
            if (phase == 1 && t == 0) s_need = 0;   // every lane has read it (phase 0's barrier)
            const T sg = phase == 0 ? T(1.0) : -T(1.0);
            // One branch around the whole phase (pencil-major lanes all come
            // along for its barriers): split into several, each branch's results
            // live on as merged values and spill.  With it every tracer
            // count runs two waves per SIMD in FP64 and three in FP32: 128 x 100
            // x 150 with five tracers 1.74 -> 1.27 ms per step, with three
            // 1.59 -> 1.09; FP32 181 x 160 x 243 2.06 -> 1.74.
            if (PM || on) {
            WaveT<T> y[3] = {}, z[3] = {}, N = {};
            if (!PM || on) {
                const T s3q = T(3.0) * sg, s2q = T(2.0) * sg;
                const WaveT<T> X(l1, hm * x4, hm * xa, hm * xb, l5, snd), Q(q1, q4, qsa, qsb, q5, snd);
                const WaveT<T> F = WaveT<T>::comb(kf, X, s3q, Q), E = WaveT<T>::comb(T(1.0), X, s2q, Q);
                if constexpr (!PERT) N = WaveT<T>::comb(-d, X, sg, Q);
                y[0] = vb.template split_b<0>(F, snd, isnd);
                y[2] = vb.template split_b<2>(F, snd, isnd);
                z[0] = va.template split_a<0>(F, snd, isnd);
                z[2] = va.template split_a<2>(F, snd, isnd);
                // rptt3euX.f:169: the split along h takes its first shear
                // from the h momentum
                if (a_is_g) {
#pragma unroll
                    for (int r = 0; r < 3; r += 2) z[r].n = z[r].b + (ub - un) * (z[r].s + z[r].p);
                } else {
#pragma unroll
                    for (int r = 0; r < 3; r += 2) y[r].n = y[r].a + (ua - un) * (y[r].s + y[r].p);
                }
                y[1] = WaveT<T>::middle(y[0], y[2], kea, E);
                z[1] = WaveT<T>::middle(z[0], z[2], keb, E);
            }
            // One tracer goes with the five components' targets, more come after
            // them, one after the other: all at once they would hold 7 values
            // each.
            constexpr bool APART = NTR >= 2;
            struct Tracer {
                T y[3], z[3], n;
            };
            auto tracer = [&](int k) __attribute__((always_inline)) {
                Tracer w;
                const T at = hm * trw[k];
                const T ft = kf * (at + T(3.0) * sg * trq[k]), et = at + T(2.0) * sg * trq[k];
                w.n = -d * (at + sg * trq[k]);
#pragma unroll
                for (int r = 0; r < 3; r += 2) {
                    w.y[r] = vb.w2(r) * ft;
                    w.z[r] = va.w2(r) * ft;
                }
                w.y[1] = kea * et - (w.y[0] + w.y[2]);
                w.z[1] = keb * et - (w.z[0] + w.z[2]);
                return w;
            };
            auto tracer_add = [&](T *row, int k, const Tracer &w, int r, int j) __attribute__((always_inline)) {
                T v = va.w2(r) * w.y[j] + vb.w2(j) * w.z[r];
                if (r == 1 && j == 1) v += w.n;
                lds_add(row[(5 + k) * NPOS], v);
            };
            Tracer trs[!APART && NTR > 0 ? NTR : 1];
            if constexpr (!APART) {
#pragma unroll
                for (int k = 0; k < NTR; k++)
                    if (!PM || on) trs[k] = tracer(k);
            }
            // one sub-step per offset along a: lanes then add to distinct T entries
            auto substep = [&](auto rc) {
                constexpr int r = decltype(rc)::value;
                if (!PM || on) {
                    auto target = [&](auto jc) {
                        constexpr int j = decltype(jc)::value;
                        T *row = LT + (j == 0 ? r0 : j == 1 ? r1 : r2) * (NC * NPOS) + pix(pa + r, ci);
                        WaveT<T> D = va.template split_a<r>(y[j], snd, isnd);
                        D.add(vb.template split_b<j>(z[r], snd, isnd));
                        if constexpr (!PERT && r == 1 && j == 1) D.add(N);
                        const T rho = D.s + D.p;
                        T o[5] = {rho, un * rho + D.n, ua * rho + D.a, ub * rho + D.b,
                                  hk * D.p + kin * rho + un * D.n + ua * D.a + ub * D.b};
                        if constexpr (PERT && r == 1 && j == 1) {
#pragma unroll
                            for (int m = 0; m < 5; m++) o[m] += phase == 0 ? nrm[0][m] : nrm[1][m];
                        }
#pragma unroll
                        for (int m = 0; m < 5; m++) lds_add(row[m * NPOS], o[m]);
                        if constexpr (!APART) {
#pragma unroll
                            for (int k = 0; k < NTR; k++) tracer_add(row, k, trs[k], r, j);
                        }
                    };
                    target(IConst<0>{});
                    target(IConst<1>{});
                    target(IConst<2>{});
                }
                // With tile-axis-major lanes a wave holds every pencil of
                // its chunk cells, so the entries one phase's sub-steps add
                // to are the wave's own (cells c-1 or c of its lanes): only
                // the wave's program order separates its sub-steps (the
                // fence keeps the compiler from moving one sub-step's tile
                // reads above the previous one's writes; it emits nothing),
                // and the workgroup waits once per phase.  Pencil-major
                // waves share entries: a barrier after every sub-step.
                if constexpr (PM) __syncthreads();
                else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            };
            substep(IConst<0>{});
            substep(IConst<1>{});
            substep(IConst<2>{});
            if constexpr (APART) {
#pragma unroll
                for (int k = 0; k < NTR; k++) {
                    Tracer w = {};
                    if (!PM || on) w = tracer(k);
#pragma unroll
                    for (int r = 0; r < 3; r++) {
                        if (!PM || on) {
#pragma unroll
                            for (int j = 0; j < 3; j++)
                                tracer_add(LT + (j == 0 ? r0 : j == 1 ? r1 : r2) * (NC * NPOS) + pix(pa + r, ci), k, w, r, j);
                        }
                        if constexpr (PM) __syncthreads();
                        else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    }
                }
            }
            }
            if constexpr (!PM) __syncthreads();
            l1 = x1 - l1;   // phase 1: the right-going parts
            l5 = x5 - l5;
            hm = T(1.0) - hm;
        }

        // ---------------- flush: plane b-1 has all its increments
        if (!EARLY && plane + 1 < nplane) fetch(I0, b + 1);
        flush(plane, r0);
    }
    flush(nplane, nplane % 3);
    flush(nplane + 1, (nplane + 1) % 3);
    for (int o = 32; o > 0; o >>= 1) cflmax = fmaxF(cflmax, __shfl_xor(cflmax, o, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(A.cfl_bits, (unsigned long long)__double_as_longlong(cflmax));
}


// Waves per SIMD the register allocation aims at
template <typename T, int NTR, int SH>
constexpr int tile_waves()
{
    return sizeof(T) == 8 ? 2 : 3;
}

// The sweep kernel, for one grid and for a batch of grids alike (one
// compiled body with one call site, so both round alike): workgroup g takes
// block items[g] = {argument block, tile, chunk, segment}; blocks of grids
// whose control flag (*run) is 0 in this attempt end at once.
template <typename T, bool PERT, int NTR, int SH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(tile_waves<T, NTR, SH>())))
void tile_sweep(const SweepArgsT<T> *__restrict__ args, const int4 *__restrict__ items,
                const int *const *__restrict__ run)
{
    // the item is the same for the whole workgroup: scalar, so that the
    // argument block is read with scalar loads
    const int4 w = items[blockIdx.x];
    const int ai = __builtin_amdgcn_readfirstlane(w.x);
    if (*run[ai] == 0) return;
    tile_sweep_body<T, PERT, NTR, SH>(args[ai], __builtin_amdgcn_readfirstlane(w.y),
                                      __builtin_amdgcn_readfirstlane(w.z), __builtin_amdgcn_readfirstlane(w.w));
}

}  // namespace magic
