// Per-interface solver math of the sweep kernels: Roe state, limiters,
// transverse splits and the 9-point increment accumulator, for a
// floating-point type T (double: the FP64 form; float: the FP32 perturbation
// form).  What the pencil kernel uses (cflsupbee, suppow, tsplit, Acc) performs
// exactly the reference's operations.  The tiled sweep's own (rcp1, quot,
// root_rcp, one_minus_pow, LimT, suppow1, WaveT) round otherwise, within the
// errors stated at each.
#pragma once
#include "magic_dev.h"

namespace magic {

template <typename T>
struct RoeT {
    T u, v, w, enth, a, g1a2, euv, u2v2w2;
    T i2a;   // 1 / (2 a): the wave-strength divisor of rpn3 and of every transverse split
};
using Roe = RoeT<double>;

// The well-balanced gravity jump (rpn3euX.f:194-208): across a hydrostatic
// column p_b - p_a - .5 (rho_a + rho_b) aux17 cancels to rounding, so a
// single fused multiply-add in it, or in the pressures it is made of, moves
// the jump by a unit of the pressure.  These pieces are rounded as the
// reference rounds them (no contraction) whatever the surrounding code's
// contraction setting.
template <typename T>
__device__ __forceinline__ T pressure_nc(T gam, T E, T m1, T m2, T m3, T irho)
{
#pragma clang fp contract(off)
    return (gam - T(1.0)) * (E - T(0.5) * (m1 * m1 + m2 * m2 + m3 * m3) * irho);
}
template <typename T>
__device__ __forceinline__ T flux_jump_nc(T mb, T ub, T pb, T ma, T ua, T pa)
{
#pragma clang fp contract(off)
    return (mb * ub + pb) - (ma * ua + pa);
}
template <typename T>
__device__ __forceinline__ T gravity_jump_nc(T d, T ra, T rb, T vg)
{
#pragma clang fp contract(off)
    return d - T(0.5) * (rb + ra) * vg;
}

// The FP32 form solves the normal Riemann problem in FP64 (the sweep's
// part 1): its jumps and wave strengths subtract background-sized products
// (enthalpy times velocity, enthalpy times the density jump), whose FP32
// rounding the flow carries up into the thin upper layers; in FP32 the
// form's temperature error there grew to 3e-4 of the field peak in 300
// steps, in FP64 to 3e-5-6e-5.  Its reciprocals and square roots are the
// hardware's FP64 approximations refined by one Newton step (relative error
// near 1e-14, far inside that form's error bar).  RF selects them (true: the
// FP32 form) over those of the FP64 form: one third-order step from the
// hardware's 2**-24 (largest error over 5e8 arguments 1.0 x 2**-53, the bound of
// a correctly rounded quotient, as two Newton steps have, in three operations
// for their four).  Quotients are corrected by their remainder (quot).
template <bool RF>
__device__ __forceinline__ double rcp1(double x)
{
    const double r = __builtin_amdgcn_rcp(x), e = fma(-x, r, 1.0);
    return fma(r, RF ? e : fma(e, e, e), r);
}
// num / den from an approximate reciprocal r of den: corrected by its
// remainder, as the correctly rounded quotient is, without that one's scaling.
// One rounding (a unit of 2**-53) whatever error r has up to 1e-14 or so.
__host__ __device__ __forceinline__ double quot(double num, double den, double r)
{
    const double q = num * r;
    return fma(fma(-den, q, num), r, q);
}
// g / b of the limiters: NaN where b is zero or its reciprocal overflows,
// which the limiters take (they then multiply b).
template <bool RF>
__device__ __forceinline__ double ratio(double g, double b)
{
    return quot(g, b, rcp1<RF>(b));
}
// 1/x of the limiters' clamped Courant numbers and 1 + r (normal range)
__device__ __forceinline__ double rcpL(double x) { return rcp1<false>(x); }
__device__ __forceinline__ float rcpL(float x) { return __builtin_amdgcn_rcpf(x); }
template <bool RF>
__device__ __forceinline__ double sqrt1(double x)
{
    if constexpr (RF) {
        // Goldschmidt step from the reciprocal square root; 0 and negative
        // (or NaN) arguments take the plain hardware square root
        const double y = __builtin_amdgcn_rsq(x);
        const double s0 = x * y, h = 0.5 * y;
        const double r = fma(-s0, h, 0.5);
        const double s1 = fma(s0, r, s0);
        return x > 0.0 ? s1 : __builtin_amdgcn_sqrt(x);
    } else {
        return sqrt(x);
    }
}

// Square root s and its reciprocal i of x > 0 together, from one hardware
// reciprocal square root and a Goldschmidt step (of first order for the FP32
// form; in FP64 of second, and a last residual step for the root: largest
// errors 1.0 x 2**-53 of the root and 2.0 x 2**-53 of the reciprocal, 1.0 and
// 2.6 with two first-order steps).
template <bool RF>
__device__ __forceinline__ void root_rcp(double x, double &s, double &i)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double r = fma(-g, h, 0.5);
    if constexpr (!RF) r = fma(1.5 * r, r, r);
    g = fma(g, r, g);
    h = fma(h, r, h);
    if constexpr (!RF) g = fma(fma(-g, g, x), h, g);
    s = g;
    i = h + h;
}

// flang's MIN/MAX: a < b ? a : b, a > b ? a : b
template <typename T>
__device__ __forceinline__ T fminF(T a, T b) { return a < b ? a : b; }
template <typename T>
__device__ __forceinline__ T fmaxF(T a, T b) { return a > b ? a : b; }

// MIN/MAX in one instruction, where neither operand is NaN in a state that
// goes on (the limiters' and splits' own)
__device__ __forceinline__ double fminT(double a, double b) { return __builtin_fmin(a, b); }
__device__ __forceinline__ double fmaxT(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ float fminT(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ float fmaxT(float a, float b) { return __builtin_fmaxf(a, b); }

// 1 - x**p for 0 <= x <= 1, p > 0 (suppow's 1 - rfrac**pp).  FP64: ln x from
// the odd series of ln((1+s)/(1-s)) with x = m 2**k, sqrt(1/2) <= m <
// sqrt(2), s = (m-1)/(m+1), and -expm1(p ln x) from the Taylor series of the
// exponential on [-ln 2 / 2, ln 2 / 2]; both series run until the next term is
// below 2**-54 of the sum, and ln x and p ln x keep their rounding errors.
// Largest error over 2e7 arguments: 0.74 units of 2**-53, as
// 1 - pow(x, p) has (0.75).  The limiter needs none of the
// library function's special cases.
__device__ __forceinline__ double one_minus_pow(double x, double p)
{
    const double xc = fmaxT(x, 1e-300);   // x = 0: the power is 0 either way
    // k from the high words of x and sqrt(1/2) (0x3fe6a09e): m in [0.70711, 1.41422)
    const int k = (__double2hiint(xc) - 0x3fe6a09e) >> 20;
    const double m = __hiloint2double(__double2hiint(xc) - (k << 20), __double2loint(xc));
    const double kd = (double)k;
    const double f = m - 1.0, g = m + 1.0, i = rcp1<false>(g);
    // (m-1)/(m+1) = s + sl (m - (g - 1): what rounding m + 1 left out)
    const double s = f * i, sl = fma(-s, m - (g - 1.0), fma(-s, g, f)) * i;
    const double z = s * s;
    double h = 1.0 / 21.0;
    h = fma(h, z, 1.0 / 19.0);
    h = fma(h, z, 1.0 / 17.0);
    h = fma(h, z, 1.0 / 15.0);
    h = fma(h, z, 1.0 / 13.0);
    h = fma(h, z, 1.0 / 11.0);
    h = fma(h, z, 1.0 / 9.0);
    h = fma(h, z, 1.0 / 7.0);
    h = fma(h, z, 1.0 / 5.0);
    h = fma(h, z, 1.0 / 3.0);
    // ln x = hi + lo; ln 2 in two parts, the first with 33 significant bits,
    // so that kd times it is exact
    const double s2 = s + s;
    const double ln2h = 0x1.62e42fefp-1, ln2l = 0x1.473de6af278edp-34;
    const double A = kd * ln2h, hi = A + s2;
    const double lo = fma(s2 * z, h, fma(kd, ln2l, (s2 - (hi - A)) + (sl + sl)));
    const double pc = fminT(p, 4000.0);
    const double L = fmaxT(pc * hi, -60.0), Ll = fma(pc, hi, -(pc * hi)) + pc * lo;   // the power is below 2**-53 beyond -60
    const double n = rint((L + Ll) * 1.4426950408889634);
    const double r = fma(-n, ln2h, L) + fma(-n, ln2l, Ll);
    double e = 1.0 / 6227020800.0;
    e = fma(e, r, 1.0 / 479001600.0);
    e = fma(e, r, 1.0 / 39916800.0);
    e = fma(e, r, 1.0 / 3628800.0);
    e = fma(e, r, 1.0 / 362880.0);
    e = fma(e, r, 1.0 / 40320.0);
    e = fma(e, r, 1.0 / 5040.0);
    e = fma(e, r, 1.0 / 720.0);
    e = fma(e, r, 1.0 / 120.0);
    e = fma(e, r, 1.0 / 24.0);
    e = fma(e, r, 1.0 / 6.0);
    e = fma(e, r, 0.5);
    const double em1 = fma(e, r * r, r);
    const double sc = __builtin_ldexp(1.0, (int)n);
    return fma(-sc, em1, 1.0 - sc);
}
// FP32 form: 2**(p log2 x) from the hardware's exp2 and log2 (log2 0 = -inf
// gives 0, as pow does)
__device__ __forceinline__ float one_minus_pow(float x, float p)
{
    return 1.0f - __builtin_amdgcn_exp2f(p * __builtin_amdgcn_logf(x));
}

// rpn3euX.f:686-705
__device__ __forceinline__ double cflsupbee(double theta, double beta, double r, double cfl, double cflup)
{
    const double cfle = fmaxF(0.001, fminF(0.999, cfl)), cflupe = fmaxF(0.001, fminF(0.999, cflup));
    // cfle is clamped to [0.001, 0.999]: its reciprocals are taken once
    const double i1mc = 1.0 / (1.0 - cfle), icfle = 1.0 / cfle;
    const double weight = (1.0 - cflupe) * i1mc;
    const double s1 = theta * weight * 2.0 * icfle;
    const double s2 = (1.0 + cfle) * (1.0 / 3.0);
    const double phimax = theta * 2.0 * i1mc;
    const double ultra = fmaxF(0.0, fminF(s1 * r, phimax));
    const double c1 = 1.0 + (s2 - beta / 2.0) * (r - 1.0);
    const double c2 = 1.0 + (s2 + beta / 2.0) * (r - 1.0);
    return fmaxF(0.0, fminF(ultra, fmaxF(c1, c2)));
}

// rpn3euX.f:709-731
__device__ __forceinline__ double suppow(double r, double cfl, double cflup)
{
    const double cfle = fmaxF(0.001, fminF(0.999, cfl)), cflupe = fmaxF(0.001, fminF(0.999, cflup));
    const double i1mc = 1.0 / (1.0 - cfle), icfle = 1.0 / cfle;
    const double s2 = (1.0 + cfle) * (1.0 / 3.0), s3 = 1.0 - s2;
    const double weight = (1.0 - cflupe) * i1mc;
    const double pp = (r <= 1.0) ? weight * (2.0 * icfle) * 2.0 * s3 : fabs(2.0 * i1mc) * 2.0 * s2;
    const double rabs = fabs(r);
    const double rfrac = fabs((1.0 - rabs) * (1.0 / (1.0 + rabs)));
    const double signum = fmaxF(0.0, copysign(1.0, r));
    return signum * (s3 + s2 * r) * (1.0 - pow(rfrac, pp));
}

// The limiters of one interface's waves that move at one speed: with the
// clamped Courant number e, the reciprocals of e and 1 - e are taken once.
template <typename T>
struct LimT {
    T e, i1mc, icfl;
    __device__ __forceinline__ explicit LimT(T cfl)
        : e(fmaxT(T(0.001), fminT(T(0.999), cfl))), i1mc(rcpL(T(1.0) - e)), icfl(rcpL(e)) {}
    // weight of the upwind interface's Courant number (rpn3euX.f:693)
    __device__ __forceinline__ T weight(T cflup) const
    {
        return (T(1.0) - fmaxT(T(0.001), fminT(T(0.999), cflup))) * i1mc;
    }
    // cflsupbee, rpn3euX.f:686-705
    __device__ __forceinline__ T bee(T theta, T beta, T r, T weight) const
    {
        const T s1 = theta * weight * T(2.0) * icfl;
        const T s2 = (T(1.0) + e) * (T(1.0) / T(3.0));
        const T ultra = fmaxT(T(0.0), fminT(s1 * r, theta * T(2.0) * i1mc));
        const T c1 = T(1.0) + (s2 - beta / T(2.0)) * (r - T(1.0));
        const T c2 = T(1.0) + (s2 + beta / T(2.0)) * (r - T(1.0));
        return fmaxT(T(0.0), fminT(ultra, fmaxT(c1, c2)));
    }
};

// suppow (rpn3euX.f:709-731) with the interface's own Courant number as the
// upwind one (its weight is then 1), so that each branch of the exponent
// needs one reciprocal; zero for a ratio that is not positive, NaN among them.
template <typename T>
__device__ __forceinline__ T suppow1(T r, T cfl)
{
    const T big = sizeof(T) == 4 ? T(1e30) : T(1e300);
    r = r > big ? big : r;   // a ratio beyond it: (1-r)/(1+r) is 1 to rounding and the limiter 0
    const T e = fmaxT(T(0.001), fminT(T(0.999), cfl));
    const T s2 = (T(1.0) + e) * (T(1.0) / T(3.0)), s3 = T(1.0) - s2;
    const bool lo = r <= T(1.0);
    const T pp = T(4.0) * (lo ? s3 : s2) * rcpL(lo ? e : T(1.0) - e);
    const T rfrac = fabs((T(1.0) - r) * rcpL(T(1.0) + r));
    const T y = (s3 + s2 * r) * one_minus_pow(rfrac, pp);
    return r > T(0.0) ? y : T(0.0);
}

// Transverse split of a flux difference by the Roe eigensystem of the
// interface: rpt3euX.f:106-214; QUIRK = rptt3's icoor = 3 coefficient
// (rptt3euX.f:169).  Local components: 0 rho, 1 normal momentum, 2/3 the
// transverse momenta (mv, mw of rpn3euX.f:109-121), 4 energy, 5.. tracers.
template <int NC, int ICOOR, bool QUIRK, typename T>
__device__ __forceinline__ void tsplit(const RoeT<T> &R, const T (&in)[NC], T (&bm)[NC], T (&bp)[NC])
{
    const T q1 = in[0], qu = in[1], qv = in[2], qw = in[3], q5 = in[4];
    const T a4 = R.g1a2 * (R.euv * q1 + R.u * qu + R.v * qv + R.w * qw - q5);
    T w1[5], w2[5], w3[5], sb1, sb2, sb3;
    if (ICOOR == 2) {
        const T a2 = qu - R.u * q1, a3 = qw - R.w * q1;
        const T a5 = (qv + (R.a - R.v) * q1 - R.a * a4) * R.i2a;
        const T a1 = q1 - a4 - a5;
        w1[0] = a1; w1[1] = a1 * R.u; w1[2] = a1 * (R.v - R.a); w1[3] = a1 * R.w;
        w1[4] = a1 * (R.enth - R.v * R.a); sb1 = R.v - R.a;
        w2[0] = a4; w2[1] = a2 + R.u * a4; w2[2] = R.v * a4; w2[3] = a3 + R.w * a4;
        w2[4] = a4 * T(0.5) * R.u2v2w2 + a2 * R.u + a3 * R.w; sb2 = R.v;
        w3[0] = a5; w3[1] = a5 * R.u; w3[2] = a5 * (R.v + R.a); w3[3] = a5 * R.w;
        w3[4] = a5 * (R.enth + R.v * R.a); sb3 = R.v + R.a;
    } else {
        const T a2 = (QUIRK ? qw : qu) - R.u * q1, a3 = qv - R.v * q1;
        const T a5 = (qw + (R.a - R.w) * q1 - R.a * a4) * R.i2a;
        const T a1 = q1 - a4 - a5;
        w1[0] = a1; w1[1] = a1 * R.u; w1[2] = a1 * R.v; w1[3] = a1 * (R.w - R.a);
        w1[4] = a1 * (R.enth - R.w * R.a); sb1 = R.w - R.a;
        w2[0] = a4; w2[1] = a2 + R.u * a4; w2[2] = a3 + R.v * a4; w2[3] = R.w * a4;
        w2[4] = a4 * T(0.5) * R.u2v2w2 + a2 * R.u + a3 * R.v; sb2 = R.w;
        w3[0] = a5; w3[1] = a5 * R.u; w3[2] = a5 * R.v; w3[3] = a5 * (R.w + R.a);
        w3[4] = a5 * (R.enth + R.w * R.a); sb3 = R.w + R.a;
    }
    const T m1 = fminF(sb1, T(0.0)), m2 = fminF(sb2, T(0.0)), m3 = fminF(sb3, T(0.0));
    const T p1 = fmaxF(sb1, T(0.0)), p2 = fmaxF(sb2, T(0.0)), p3 = fmaxF(sb3, T(0.0));
#pragma unroll
    for (int m = 0; m < 5; m++) {
        bm[m] = m1 * w1[m] + m2 * w2[m] + m3 * w3[m];
        bp[m] = p1 * w1[m] + p2 * w2[m] + p3 * w3[m];
    }
#pragma unroll
    for (int m = 5; m < NC; m++) {
        bm[m] = m2 * in[m];
        bp[m] = p2 * in[m];
    }
}

// A vector of the transverse splits in variables relative to the Roe
// velocity, scaled so that the splits need the fewest operations: entropy
// s = rho - p, pressure p (divided by a^2) and the momenta n, a, b along the
// normal and the two transverse directions, less rho times the Roe velocity.
// An acoustic wave of strength x along the normal is p = x, n = -+ a x; the
// contact wave is s; the shear waves are a and b.
template <typename T>
struct WaveT {
    T s, p, n, a, b;
    __device__ __forceinline__ WaveT() : s(0), p(0), n(0), a(0), b(0) {}
    __device__ __forceinline__ WaveT(T x1, T x4, T xa, T xb, T x5, T snd)
        : s(x4), p(x1 + x5), n(snd * (x5 - x1)), a(xa), b(xb) {}
    __device__ __forceinline__ void add(const WaveT &o) { s += o.s; p += o.p; n += o.n; a += o.a; b += o.b; }
    // k (x + c y)
    __device__ __forceinline__ static WaveT comb(T k, const WaveT &x, T c, const WaveT &y)
    {
        WaveT o;
        o.s = k * (x.s + c * y.s);
        o.p = k * (x.p + c * y.p);
        o.n = k * (x.n + c * y.n);
        o.a = k * (x.a + c * y.a);
        o.b = k * (x.b + c * y.b);
        return o;
    }
    // k e - (lo + hi): the middle one of three splits that sum to k e
    __device__ __forceinline__ static WaveT middle(const WaveT &lo, const WaveT &hi, T k, const WaveT &e)
    {
        WaveT o;
        o.s = k * e.s - (lo.s + hi.s);
        o.p = k * e.p - (lo.p + hi.p);
        o.n = k * e.n - (lo.n + hi.n);
        o.a = k * e.a - (lo.a + hi.a);
        o.b = k * e.b - (lo.b + hi.b);
        return o;
    }
};

// The three speeds of a transverse direction (half of u - c and u + c: a
// split halves the acoustic parts) and the splits with the weights
// -min(speed, 0), -|speed| and max(speed, 0) (R = 0, 1, 2).
template <typename T>
struct SpeedT {
    T h1, h2, h3;
    __device__ __forceinline__ SpeedT(T v, T snd) : h1(T(0.5) * (v - snd)), h2(v), h3(T(0.5) * (v + snd)) {}
    template <int R>
    __device__ __forceinline__ static T weight(T x)
    {
        return R == 0 ? -fminT(x, T(0.0)) : R == 1 ? -fabs(x) : fmaxT(x, T(0.0));
    }
    __device__ __forceinline__ T w2(int r) const { return r == 0 ? weight<0>(h2) : r == 1 ? weight<1>(h2) : weight<2>(h2); }
    // (normal, other, split) momenta of x -> split along this direction
    template <int R>
    __device__ __forceinline__ void split(const WaveT<T> &x, T along, T snd, T isnd, T &p, T &al, T &s) const
    {
        const T y1 = weight<R>(h1) * (x.p - along * isnd), y3 = weight<R>(h3) * (x.p + along * isnd);
        p = y1 + y3;
        al = snd * (y3 - y1);
        s = weight<R>(h2) * x.s;
    }
    template <int R>
    __device__ __forceinline__ WaveT<T> split_a(const WaveT<T> &x, T snd, T isnd) const
    {
        WaveT<T> o;
        split<R>(x, x.a, snd, isnd, o.p, o.a, o.s);
        o.n = weight<R>(h2) * x.n;
        o.b = weight<R>(h2) * x.b;
        return o;
    }
    template <int R>
    __device__ __forceinline__ WaveT<T> split_b(const WaveT<T> &x, T snd, T isnd) const
    {
        WaveT<T> o;
        split<R>(x, x.b, snd, isnd, o.p, o.b, o.s);
        o.n = weight<R>(h2) * x.n;
        o.a = weight<R>(h2) * x.a;
        return o;
    }
};

// Accumulators D[da+1][db+1][m] of the increments a cell receives, for the
// target cell offset (da, db) in the (g, h) plane (step3.f:189-226).
template <int NC, typename T = double>
struct Acc {
    T D[3][3][NC];
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int x = 0; x < 3; x++)
#pragma unroll
            for (int y = 0; y < 3; y++)
#pragma unroll
                for (int m = 0; m < NC; m++) D[x][y][m] = T(0.0);
    }
    // gadd(side, off) += c*v  folded with factor fg: side 1 -> da = -1,
    // side 2 -> da = +1, each also entering the own column with the
    // opposite sign (flux difference).
    __device__ __forceinline__ void g(int side, int off, T c, const T (&v)[NC])
    {
#pragma unroll
        for (int m = 0; m < NC; m++) {
            const T x = c * v[m];
            if (side == 1) { D[0][off + 1][m] -= x; D[1][off + 1][m] += x; }
            else           { D[2][off + 1][m] += x; D[1][off + 1][m] -= x; }
        }
    }
    __device__ __forceinline__ void h(int side, int off, T c, const T (&v)[NC])
    {
#pragma unroll
        for (int m = 0; m < NC; m++) {
            const T x = c * v[m];
            if (side == 1) { D[off + 1][0][m] -= x; D[off + 1][1][m] += x; }
            else           { D[off + 1][2][m] += x; D[off + 1][1][m] -= x; }
        }
    }
    __device__ __forceinline__ void c11(int m, T x) { D[1][1][m] += x; }
};

template <int NC, typename T>
__device__ __forceinline__ void axpy3(T (&out)[NC], const T (&a)[NC], T c, const T (&b)[NC])
{
#pragma unroll
    for (int m = 0; m < NC; m++) out[m] = a[m] + c * b[m];
}

template <int NC>
__device__ __forceinline__ void scatter(const SweepArgs &A, long long base, const Acc<NC> &acc)
{
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int y = 0; y < 3; y++) {
            const long long off = base + (long long)(x - 1) * A.sA + (long long)(y - 1) * A.sB;
#pragma unroll
            for (int m = 0; m < NC; m++) {
                double *p = A.qnew + (long long)A.comp[m] * A.P + off;
                *p = *p + acc.D[x][y][m];
            }
        }
}


}  // namespace magic
