// bx_math.h -- device arithmetic of the hydro step, written to reproduce the
// reference's FP64 evaluation order exactly.  Build with -ffp-contract=off and
// without fast-math: every +, *, / and sqrt below is one IEEE-754 operation.
#pragma once

#include <hip/hip_runtime.h>

#ifndef BX_THETA
#define BX_THETA 1.25  // generalized-minmod theta: Makefile:20 -DSLOPE_THETA=1.25
#endif

namespace bx {

// Division and square root per arithmetic type: IEEE correctly rounded for
// double (the reference's arithmetic); for float (the mixed-precision
// reconstruction only) the hardware reciprocal and square root, ~1-2 ulp.
template <typename T>
struct Arith;
template <>
struct Arith<double> {
    static __device__ __forceinline__ double div(double a, double b) { return a / b; }
    static __device__ __forceinline__ double root(double x) { return sqrt(x); }
    static __device__ __forceinline__ double fmin(double a, double b) { return __builtin_fmin(a, b); }
    static __device__ __forceinline__ double fmax(double a, double b) { return __builtin_fmax(a, b); }
    static __device__ __forceinline__ double fabs(double a) { return __builtin_fabs(a); }
    static __device__ __forceinline__ double copysign(double a, double b) { return __builtin_copysign(a, b); }
};
template <>
struct Arith<float> {
    static __device__ __forceinline__ float div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
    static __device__ __forceinline__ float root(float x) { return __builtin_amdgcn_sqrtf(x); }
    static __device__ __forceinline__ float fmin(float a, float b) { return __builtin_fminf(a, b); }
    static __device__ __forceinline__ float fmax(float a, float b) { return __builtin_fmaxf(a, b); }
    static __device__ __forceinline__ float fabs(float a) { return __builtin_fabsf(a); }
    static __device__ __forceinline__ float copysign(float a, float b) { return __builtin_copysignf(a, b); }
};

template <typename T>
__device__ __forceinline__ T vmax(T a, T b) { return a > b ? a : b; }
template <typename T>
__device__ __forceinline__ T vmin(T a, T b) { return a < b ? a : b; }

// vmax(x, c) for a floor c >= +0: x > c ? x : c and the hardware maximum
// give the same value for every x (a NaN x gives c either way; a zero x of
// either sign is not above c, and for c = +0 both give +0), so the single
// instruction is used.
template <typename T>
__device__ __forceinline__ T floor_at(T x, T c) { return Arith<T>::fmax(x, c); }

// FP64 square roots as the compiler lowers sqrt() (correctly rounded): for
// x below 2^-767 it scales x by 2^256 and the root by 2^-128, and it answers
// x itself for +-0 and +inf; otherwise the lowering is
//     y = rsq(x); s0 = x*y; h0 = 0.5*y; r = fma(-h0, s0, 0.5)
//     h1 = fma(h0, r, h0); s1 = fma(s0, r, s0)
//     s2 = fma(fma(-s1, s1, x), h1, s1); root = fma(fma(-s2, s2, x), h1, s2)
// which is taken here for x in [2^-767, inf); a lane with another x (zero,
// negative, infinite, NaN or tiny) takes sqrt() for all N.
template <int N>
__device__ __forceinline__ void sqrt_n(const double *x, double *r)
{
    bool ok = true;
    for (int i = 0; i < N; i++) {
        const double v = x[i];
        const double y = __builtin_amdgcn_rsq(v);
        const double s0 = v * y, h0 = y * 0.5;
        const double rr = __builtin_fma(-h0, s0, 0.5);
        const double h1 = __builtin_fma(h0, rr, h0), s1 = __builtin_fma(s0, rr, s0);
        const double s2 = __builtin_fma(__builtin_fma(-s1, s1, v), h1, s1);
        r[i] = __builtin_fma(__builtin_fma(-s2, s2, v), h1, s2);
        ok = ok && v >= 0x1p-767 && v < __builtin_huge_val();
    }
    if (__builtin_expect(!ok, 0))
        for (int i = 0; i < N; i++) r[i] = __builtin_sqrt(x[i]);
}

// utils.f90:696-707
template <typename T>
__device__ __forceinline__ T genminmod(T x1, T x2, T x3)
{
    if ((x1 > T(0)) && ((x2 > T(0)) && (x3 > T(0)))) {
        T tmp = vmin(x2, x3);
        return vmin(x1, tmp);
    } else if ((x1 < T(0)) && ((x2 < T(0)) && (x3 < T(0)))) {
        T tmp = vmax(x2, x3);
        return vmax(x1, tmp);
    }
    return T(0);
}

// utils.f90:738-741: slope(c0,c1,c2) = genminmod(tt*(c1-c0), half*(c2-c0), tt*(c2-c1))
template <typename T>
__device__ __forceinline__ T slope(T c0, T c1, T c2)
{
    const T tt = T(BX_THETA);
    return genminmod(tt * (c1 - c0), T(0.5) * (c2 - c0), tt * (c2 - c1));
}

// genminmod for finite (non-NaN) inputs with three min/max instructions:
// "all three > 0" is exactly "their minimum > 0" and "all three < 0" is
// "their maximum < 0"; min/max of same-signed nonzero values is exact.  For
// finite data the result equals genminmod() above bit for bit.
template <typename T>
__device__ __forceinline__ T genminmod_finite(T x1, T x2, T x3)
{
    const T mn = Arith<T>::fmin(x1, Arith<T>::fmin(x2, x3));
    const T mx = Arith<T>::fmax(x1, Arith<T>::fmax(x2, x3));
    return mn > T(0) ? mn : (mx < T(0) ? mx : T(0));
}

template <typename T>
__device__ __forceinline__ T slope_finite(T c0, T c1, T c2)
{
    const T tt = T(BX_THETA);
    return genminmod_finite(tt * (c1 - c0), T(0.5) * (c2 - c0), tt * (c2 - c1));
}

// Twice slope_finite, up to the sign of a zero result.  With a = c1-c0 and b =
// c2-c1 of one sign, t is the smaller in magnitude, c2-c0 has that sign too
// (subtraction is monotonic), and the limiter picks min(tt|t|, |c2-c0|/2);
// otherwise t is a zero.  tt*min(a,b) is min(tt*a,tt*b) because rounding is
// monotonic, and the doubling is exact (the same product of real numbers goes
// into q + c*s; below 2^-1021 a slope may differ in a denormal's last place).
// For use where the slope only enters q + c*s with a canonical (never -0) q,
// which gives the same value for a zero slope of either sign.  11 operations
// where the three arguments with their minimum and maximum take 13.
template <typename T>
__device__ __forceinline__ T slope2_fz(T c0, T c1, T c2)
{
    const T a = c1 - c0, b = c2 - c1;
    const T t = Arith<T>::fmax(Arith<T>::fmin(a, b), T(0)) + Arith<T>::fmin(Arith<T>::fmax(a, b), T(0));
    const T m = Arith<T>::fmin(Arith<T>::fabs(T(2 * BX_THETA) * t), Arith<T>::fabs(c2 - c0));
    return Arith<T>::copysign(m, t);
}

// Primitive variables of one cell as the flux routine sees them.
template <typename T>
struct Prim {
    T d, u[3], p, e;  // rho, velocity, pressure, internal energy (eps)
};

// One directional interface state (flux.f90:336-351): rho, velocity, p, eps, gamma.
template <typename T>
struct Side {
    T d, v[3], p, e, g;
    T s1, s2;  // flux_ang: r- and angular momentum; elsewhere unused
};

// flux.f90:299-308 interface_muscl
template <typename T>
__device__ __forceinline__ void muscl(T q, T lm, T lp, T s, T &minus, T &plus)
{
    minus = q + T(0.5) * (T(-1) - lm) * s;
    plus = q + T(0.5) * (T(1) - lp) * s;
}

// Correctly rounded quotients a[i]/b (i < N) that share one reciprocal, for
// FP64.  The hardware's IEEE division is v_div_scale (numerator and
// denominator), v_rcp, two Newton steps on the reciprocal, the quotient and
// its residual, v_div_fmas and v_div_fixup.  When b lies in [2^-300, 2^300]
// and each a is zero or lies in [2^-299, 2^302] in magnitude, v_div_scale
// leaves both operands as they are (exponent difference below 768, no
// denormal reciprocal or quotient, numerator exponent far above 53), VCC is
// clear and v_div_fixup returns its input for a nonzero quotient, so that
// sequence is
//     y0 = rcp(b); y1 = fma(y0, fma(-b, y0, 1), y0); y = fma(y1, fma(-b, y1, 1), y1)
//     q0 = a*y;    r = fma(-b, q0, a);              q = fma(r, y, q0)
// and y does not depend on a.  Here the residual is formed negated,
// r' = fma(b, q0, -a), and q = fma(-r', y, q0): for a nonzero the same bits
// (round-to-nearest is symmetric), and for a zero the signed zero that
// v_div_fixup gives (q0 = +-0, r' = +0, q = -0*y + q0 = q0).  A lane with an
// operand outside the range takes the plain division for all N.
template <int N>
__device__ __forceinline__ void div_shared(const double *a, double b, double *q)
{
    const double y0 = __builtin_amdgcn_rcp(b);
    const double y1 = __builtin_fma(y0, __builtin_fma(-b, y0, 1.0), y0);
    const double y = __builtin_fma(y1, __builtin_fma(-b, y1, 1.0), y1);
    double mag = 0.0;
    int emin = 0;
    for (int i = 0; i < N; i++) {
        const double q0 = a[i] * y;
        q[i] = __builtin_fma(-__builtin_fma(b, q0, -a[i]), y, q0);
        mag += __builtin_fabs(a[i]);
        const int e = __builtin_amdgcn_frexp_exp(a[i]);  // 0 for a zero
        emin = i == 0 ? e : min(emin, e);
    }
    // |a[i]| <= sum <= 2^302 (false for NaN or inf), exponent(a[i]) >= -298
    // for a[i] != 0 (frexp: a = m 2^e, 0.5 <= |m| < 1), b in [2^-300, 2^300]
    const bool ok = mag <= 0x1p302 && emin >= -298 && b >= 0x1p-300 && b <= 0x1p300;
    if (__builtin_expect(!ok, 0))
        for (int i = 0; i < N; i++) q[i] = a[i] / b;
}

// sqrt(a[i]/b[i]) (i < N) with both roundings, for FP64, on operands in
// [2^-299, 2^300]: the quotient as in div_shared (and then in sqrt_n's range),
// the root as in sqrt_n.  lo, hi: the least and greatest operand; a NaN operand
// does not enter them and gives NaN.
template <int N>
__device__ __forceinline__ void root_quotients_core(const double *a, const double *b, double *r, double &lo,
                                                    double &hi)
{
    for (int i = 0; i < N; i++) {
        const double y0 = __builtin_amdgcn_rcp(b[i]);
        const double y1 = __builtin_fma(y0, __builtin_fma(-b[i], y0, 1.0), y0);
        const double y = __builtin_fma(y1, __builtin_fma(-b[i], y1, 1.0), y1);
        const double q0 = a[i] * y;
        const double v = __builtin_fma(-__builtin_fma(b[i], q0, -a[i]), y, q0);
        const double z = __builtin_amdgcn_rsq(v);
        const double s0 = v * z, h0 = z * 0.5;
        const double rr = __builtin_fma(-h0, s0, 0.5);
        const double h1 = __builtin_fma(h0, rr, h0), s1 = __builtin_fma(s0, rr, s0);
        const double s2 = __builtin_fma(__builtin_fma(-s1, s1, v), h1, s1);
        r[i] = __builtin_fma(__builtin_fma(-s2, s2, v), h1, s2);
        const double l = __builtin_fmin(a[i], b[i]), h = __builtin_fmax(a[i], b[i]);
        lo = i == 0 ? l : __builtin_fmin(lo, l);
        hi = i == 0 ? h : __builtin_fmax(hi, h);
    }
}
constexpr double kRootLo = 0x1p-299, kRootHi = 0x1p300;
template <int N>
__device__ __forceinline__ void root_quotients(const double *a, const double *b, double *r)
{
    double lo, hi;
    root_quotients_core<N>(a, b, r, lo, hi);
    if (__builtin_expect(!(lo >= kRootLo && hi <= kRootHi), 0))
        for (int i = 0; i < N; i++) r[i] = __builtin_sqrt(a[i] / b[i]);
}

// The signal speeds of one face (flux.f90:583-585): ap = max(0, vr+cr, vl+cl),
// am = max(0, -(vr-cr), -(vl-cl)) with c = sqrt(g p/d), as the reference's
// comparisons give them.  The hardware maximum gives the same but for NaN and
// for a -0 that a comparison with +0 lets through, which only -(v-c) can be
// (at v = c).  Operands of the roots outside their range, and faces where the
// product of both v-c is a zero or NaN, take the comparisons.
__device__ __forceinline__ void hll_speeds(const double gp[2], const double d[2], double vl, double vr, double &ap,
                                           double &am)
{
    double c[2], lo, hi;  // right, left
    root_quotients_core<2>(gp, d, c, lo, hi);
    const double er = vr - c[0], el = vl - c[1];
    ap = __builtin_fmax(__builtin_fmax(vr + c[0], 0.0), vl + c[1]);
    am = __builtin_fmax(__builtin_fmax(-er, 0.0), -el);
    if (__builtin_expect(!(lo >= kRootLo && hi <= kRootHi && __builtin_fabs(er * el) > 0.0), 0)) {
        const double cr = __builtin_sqrt(gp[0] / d[0]), cl = __builtin_sqrt(gp[1] / d[1]);
        ap = vmax(vmax(0.0, vr + cr), vl + cl);
        am = vmax(vmax(0.0, -(vr - cr)), -(vl - cl));
    }
}

// flux.f90:512-590 for one face: L = plus state of the cell below the face,
// R = minus state of the cell above it, direction dir (0,1,2).
template <typename T, int dir>
__device__ __forceinline__ void face_flux(const Side<T> &L, const Side<T> &R, T F[5])
{
    const T h = T(0.5);
    T sl[5], sr[5], fl[5], fr[5];
    sl[0] = L.d;
    sl[1] = L.d * L.v[0];
    sl[2] = L.d * L.v[1];
    sl[3] = L.d * L.v[2];
    sl[4] = L.e + h * L.d * (L.v[0] * L.v[0] + L.v[1] * L.v[1] + L.v[2] * L.v[2]);
    sr[0] = R.d;
    sr[1] = R.d * R.v[0];
    sr[2] = R.d * R.v[1];
    sr[3] = R.d * R.v[2];
    sr[4] = R.e + h * R.d * (R.v[0] * R.v[0] + R.v[1] * R.v[1] + R.v[2] * R.v[2]);
    const T vl = L.v[dir], vr = R.v[dir];
    const T zero = T(0);
    // fluxes_l = 0; fluxes_l(2+dir) = pl; then fluxes_l(k) = fluxes_l(k) + states_l(k)*vl
    fl[0] = sl[0] * vl;
    fl[1] = (dir == 0 ? L.p : zero) + sl[1] * vl;
    fl[2] = (dir == 1 ? L.p : zero) + sl[2] * vl;
    fl[3] = (dir == 2 ? L.p : zero) + sl[3] * vl;
    fl[4] = (sl[4] + L.p) * vl;
    fr[0] = sr[0] * vr;
    fr[1] = (dir == 0 ? R.p : zero) + sr[1] * vr;
    fr[2] = (dir == 1 ? R.p : zero) + sr[2] * vr;
    fr[3] = (dir == 2 ? R.p : zero) + sr[3] * vr;
    fr[4] = (sr[4] + R.p) * vr;
    // flux_hll, flux.f90:583-589
    T ap, am;
    if constexpr (sizeof(T) == 8) {
        const double gp[2] = {R.g * R.p, L.g * L.p}, d[2] = {R.d, L.d};
        hll_speeds(gp, d, vl, vr, ap, am);
    } else {
        const T cr = Arith<T>::root(Arith<T>::div(R.g * R.p, R.d));
        const T cl = Arith<T>::root(Arith<T>::div(L.g * L.p, L.d));
        ap = vmax(vmax(zero, vr + cr), vl + cl);
        am = vmax(vmax(zero, -(vr - cr)), -(vl - cl));
    }
    const T apam = ap * am;
    const T den = ap + am;
    if constexpr (sizeof(T) == 8) {
        double num[5];
#pragma unroll
        for (int i = 0; i < 5; i++) num[i] = ap * fl[i] + am * fr[i] - apam * (sr[i] - sl[i]);
        div_shared<5>(num, den, F);
    } else {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const T num = ap * fl[i] + am * fr[i] - apam * (sr[i] - sl[i]);
            F[i] = Arith<T>::div(num, den);
        }
    }
}

// centred coordinate of cell index i (1-based) on an axis of n cells (init_grid.f90:85-93)
__device__ __forceinline__ double centre(double d, int i, int n) { return d * ((double)i - ((double)n + 1.0) / 2.0); }

// flux_ang.f90:523-618 (get_fluxes_ang) for one face: the momentum slots carry
// the reconstructed r- and angular momenta, and the pressure force is projected
// with the centre (x, y, r) of the cell whose flux it is: the cell above the
// face (F, all five) and the cell below it (G, the two momentum slots; the
// others are F's).  Along z there is no projection and G is F's.
struct AngCentre {
    double x, y, r;
    // flux_ang.f90:40-61: linear momenta to r- and angular momentum
    __device__ __forceinline__ void to(double m1, double m2, double &rm, double &am) const
    {
        am = x * m2 - y * m1;
        rm = (m1 * x + m2 * y) / r;
    }
    // flux_ang.f90:245-268: and back
    __device__ __forceinline__ void back(double rm, double am, double &m1, double &m2) const
    {
        m1 = (rm * x - am * y / r) / r;
        m2 = (rm * y + am * x / r) / r;
    }
};
template <int dir>
__device__ __forceinline__ void face_flux_ang(const Side<double> &L, const Side<double> &R, const AngCentre &up,
                                              const AngCentre &below, double F[5], double G[2])
{
    const double sl[5] = {L.d, L.s1, L.s2, L.d * L.v[2],
                          L.e + 0.5 * L.d * (L.v[0] * L.v[0] + L.v[1] * L.v[1] + L.v[2] * L.v[2])};
    const double sr[5] = {R.d, R.s1, R.s2, R.d * R.v[2],
                          R.e + 0.5 * R.d * (R.v[0] * R.v[0] + R.v[1] * R.v[1] + R.v[2] * R.v[2])};
    const double vl = L.v[dir], vr = R.v[dir];
    // flux_hll, flux.f90:583-589
    const double gp[2] = {R.g * R.p, L.g * L.p}, d[2] = {R.d, L.d};
    double ap, am;
    hll_speeds(gp, d, vl, vr, ap, am);
    const double apam = ap * am;
    auto numerator = [&](int i, double pl, double pr) {
        const double fl = pl + sl[i] * vl, fr = pr + sr[i] * vr;
        return ap * fl + am * fr - apam * (sr[i] - sl[i]);
    };
    auto momenta = [&](const AngCentre &c, double num[2]) {
        double pl1 = 0.0, pl2 = 0.0, pr1 = 0.0, pr2 = 0.0;
        if (dir < 2) {
            const double q[2] = {L.p * (dir == 0 ? c.x : c.y), R.p * (dir == 0 ? c.x : c.y)};
            double o[2];
            div_shared<2>(q, c.r, o);
            pl1 = o[0];
            pr1 = o[1];
            pl2 = dir == 0 ? -(L.p * c.y) : L.p * c.x;
            pr2 = dir == 0 ? -(R.p * c.y) : R.p * c.x;
        }
        num[0] = numerator(1, pl1, pr1);
        num[1] = numerator(2, pl2, pr2);
    };
    double num[7];
    num[0] = ap * (sl[0] * vl) + am * (sr[0] * vr) - apam * (sr[0] - sl[0]);
    momenta(up, num + 1);
    num[3] = numerator(3, dir == 2 ? L.p : 0.0, dir == 2 ? R.p : 0.0);
    num[4] = ap * ((sl[4] + L.p) * vl) + am * ((sr[4] + R.p) * vr) - apam * (sr[4] - sl[4]);
    double q[7];
    if constexpr (dir < 2) {
        momenta(below, num + 5);
        div_shared<7>(num, ap + am, q);
        G[0] = q[5];
        G[1] = q[6];
    } else {
        div_shared<5>(num, ap + am, q);
        G[0] = q[1];
        G[1] = q[2];
    }
    for (int i = 0; i < 5; i++) F[i] = q[i];
}

}  // namespace bx
