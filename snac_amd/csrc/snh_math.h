/*
 * snh_math.h -- scalar arithmetic of the explicit step, shared by the gfx950
 * kernels and host-side checks.  Every expression keeps the operand order of
 * the reference line it cites, so that with FMA contraction off the device
 * produces the reference's IEEE-754 double results.
 */
#ifndef SNH_MATH_H
#define SNH_MATH_H

#ifdef __HIPCC__
#define SNH_HD __host__ __device__ __forceinline__
#else
#include <math.h>
#define SNH_HD static inline
#endif

#include <limits.h>

/* x86-64 meaning of the reference's abs() applied to a double
 * (plastic_BI/Constitutive.c:290,409,413,483): cvttsd2si truncation, which
 * gives INT_MIN for NaN and out-of-range inputs, then abs(), which leaves
 * INT_MIN unchanged.  gfx950's own conversion saturates, so it is spelled out. */
SNH_HD int snh_ref_iabs(double x) {
    int t = (x > -2147483649.0 && x < 2147483648.0) ? (int)x : INT_MIN;
    if (t == INT_MIN) return INT_MIN;
    return t < 0 ? -t : t;
}

/* int + int of two abs() results, wrapping as the x86 add does */
SNH_HD int snh_iadd_wrap(int a, int b) { return (int)((unsigned)a + (unsigned)b); }

/* A divisor b as the unevaluated sum hi + lo = 1 / b (1 + 2^-104): quotients
 * by it are a product and an FMA, RN(a hi + RN(a lo)) (N. Brisebarre,
 * J.-M. Muller and S. K. Raina, "Accelerating correctly rounded
 * floating-point division when the divisor is known in advance", IEEE Trans.
 * Computers 53 (2004), method 1).  The sum before the rounding is within
 * 2^-52 ulp of a / b, so the result is RN(a / b) unless the quotient lies that
 * close to a rounding midpoint.  That takes a dividend and a divisor made for
 * it: 2^n over the largest number below a power of two, and one pair besides
 * in 1.7e7 built near such midpoints; 4e9 random quotients on gfx950 gave no
 * difference from the division.  Either sign of b; normal range only.
 *
 * From an estimate of 1 / b good to 2^-23 (v_rcp_f64, v_rsq_f64), one or two
 * Newton steps (P. Markstein, 1990) make hi faithful; the residual
 * 1 - b hi is then exact, and lo is its product with hi.  hi itself is RN(1/b)
 * for all but a few b just below a power of two: snh_recip_rn gives that. */
typedef struct {
    double hi, lo;
} snh_recip;
SNH_HD snh_recip snh_recip_of(double b, double y) {
    snh_recip r;
    double e = fma(-b, y, 1.0);
    r.hi = fma(e, y, y);
    e = fma(-b, r.hi, 1.0);
    r.lo = e * r.hi;
    return r;
}
SNH_HD double snh_quot(double a, snh_recip r) { return fma(a, r.hi, a * r.lo); }

/* RN(1 / b).  For b = 2 - k 2^-52 (times a power of two) with a small odd k,
 * 1 / b lies k^2 2^-54 ulp beyond a midpoint, so hi, the nearest to within
 * 2^-49 ulp, may be the number on the other side, and for k = 1 so may the
 * rounded sum hi + lo; a 2^-105 part of hi more settles that case and is too
 * little to matter in any other. */
SNH_HD double snh_recip_rn(snh_recip r) { return r.hi + fma(r.hi, 0x1p-105, r.lo); }

/* the pair from an estimate y of 1 / b good to 2^-23 */
SNH_HD snh_recip snh_recip_refine(double b, double y) { return snh_recip_of(b, fma(fma(-b, y, 1.0), y, y)); }
SNH_HD snh_recip snh_recip_make(double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return snh_recip_refine(b, __builtin_amdgcn_rcp(b));
#else
    return snh_recip_refine(b, 1.0 / b);
#endif
}

/* RN(sqrt(x)) for x > 0 and, in r, the reciprocal of that root, from an
 * estimate y of 1 / sqrt(x) good to 2^-23.  Goldschmidt's coupled iteration
 * for sqrt(x) and 1 / (2 sqrt(x)), then two residual corrections of the root
 * (Markstein 1990; Muller et al., Handbook of Floating-Point Arithmetic, 2nd
 * ed., sec. 4.7), which give the correctly rounded root; the reciprocal comes
 * out of the same iteration instead of a division.  Without the scaling of the
 * library's sqrt: x from 2^-918 to 2^1023 (x = 0 gives NaN, as the 0 / 0 of a
 * face without area does).  13 instructions for root and reciprocal and 2 per
 * quotient, against 31 and 5 with sqrt, 1 / s and quotients corrected twice by
 * their residual. */
SNH_HD double snh_sqrt_refine(double x, double y, snh_recip* r) {
    double g = x * y, h = 0.5 * y;
    const double t = fma(-h, g, 0.5);
    g = fma(g, t, g);
    h = fma(h, t, h);
    double d = fma(-g, g, x);
    g = fma(d, h, g);
    d = fma(-g, g, x);
    g = fma(d, h, g);
    *r = snh_recip_of(g, h + h);
    return g;
}
SNH_HD double snh_sqrt_recip(double x, snh_recip* r) {
#if defined(__HIP_DEVICE_COMPILE__)
    return snh_sqrt_refine(x, __builtin_amdgcn_rsq(x), r);
#else
    return snh_sqrt_refine(x, 1.0 / sqrt(x), r);
#endif
}

/* hypot(x, y) as the reference's libm computes it.  The reference calls the
 * system hypot in tql2 (plastic_BI/Constitutive.c:430,462); on x86-64 with
 * glibc 2.35 that is the unfused form of C. F. Borges' corrected square root
 * ("An improved algorithm for hypot(a,b)", arXiv:1904.09481, MyHypot3):
 * h = sqrt(ax^2 + ay^2) rounded, then one correction h -= (t1 + t2) / 2h
 * with the error terms of the branch h <= 2 ay or h > 2 ay, evaluated in
 * plain double arithmetic (no FMA).  Operands below 2^-459 or above 2^511
 * are scaled by 2^600; a term below 2^-54 of the other is added directly.
 * The result is faithful, not always correctly rounded (about 2 in 10^3
 * results are one ulp from the correctly rounded value), and this restatement
 * gives the system hypot's bits: checked on the host against the libm
 * function.  Requires FMA contraction off. */
SNH_HD double snh_hypot_kernel(double ax, double ay) {
    snh_recip rh;
    double h = snh_sqrt_recip(ax * ax + ay * ay, &rh);
    double t1, t2;
    if (h <= 2.0 * ay) {
        const double delta = h - ay;
        t1 = ax * (2.0 * delta - ax);
        t2 = (delta - 2.0 * (ax - ay)) * delta;
    } else {
        const double delta = h - ax;
        t1 = 2.0 * delta * (ax - 2.0 * ay);
        t2 = (4.0 * delta - ay) * ay + delta * delta;
    }
    h -= 0.5 * snh_quot(t1 + t2, rh);   /* (t1 + t2) / (2 h) */
    return h;
}

SNH_HD double snh_hypot(double x, double y) {
    if (!isfinite(x) || !isfinite(y)) {
        if (isinf(x) || isinf(y)) return INFINITY;
        return x + y;
    }
    x = fabs(x);
    y = fabs(y);
    const double ax = x < y ? y : x, ay = x < y ? x : y;
    if (ax > 0x1p+511) {
        if (ay <= ax * 0x1p-54) return ax + ay;
        return snh_hypot_kernel(ax * 0x1p-600, ay * 0x1p-600) / 0x1p-600;
    }
    if (ay < 0x1p-459) {
        if (ax >= ay / 0x1p-54) return ax + ay;
        return snh_hypot_kernel(ax / 0x1p-600, ay / 0x1p-600) * 0x1p-600;
    }
    if (ay <= ax * 0x1p-54) return ax + ay;
    return snh_hypot_kernel(ax, ay);
}

/* RN(x / 3) without a division.  x = M 2^e with integer M, and ulp(x/3) <=
 * ulp(x), so x/3 measured in ulps of the result has fractional part 0, 1/3 or
 * 2/3: the exact quotient is at least 1/6 ulp from every rounding midpoint.
 * q = RN(x * RN(1/3)) is within 1.5 ulp; r = x - 3q is then a multiple of
 * ulp(q) of magnitude <= 3 ulp(q), so the FMA computes it exactly; and
 * q + r*RN(1/3) differs from x/3 by r*(RN(1/3) - 1/3) < 2^-53 ulp, which
 * cannot move it across a midpoint.  Hence one rounding gives RN(x/3), for all
 * normal x (zero keeps its magnitude; -0 may come out as +0). */
SNH_HD double snh_div3(double x) {
    const double y = 0x1.5555555555555p-2; /* RN(1/3) */
    double q = x * y;
    double r = fma(-3.0, q, x);
    return fma(r, y, q);
}

/* RN(c x / 3) for c a power of two, of either sign: c times the steps above,
 * exactly (a power of two commutes with rounding in the normal range), so a
 * halving, quartering or sign beside the division costs nothing.
 * RN(x / 6) is c = 1/2. */
#define SNH_DIV3C(name, c)                               \
    SNH_HD double name(double x) {                       \
        const double y = (c) * 0x1.5555555555555p-2;     \
        double q = x * y;                                \
        double r = fma(-3.0 / (c), q, x);                \
        return fma(r, y, q);                             \
    }
SNH_DIV3C(snh_div6, 0.5)
SNH_DIV3C(snh_div12, 0.25)
SNH_DIV3C(snh_ndiv6, -0.5)
SNH_DIV3C(snh_ndiv12, -0.25)

#endif
