// The line-vortex kernel K(line, p) of the reference (src/core/flow_solver.c:114-135):
//
//   dr1 = p - r1, dr2 = p - r2, t_i = e . dr_i, h^2 = ((|dr1|^2 - t1^2) + (|dr2|^2 - t2^2)) / 2
//   K = 0                                            if |d| < tol or h^2 < tol^2
//   K = cross(dr1, e) * (atan2(t2, h) - atan2(t1, h)) / h   otherwise
//
// |K| is the angle the segment subtends from p (no 1/(4 pi) factor).  The file must be
// compiled with -ffp-contract=off: in PVL_FP64_REF, in the tensors, and wherever else the general
// form is taken from both end points (pair_m), the dot products, h^2 and the cut-off test
// round exactly as the reference's GCC x86-64 build (left to right, no FMA), so the cut-off
// branch is decided identically and the cancellation in h^2 near a segment's line (which
// the reference's values carry) is reproduced.  FMAs appear only where written explicitly:
// in the angle evaluation and, for the non-reference forms, in the cross product and the
// circulation-weighted accumulation (1-ulp differences, no effect on the cut-off).
// Two forms take h^2 = |dr1 x e|^2 with FMAs and decide the cut-off by that: the wake's
// self-induction (cross_m, far_add) and the far form of the FP64 assembly and point sums (line_nk,
// line_k_acc).  Its error is of the order of eps |dr1| h + (eps |dr1|)^2, the reference's of eps |dr1|^2, so the
// decisions differ only where |h^2 - tol^2| is within a few eps |dr1|^2: beside a line's extension,
// for a pair worth at most 2 len sqrt(tol^2 + 8 eps |dr1|^2) / |dr1|^2.
//
// Angle forms:
//   PVL_FP64_REF  the reference's expression: two FP64 atan2 calls of the HIP math library.
//   PVL_FP64      one angle: atan2(t2, h) - atan2(t1, h) = atan2((t2 - t1) h, h^2 + t1 t2).
//                 Both sides lie in (-pi, pi): with r_i = sqrt(h^2 + t_i^2) > 0, the sine and
//                 cosine of the difference are (t2 - t1) h / (r1 r2) and (h^2 + t1 t2) /
//                 (r1 r2).  The error of this form is a few 1e-15 relative to the angle
//                 everywhere (the atan polynomial, the quotient and 1/h below, each ~1e-15),
//                 whereas the difference of two atan2 values loses digits in the far field
//                 (|angle| << pi); the two forms agree to that loss (~1e-14 at r/len ~ 100).
//                 atan2 is this library's own (pvl_atan2 below), 1/h comes from a
//                 refined reciprocal square root.  Far from a line (all points of a wave) a
//                 polynomial in h^2 / B^2 takes the place of both (far forms below).
//   PVL_FP32      as PVL_FP64's general form at every distance, with the angle, h and 1/h in FP32
//                 (cut-off, dots, h^2 and cross(dr1, e) stay FP64); ~1e-7 relative.
#pragma once

#include "pvl_internal.hpp"

enum
{
    PVL_FP64_REF_FORM = 2
};

// atan(a) = a + a s P(s), s = a^2, 0 <= a <= 1.  Minimax coefficients fitted by
// pyvl_amd/csrc/tools/fit_atan.py (Lawson iteration in 60-digit arithmetic): P of degree 16
// for FP64 (maximum relative error of the polynomial 1.1e-15, ~5 ulp: the pair's other
// rounding errors are of that order), degree 7 for FP32 (1.7e-8).
// VGPR_COEF: every Horner step as one three-address v_fma_f64 with the coefficient in VGPRs, where
// the kernel has those to spare.  In loops with enough control flow around the evaluation the
// compiler otherwise keeps the loop-invariant coefficients in VGPRs all the same and emits every
// step as a copy plus the two-address v_fmac_f64 (twice the instructions); the same FMAs in the same
// order, so the results are bit-identical.
template <bool VGPR_COEF> __device__ __forceinline__ double fma_step(double p, double s, double c)
{
    if constexpr (VGPR_COEF)
    {
        double r;
        asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(p), "v"(s), "v"(c));
        return r;
    }
    else
        return fma(p, s, c);
}
template <bool V = false> __device__ __forceinline__ double atan_poly64(double a)
{
    const double s = a * a;
    double p = -4.7926633120228785553e-5;
    p = fma_step<V>(p, s, 4.800660567800612957e-4);
    p = fma_step<V>(p, s, -2.2725728333658927666e-3);
    p = fma_step<V>(p, s, 6.8183912427924839848e-3);
    p = fma_step<V>(p, s, -1.4739706399322470277e-2);
    p = fma_step<V>(p, s, 2.4909137877934616446e-2);
    p = fma_step<V>(p, s, -3.5142229350564300719e-2);
    p = fma_step<V>(p, s, 4.3938991765738211806e-2);
    p = fma_step<V>(p, s, -5.1356486201903778769e-2);
    p = fma_step<V>(p, s, 5.8483233451193392607e-2);
    p = fma_step<V>(p, s, -6.6598275562737410628e-2);
    p = fma_step<V>(p, s, 7.6913027337110721971e-2);
    p = fma_step<V>(p, s, -9.090805442522420044e-2);
    p = fma_step<V>(p, s, 1.1111104041852547122e-1);
    p = fma_step<V>(p, s, -1.4285713995249626285e-1);
    p = fma_step<V>(p, s, 1.9999999993898812193e-1);
    p = fma_step<V>(p, s, -3.3333333333288106455e-1);
    return fma(a * s, p, a);
}

// The same polynomial with its coefficients loaded (scalar loads): for a less often taken branch
// beside a loop that needs the scalar registers itself.  atan_table() at the branch's start gives
// an address that is opaque to the compiler, which would otherwise hoist the loads out of it.
static __constant__ double kAtanTable[17] = {
    -4.7926633120228785553e-5, 4.800660567800612957e-4,  -2.2725728333658927666e-3, 6.8183912427924839848e-3,
    -1.4739706399322470277e-2, 2.4909137877934616446e-2, -3.5142229350564300719e-2, 4.3938991765738211806e-2,
    -5.1356486201903778769e-2, 5.8483233451193392607e-2, -6.6598275562737410628e-2, 7.6913027337110721971e-2,
    -9.090805442522420044e-2,  1.1111104041852547122e-1, -1.4285713995249626285e-1, 1.9999999993898812193e-1,
    -3.3333333333288106455e-1};
using AtanTable = const __attribute__((address_space(4))) double *; // constant memory: scalar loads
__device__ __forceinline__ AtanTable atan_table()
{
    AtanTable t = (AtanTable)kAtanTable;
    asm volatile("" : "+s"(t));
    return t;
}
__device__ __forceinline__ double atan_poly64_table(double a, AtanTable t)
{
    const double s = a * a;
    double p = t[0];
#pragma unroll
    for (int k = 1; k < 17; ++k)
        p = fma(p, s, t[k]);
    return fma(a * s, p, a);
}

__device__ __forceinline__ float atan_poly32(float a)
{
    const float s = a * a;
    float p = 2.9206460455115316945e-3f;
    p = fmaf(p, s, -1.6367743921648625112e-2f);
    p = fmaf(p, s, 4.3211563153423941466e-2f);
    p = fmaf(p, s, -7.5521892793692703723e-2f);
    p = fmaf(p, s, 1.0665993049895164418e-1f);
    p = fmaf(p, s, -1.4211052413584158043e-1f);
    p = fmaf(p, s, 1.9993772488057382827e-1f);
    p = fmaf(p, s, -3.3333152721644904729e-1f);
    return fmaf(a * s, p, a);
}

// atan2(y, x) for finite arguments not both zero: a = min(|x|,|y|) / max(|x|,|y|) in [0, 1]
// (the hardware reciprocal, within 2^-24 relative on gfx950 (measured), refined by one
// Newton step to ~2^-48: a within ~4e-15 relative, and atan(a) within that as well since
// a / ((1 + a^2) atan(a)) <= 1), atan(a) from the polynomial, then the octant:
// pi/2 - . when |y| > |x|, pi - . when x < 0, sign of y.
__device__ __forceinline__ double pvl_atan2(double y, double x)
{
    const double ax = fabs(x), ay = fabs(y);
    const double mn = fmin(ax, ay), mx = fmax(ax, ay);
    double r = __builtin_amdgcn_rcp(mx);
    r = fma(r, fma(-mx, r, 1.0), r);
    const double a = mn * r;
    double t = atan_poly64(a);
    t = (ay > ax) ? (1.57079632679489661923 - t) : t;
    t = (x < 0.0) ? (3.14159265358979323846 - t) : t;
    return copysign(t, y);
}

// atan2(-ay, x) for ay >= 0 (the segment's angle below: its sine is never positive), as
// pvl_atan2 without the sign transfer.
template <int COEF = 0>
__device__ __forceinline__ double pvl_atan2_neg(double ay, double x, AtanTable table = nullptr)
{
    const double ax = fabs(x);
    const double mn = fmin(ax, ay), mx = fmax(ax, ay);
    double r = __builtin_amdgcn_rcp(mx);
    r = fma(r, fma(-mx, r, 1.0), r);
    const double a = mn * r;
    double t;
    if constexpr (COEF == 2)
        t = atan_poly64_table(a, table);
    else
        t = atan_poly64<COEF == 1>(a);
    t = (ay > ax) ? (1.57079632679489661923 - t) : t;
    t = (x < 0.0) ? (3.14159265358979323846 - t) : t;
    return -t;
}

__device__ __forceinline__ float pvl_atan2f(float y, float x)
{
    const float ax = fabsf(x), ay = fabsf(y);
    const float mn = fminf(ax, ay), mx = fmaxf(ax, ay);
    const float a = mn * __builtin_amdgcn_rcpf(mx);
    float t = atan_poly32(a);
    t = (ay > ax) ? (1.57079632679489661923f - t) : t;
    t = (x < 0.0f) ? (3.14159265358979323846f - t) : t;
    return copysignf(t, y);
}

// 1/sqrt(x) for x > 0 normal: the hardware estimate y (within 2^-23 relative on gfx950,
// measured) and one third-order step of 1/sqrt(x) = y (1 - e)^(-1/2) =
// y (1 + e/2 + 3 e^2/8 + 5 e^3/16 + ...), e = 1 - x y^2: the first omitted term is below
// 2^-66 relative for |e| <= 2^-22, so the result is within rounding of 1/sqrt(x).
__device__ __forceinline__ double pvl_rsqrt(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Scalar factor of K from the pair's endpoint terms: dr1 = p - r1 and q1 = |dr1|^2, dr2 and
// q2 likewise (each dot product left to right, no FMA, as the reference), e = the unit
// direction.  The cut-off is decided here.  Split from line_m so that a walk along a chain of
// segments can reuse one endpoint's terms for the next segment (bit-identical values).
template <int PREC, int COEF = 0>
__device__ __forceinline__ double pair_m(double ex, double ey, double ez, double len, double d1x, double d1y,
                                         double d1z, double q1, double d2x, double d2y, double d2z, double q2,
                                         double tol, double tol2, bool &cut, AtanTable table = nullptr)
{
    const double t1 = ex * d1x + ey * d1y + ez * d1z;
    const double t2 = ex * d2x + ey * d2y + ez * d2z;
    const double n1 = q1 - t1 * t1;
    const double n2 = q2 - t2 * t2;
    const double h2 = (n1 + n2) / 2.0;
    double m;
    if constexpr (PREC == PVL_FP64_REF_FORM)
    {
        cut = (len < tol) || (h2 < tol2);
        const double hh = cut ? 1.0 : h2;
        const double h = sqrt(hh);
        m = (atan2(t2, h) - atan2(t1, h)) / h;
    }
    else
    {
        // Only h2 < tol^2 is tested here: a line shorter than tol has direction 0 and length 0
        // (line_geom_kernel), so t1 = t2 = 0, the angle atan2(-0, h2 > 0) is 0 and the line
        // adds exactly 0, as the reference's cut-off does.  A cut pair's h2 (possibly <= 0)
        // may give NaN or Inf below; the caller replaces the pair's value by 0.
        // t2 - t1 = e . (r1 - r2) = -len exactly in exact arithmetic; -len is used (the
        // rounded difference of t1 and t2 carries an error of eps |dr| / len relative in the
        // far field).  A line cut by length has len = 0 (line_geom_kernel), so its angle is 0.
        cut = h2 < tol2;
        if constexpr (PREC == PVL_FP64)
        {
            const double ih = pvl_rsqrt(h2);
            const double h = h2 * ih;
            const double dphi = pvl_atan2_neg<COEF>(len * h, fma(t1, t2, h2), table);
            m = dphi * ih;
        }
        else
        {
            const float hf = sqrtf((float)h2);
            const float ihf = __builtin_amdgcn_rcpf(hf);
            const float num = -(float)len * hf;
            const float den = (float)fma(t1, t2, h2);
            m = (double)(pvl_atan2f(num, den) * ihf);
        }
    }
    return m;
}

// K = c m for the wake's self-induction in the accurate forms (PVL_FP64, PVL_FP32), from
// dr1 = p - r1 and the segment's unit direction e and length: c = dr1 x e (K's direction,
// |c| = h, the distance of p from the segment's line), h^2 = |c|^2, t1 = e . dr1 (FMAs),
// t2 = t1 - len; returns m = angle / h and decides the cut-off (h^2 < tol^2).  Mathematically
// the reference's h^2; numerically its error is ~eps |dr1| / h relative (the cross product's
// own, which K's direction carries in every form), where the reference's |dr|^2 - t^2 loses
// ~eps |dr|^2 / h^2, so the two differ by the reference's rounding, which is of the order of
// eps wherever |dr| / h is of the order of one (a sheet of segments of similar length, as a
// free wake is).  It needs neither |dr1|^2 nor dr2, ~18 instructions fewer per pair.  A line
// shorter than tol has direction 0 and length 0 (chain records), so c = 0, h^2 = 0 and it is
// cut, as the reference's length test cuts it.  A cut pair's m may be NaN or Inf; the caller
// replaces the pair's value by 0.
template <int PREC, int COEF = 0>
__device__ __forceinline__ double cross_m(double ex, double ey, double ez, double len, double d1x, double d1y,
                                          double d1z, double tol2, double &cx, double &cy, double &cz, bool &cut,
                                          AtanTable table = nullptr)
{
    cx = fma(d1y, ez, -(d1z * ey));
    cy = fma(d1z, ex, -(d1x * ez));
    cz = fma(d1x, ey, -(d1y * ex));
    const double h2 = fma(cx, cx, fma(cy, cy, cz * cz));
    const double t1 = fma(ex, d1x, fma(ey, d1y, ez * d1z));
    const double t2 = t1 - len;
    cut = h2 < tol2;
    if constexpr (PREC == PVL_FP64)
    {
        const double ih = pvl_rsqrt(h2);
        const double h = h2 * ih;
        return pvl_atan2_neg<COEF>(len * h, fma(t1, t2, h2), table) * ih;
    }
    else
    {
        const float hf = sqrtf((float)h2);
        const float ihf = __builtin_amdgcn_rcpf(hf);
        const float num = -(float)len * hf;
        const float den = (float)fma(t1, t2, h2);
        return (double)(pvl_atan2f(num, den) * ihf);
    }
}

// Far form of angle / h, for pairs whose point is further than about four segment lengths from
// the segment's midpoint: with A = len h and B = dr1 . dr2 = h^2 + t1 t2 the angle is
// atan(A / B), and angle / h = (len / B) (1 + s P(s)), s = (len / B)^2 h^2 -- a function of
// h^2 alone, so neither the square root nor the octant logic of atan2 is needed, and a short
// P suffices.  B = |m|^2 - len^2 / 4 for the distance m from the midpoint, so |m| >= 4 len makes
// B positive and gives s <= 0.0645, over which the degree-6 P below has a relative error of
// 4.6e-16 (tools/fit_atan.py 6 double 0.0645; the general form's polynomial: 1.1e-15).  1/B is
// the hardware reciprocal and one Newton step, as in pvl_atan2.  Callers decide by the boxes of
// a wave's points and of a group of lines, so the evaluation itself carries no test.
constexpr int kFarTerms = 7;
constexpr double kFar1 = -3.3333333333275589419e-1, kFar2 = 1.9999999977026864496e-1,
                 kFar3 = -1.4285711189790686119e-1, kFar4 = 1.1110912812573140192e-1,
                 kFar5 = -9.0840857012789507027e-2, kFar6 = 7.5620986412452229467e-2,
                 kFar7 = -5.3494538871327659169e-2;
// Distance of a point from a line of length len from which on the far form holds (4 len from the
// midpoint, and a margin for the rounding of the boxes).  Lines cut by length (len 0) and lengths
// whose 15th powers could leave the range of a double take the general form for every point.
__device__ __forceinline__ double far_reach(double len)
{
    return (len >= 1e-12 && len <= 1e12) ? 4.000001 * len : __builtin_inf();
}
__device__ __forceinline__ double far_rcp(double b)
{
    const double r = __builtin_amdgcn_rcp(b);
    return fma(r, fma(-b, r, 1.0), r);
}

// Scalar factor of K (angle / h; the cut-off is decided here) and dr1 = p - r1.
template <int PREC>
__device__ __forceinline__ double line_m(const LineGeom &g, double px, double py, double pz, double tol, double tol2,
                                         double &d1x, double &d1y, double &d1z, bool &cut)
{
    d1x = px - g.r1x, d1y = py - g.r1y, d1z = pz - g.r1z;
    const double d2x = px - g.r2x, d2y = py - g.r2y, d2z = pz - g.r2z;
    const double q1 = d1x * d1x + d1y * d1y + d1z * d1z;
    const double q2 = d2x * d2x + d2y * d2y + d2z * d2z;
    return pair_m<PREC>(g.ex, g.ey, g.ez, g.len, d1x, d1y, d1z, q1, d2x, d2y, d2z, q2, tol, tol2, cut);
}

// K(line, p).  The reference form keeps the reference's cross product and products; the
// others fuse the cross product's second product into an FMA (the cut-off decision and
// every quantity it depends on are unchanged).
template <int PREC>
__device__ __forceinline__ void line_k(const LineGeom &g, double px, double py, double pz, double tol, double tol2,
                                       double &kx, double &ky, double &kz)
{
    double d1x, d1y, d1z;
    bool cut;
    const double m = line_m<PREC>(g, px, py, pz, tol, tol2, d1x, d1y, d1z, cut);
    if constexpr (PREC == PVL_FP64_REF_FORM)
    {
        const double cx = d1y * g.ez - d1z * g.ey;
        const double cy = d1z * g.ex - d1x * g.ez;
        const double cz = d1x * g.ey - d1y * g.ex;
        kx = cut ? 0.0 : cx * m;
        ky = cut ? 0.0 : cy * m;
        kz = cut ? 0.0 : cz * m;
    }
    else
    {
        const double cx = fma(d1y, g.ez, -(d1z * g.ey));
        const double cy = fma(d1z, g.ex, -(d1x * g.ez));
        const double cz = fma(d1x, g.ey, -(d1y * g.ex));
        kx = cut ? 0.0 : cx * m;
        ky = cut ? 0.0 : cy * m;
        kz = cut ? 0.0 : cz * m;
    }
}

// The far form for a line tested by itself, for points in no particular order (boxes are useless
// there): from two lengths off the midpoint on B >= 3.75 len^2 and s <= 0.2845, over which the
// degree-10 P has a relative error of 3.2e-16 (tools/fit_atan.py 10 double 0.2844).  Returns
// angle / h (negative, as K's factor) from q = len / B and h^2.
template <bool VGPR_COEF> __device__ __forceinline__ double mid_far(double q, double h2)
{
    const double u = (h2 * q) * q;
    double p = -1.0530409925033454105e-2;
    if constexpr (VGPR_COEF)
    {
        p = fma_step<true>(p, u, 2.9501554043661432491e-2);
        p = fma_step<true>(p, u, -4.6025268387594494587e-2);
        p = fma_step<true>(p, u, 5.7199422485590436944e-2);
        p = fma_step<true>(p, u, -6.6394999569895820257e-2);
        p = fma_step<true>(p, u, 7.6892308217604938091e-2);
        p = fma_step<true>(p, u, -9.0906782661688777695e-2);
        p = fma_step<true>(p, u, 1.1111100144380131558e-1);
        p = fma_step<true>(p, u, -1.4285713981516674141e-1);
        p = fma_step<true>(p, u, 1.9999999995777831413e-1);
        p = fma_step<true>(p, u, -3.3333333333312912204e-1);
    }
    else
        asm("v_fma_f64 %0, %0, %1, %2\n\t"
            "v_fma_f64 %0, %0, %1, %3\n\t"
            "v_fma_f64 %0, %0, %1, %4\n\t"
            "v_fma_f64 %0, %0, %1, %5\n\t"
            "v_fma_f64 %0, %0, %1, %6\n\t"
            "v_fma_f64 %0, %0, %1, %7\n\t"
            "v_fma_f64 %0, %0, %1, %8\n\t"
            "v_fma_f64 %0, %0, %1, %9\n\t"
            "v_fma_f64 %0, %0, %1, %10\n\t"
            "v_fma_f64 %0, %0, %1, %11"
            : "+v"(p)
            : "v"(u), "s"(2.9501554043661432491e-2), "s"(-4.6025268387594494587e-2), "s"(5.7199422485590436944e-2),
              "s"(-6.6394999569895820257e-2), "s"(7.6892308217604938091e-2), "s"(-9.0906782661688777695e-2),
              "s"(1.1111100144380131558e-1), "s"(-1.4285713981516674141e-1), "s"(1.9999999995777831413e-1),
              "s"(-3.3333333333312912204e-1));
    return -fma(q * u, p, q);
}

// q = len / B also decides: 0 <= q len <= 1 / 3.75, as one unsigned comparison of the product's
// upper word, which negative values, infinities and NaN fail.  A line cut by length has q = 0 and
// adds 0.
__device__ __forceinline__ bool mid_holds(double q, double len)
{
    return (unsigned)(__double_as_longlong(q * len) >> 32) < 0x3FD11111u; // upper word of 1 / 3.75
}

// B = dr1 . dr2 from which on the far form holds for a line by itself (3.75 len^2; the same for a whole
// wave, decided before the reciprocal).  Infinite, so never reached, for lines cut by length and for lengths
// whose squares could leave the range of a double; the length is wave-uniform, its test scalar.
__device__ __forceinline__ double mid_reach(double len)
{
    const unsigned hi = (unsigned)(__double_as_longlong(len) >> 32);
    const bool in_range = hi - 0x2B300000u < 0x54C00000u - 0x2B300000u; // 2^-332 .. 2^333
    return in_range ? 3.75 * (len * len) : __builtin_inf();
}

// n . K(line, p) for the normal-reduced assembly.  The reference form dots the reference's K
// (reference rounding of every product); the others form m (n . c) with c = dr1 x e and the
// dot as FMAs and decide the cut-off once for the scalar; FP64 takes the far form when it holds for
// all points of the wave (FP32 keeps its single-precision angle at every distance).
template <int PREC>
__device__ __forceinline__ double line_nk(const LineGeom &g, double px, double py, double pz, double nx, double ny,
                                          double nz, double tol, double tol2)
{
    if constexpr (PREC == PVL_FP64_REF_FORM)
    {
        double kx, ky, kz;
        line_k<PREC>(g, px, py, pz, tol, tol2, kx, ky, kz);
        return kx * nx + ky * ny + kz * nz;
    }
    else
    {
        const double d1x = px - g.r1x, d1y = py - g.r1y, d1z = pz - g.r1z;
        const double d2x = px - g.r2x, d2y = py - g.r2y, d2z = pz - g.r2z;
        const double cx = fma(d1y, g.ez, -(d1z * g.ey));
        const double cy = fma(d1z, g.ex, -(d1x * g.ez));
        const double cz = fma(d1x, g.ey, -(d1y * g.ex));
        const double nc = fma(cx, nx, fma(cy, ny, cz * nz));
        if constexpr (PREC == PVL_FP64)
        {
            const double q = g.len * far_rcp(fma(d1x, d2x, fma(d1y, d2y, d1z * d2z)));
            if (__builtin_amdgcn_ballot_w64(!mid_holds(q, g.len)) == 0)
            {
                const double h2 = fma(cx, cx, fma(cy, cy, cz * cz));
                const double v = nc * mid_far<true>(q, h2);
                return h2 < tol2 ? 0.0 : v;
            }
        }
        const double q1 = d1x * d1x + d1y * d1y + d1z * d1z;
        const double q2 = d2x * d2x + d2y * d2y + d2z * d2z;
        bool cut;
        const double v = nc * pair_m<PREC, 1>(g.ex, g.ey, g.ez, g.len, d1x, d1y, d1z, q1, d2x, d2y, d2z, q2, tol, tol2,
                                              cut);
        return cut ? 0.0 : v;
    }
}

// v[j] += gamma K(line, p[j]): the point-velocity inner step.  FP32 and FP64 scale once and accumulate
// with FMAs.  FP64 takes the far form when it holds for all points of the wave (mid_reach): 46 issue
// slots per far pair against ~102 of the general form.  Like the general form it starts from
// the differences to the end points, so its error does not depend on where the mesh lies; records
// about the line's midpoint (three slots fewer) carry the midpoint's rounding, of the size of the
// coordinates: 4e-12 of the velocity for a body 1e5 radii off the origin, where the end points give 2e-15.
template <int PREC, int PPL>
__device__ __forceinline__ void line_k_acc(const LineGeom &g, double gamma, const double (&px)[PPL],
                                           const double (&py)[PPL], const double (&pz)[PPL], double tol, double tol2,
                                           double (&vx)[PPL], double (&vy)[PPL], double (&vz)[PPL])
{
    if constexpr (PREC == PVL_FP64_REF_FORM)
    {
#pragma unroll
        for (int j = 0; j < PPL; ++j)
        {
            double kx, ky, kz;
            line_k<PREC>(g, px[j], py[j], pz[j], tol, tol2, kx, ky, kz);
            vx[j] = vx[j] + gamma * kx;
            vy[j] = vy[j] + gamma * ky;
            vz[j] = vz[j] + gamma * kz;
        }
        return;
    }
    else if constexpr (PREC == PVL_FP32)
    {
#pragma unroll
        for (int j = 0; j < PPL; ++j)
        {
            double d1x, d1y, d1z;
            bool cut;
            const double m = line_m<PREC>(g, px[j], py[j], pz[j], tol, tol2, d1x, d1y, d1z, cut);
            const double wm = cut ? 0.0 : gamma * m;
            vx[j] = fma(wm, fma(d1y, g.ez, -(d1z * g.ey)), vx[j]);
            vy[j] = fma(wm, fma(d1z, g.ex, -(d1x * g.ez)), vy[j]);
            vz[j] = fma(wm, fma(d1x, g.ey, -(d1y * g.ex)), vz[j]);
        }
        return;
    }
    else
    {
        double cx[PPL], cy[PPL], cz[PPL], b[PPL], w[PPL];
        const double far_b = mid_reach(g.len);
        bool far = true;
#pragma unroll
        for (int j = 0; j < PPL; ++j)
        {
            const double d1x = px[j] - g.r1x, d1y = py[j] - g.r1y, d1z = pz[j] - g.r1z;
            const double d2x = px[j] - g.r2x, d2y = py[j] - g.r2y, d2z = pz[j] - g.r2z;
            b[j] = fma(d1x, d2x, fma(d1y, d2y, d1z * d2z));
            far = far && b[j] >= far_b;
            cx[j] = fma(d1y, g.ez, -(d1z * g.ey));
            cy[j] = fma(d1z, g.ex, -(d1x * g.ez));
            cz[j] = fma(d1x, g.ey, -(d1y * g.ex));
        }
        if (__builtin_amdgcn_ballot_w64(!far) == 0)
        {
#pragma unroll
            for (int j = 0; j < PPL; ++j)
            {
                const double h2 = fma(cx[j], cx[j], fma(cy[j], cy[j], cz[j] * cz[j]));
                const double f = gamma * mid_far<false>(g.len * far_rcp(b[j]), h2);
                w[j] = h2 < tol2 ? 0.0 : f;
            }
        }
        else
        {
            // one point per lane has the registers for the coefficients
            constexpr int COEF = PPL == 1 ? 1 : 2;
            AtanTable table = COEF == 2 ? atan_table() : nullptr;
#pragma unroll
            for (int j = 0; j < PPL; ++j)
            {
                const double d1x = px[j] - g.r1x, d1y = py[j] - g.r1y, d1z = pz[j] - g.r1z;
                const double d2x = px[j] - g.r2x, d2y = py[j] - g.r2y, d2z = pz[j] - g.r2z;
                const double q1 = d1x * d1x + d1y * d1y + d1z * d1z;
                const double q2 = d2x * d2x + d2y * d2y + d2z * d2z;
                bool cut;
                const double f = gamma * pair_m<PREC, COEF>(g.ex, g.ey, g.ez, g.len, d1x, d1y, d1z, q1, d2x, d2y, d2z, q2,
                                                         tol, tol2, cut, table);
                w[j] = cut ? 0.0 : f;
            }
        }
#pragma unroll
        for (int j = 0; j < PPL; ++j)
        {
            vx[j] = fma(w[j], cx[j], vx[j]);
            vy[j] = fma(w[j], cy[j], vy[j]);
            vz[j] = fma(w[j], cz[j], vz[j]);
        }
    }
}

