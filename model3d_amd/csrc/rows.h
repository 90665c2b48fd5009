// rows.h -- Solid.Contains along an axis-parallel line: where an atom is
// true on it, as an interval, so that one lane decides a whole row of
// corners (or all midpoints of an edge) instead of one point.
//
// A sphere, box, capsule or cylinder is convex, so the points of a line that
// lie in it are one interval.  atom_span bounds that interval from outside
// and from inside by more than the rounding of the reference's float64
// expressions (atom64) and of the computation here: a point past the outer
// bounds is false, a point within the inner bounds is true, and the few
// points between the two are decided by atom64 itself.  A program over such
// atoms is then a boolean expression over bit masks, one bit per point.
// Every decision is the one atom64 makes at the point.
#pragma once

#include "eval.h"

namespace mc3d {

// Along the line p + s e_k: false for s outside [ao, bo], true for s inside
// [ai, bi]; a NaN bound says nothing (row_mask).
struct Span {
    double ao, bo, ai, bi;
};
MC3D_HD inline Span span_none() { return Span{INFINITY, -INFINITY, INFINITY, -INFINITY}; }
MC3D_HD inline Span span_unsure() { return Span{-INFINITY, INFINITY, INFINITY, -INFINITY}; }
MC3D_HD inline Span span_all() { return Span{-INFINITY, INFINITY, -INFINITY, INFINITY}; }

MC3D_HD inline double sel3(int k, double a, double b, double c) { return k == 0 ? a : (k == 1 ? b : c); }

// 1 / sqrt(w) to a few digits; span_root's Newton step makes the rest.
MC3D_HD inline double rsq_estimate(double w) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(w);
#else
    return 1 / sqrt(w);
#endif
}

// ro >= sqrt(w') >= ri for every w' in [w - D, w + D] (w >= -D), with e0
// more on each side; ri < 0: w' may be below zero.
MC3D_HD inline void span_root(double w, double D, double e0, double &ro, double &ri) {
    if (w <= 4 * D) {  // the line grazes the surface
        ro = (double)sqrtf((float)(5 * D)) * 1.001 + e0;
        ri = -1;
        return;
    }
    const double y = rsq_estimate(w);
    double r = w * y;
    r = r + 0.5 * y * __builtin_fma(-r, r, w);
    const double e = 1.1 * D * y + 1e-10 * r + e0;
    ro = r + e;
    ri = r - e;
}

// Coordinates that are neither so large nor so small that a square or a
// product of two leaves the float64 range.
MC3D_HD inline bool span_range(double M) { return M > 1e-100 && M < 1e100; }

// Sphere about c with threshold T (s <= T), M bounding every coordinate and
// length: the line's squared distance is q, and s - T = x^2 + q - T.
// Rounding moves s by far less than 1e-13 M^2.
MC3D_HD inline Span sphere_span(double ck, double c1, double c2, double T, double pk, double p1, double p2, double M) {
    const double d1 = p1 - c1, d2 = p2 - c2, D = 1e-13 * M * M;
    const double w = T - (d1 * d1 + d2 * d2), m = ck - pk;
    if (w < -D) return span_none();
    double ro, ri;
    span_root(w, D, 1e-14 * M, ro, ri);
    Span s{m - ro, m + ro, INFINITY, -INFINITY};
    if (ri > 0) s.ai = m - ri, s.bi = m + ri;
    return s;
}

// Cylinder from q along the unit vector d, length L, threshold T: with
// v = p - q, c = v.d and n = v - c d, the squared distance from its axis is
// |n|^2 + 2 s n_k + s^2 (1 - d_k^2), the position along it c + s d_k.  smax:
// the largest |s| asked about (nearly parallel lines, where the roots or the
// end planes are ill-defined, are bounded over that range instead).
MC3D_HD inline Span cylinder_span(double qk, double q1, double q2, double dk, double d1, double d2, double L, double T,
                                  double pk, double p1, double p2, double smax, double M) {
    const double vk = pk - qk, v1 = p1 - q1, v2 = p2 - q2;
    const double c = vk * dk + v1 * d1 + v2 * d2;
    const double nk = vk - dk * c, n1 = v1 - d1 * c, n2 = v2 - d2 * c;
    const double w = T - (nk * nk + n1 * n1 + n2 * n2), A = d1 * d1 + d2 * d2, D = 1e-13 * M * M;
    Span s;
    if (A < 1e-6) {  // along the axis: the distance hardly changes
        const double D2 = D + 2 * fabs(nk) * smax + A * smax * smax;
        if (w < -D2) return span_none();
        s = w > D2 ? span_all() : span_unsure();
    } else {
        const double disc = nk * nk + A * w, DD = A * D + 1e-14 * nk * nk;
        if (disc < -DD) return span_none();
        double ro, ri;
        span_root(disc, DD, 0, ro, ri);
        const double iA = 1 / A, e = (1e-12 * (fabs(nk) + ro) + 1e-14 * M) * iA;
        s = Span{(-nk - ro) * iA - e, (-nk + ro) * iA + e, INFINITY, -INFINITY};
        if (ri > 0) s.ai = (-nk - ri) * iA + e, s.bi = (-nk + ri) * iA - e;
    }
    const double f = 1e-13 * M;  // rounding of the position along the axis
    if (fabs(dk) < 1e-7) {
        const double f2 = f + fabs(dk) * smax;
        if (c < -f2 || c > L + f2) return span_none();
        if (!(c > f2 && c < L - f2)) s.ai = INFINITY, s.bi = -INFINITY;
    } else {
        const double i = 1 / dk;
        const double t0 = (-f - c) * i, t1 = (L + f - c) * i, u0 = (f - c) * i, u1 = (L - f - c) * i;
        s.ao = fmax(s.ao, fmin(t0, t1)), s.bo = fmin(s.bo, fmax(t0, t1));
        s.ai = fmax(s.ai, dk > 0 ? u0 : u1), s.bi = fmin(s.bi, dk > 0 ? u1 : u0);
    }
    return s;
}

// Where an untransformed sphere, box, capsule or cylinder (params a, the
// layouts of AtomKind) is true on the line through (x, y, z) along axis k.
// mag: a bound of |x|, |y|, |z| and of the coordinates asked about.
template <class F64P>
MC3D_HD inline Span atom_span(uint32_t kind, F64P a, int k, double x, double y, double z, double smax, double mag) {
    const double pk = sel3(k, x, y, z), p1 = sel3(k, y, x, x), p2 = sel3(k, z, z, y);
    auto along = [&](int o) { return sel3(k, a[o], a[o + 1], a[o + 2]); };
    auto first = [&](int o) { return sel3(k, a[o + 1], a[o], a[o]); };
    auto second = [&](int o) { return sel3(k, a[o + 2], a[o + 2], a[o + 1]); };
    auto size = [&](int o) { return fabs(a[o]) + fabs(a[o + 1]) + fabs(a[o + 2]); };
    if (kind == A_RECT) {  // exact comparisons off the line's axis
        if (!(in_lo(p1, first(0)) && in_hi(p1, first(3)) && in_lo(p2, second(0)) && in_hi(p2, second(3))))
            return span_none();
        const double lo = along(0) - pk, hi = along(3) - pk;
        return Span{lo, hi, lo, hi};
    }
    if (kind == A_SPHERE) {
        const double M = 3 * mag + size(0) + a[3];
        if (!span_range(M)) return span_unsure();
        return sphere_span(along(0), first(0), second(0), a[4], pk, p1, p2, M);
    }
    if (kind == A_CYLINDER) {
        const double M = 3 * mag + size(0) + a[6] + a[7];
        if (!(span_range(M) && size(3) < 2)) return span_unsure();
        return cylinder_span(along(0), first(0), second(0), along(3), first(3), second(3), a[6], a[8], pk, p1, p2,
                             smax, M);
    }
    // capsule: the cylinder between two spheres; it is convex, so the hull
    // of their intervals (and of the certain parts of those) is its own
    const double M = 3 * mag + size(0) + size(3) + a[9] + a[10];
    if (!(span_range(M) && size(6) < 2)) return span_unsure();
    const Span u = sphere_span(along(0), first(0), second(0), a[11], pk, p1, p2, M);
    const Span v = sphere_span(along(3), first(3), second(3), a[11], pk, p1, p2, M);
    Span s = cylinder_span(along(0), first(0), second(0), along(6), first(6), second(6), a[9], a[11], pk, p1, p2, smax,
                           M);
    if (!(s.ao <= s.bo)) s = span_none();
    if (!(s.ai <= s.bi)) s.ai = INFINITY, s.bi = -INFINITY;
    s.ao = fmin(s.ao, fmin(u.ao, v.ao)), s.bo = fmax(s.bo, fmax(u.bo, v.bo));
    s.ai = fmin(s.ai, fmin(u.ai, v.ai)), s.bi = fmax(s.bi, fmax(u.bi, v.bi));
    return s;
}

// Bits [lo, hi] of a 64-bit mask (0 <= lo, hi <= 63; none if lo > hi).
MC3D_HD inline uint64_t bit_range(int lo, int hi) { return lo > hi ? 0 : (~0ull >> (63 - hi)) & (~0ull << lo); }

// The points s_i = i / scale, i in [0, last], of a span: `sure` those
// certainly in it, `maybe` those not certainly out of it.  The points' own
// deviation from i / scale, in units of i, is below eta.
MC3D_HD inline void row_mask(const Span &s, double scale, double eta, int last, uint64_t &sure, uint64_t &maybe) {
    const double o0 = s.ao * scale - eta, o1 = s.bo * scale + eta, i0 = s.ai * scale + eta, i1 = s.bi * scale - eta;
    // (comparisons false for a NaN: then everything may be in, nothing is sure)
    const int a = o0 > 0 ? (o0 <= last ? (int)ceil(o0) : 64) : 0;
    const int b = o1 < last ? (o1 >= 0 ? (int)o1 : -1) : last;
    const int c = i0 <= last ? (i0 > 0 ? (int)ceil(i0) : 0) : 64;
    const int d = i1 >= 0 ? (i1 < last ? (int)i1 : last) : -1;
    maybe = a <= 63 ? bit_range(a, b) : 0;
    sure = c <= 63 ? bit_range(c, d) & maybe : 0;
}

// The atom's mask over the points: sure ones, and those of the rest at
// which atom64 is true (point(i): the i-th point's coordinate along axis k).
// Only the points of `want` matter.
template <class F64P, class Point>
__device__ __forceinline__ uint64_t atom_mask(uint32_t kind, F64P a, int k, double x, double y, double z, double smax,
                                              double mag, double scale, double eta, int last, uint64_t want,
                                              Point &&point) {
    uint64_t sure, maybe;
    row_mask(atom_span(kind, a, k, x, y, z, smax, mag), scale, eta, last, sure, maybe);
    for (uint64_t open = maybe & ~sure & want; open; open &= open - 1) {
        const int i = __ffsll((unsigned long long)open) - 1;
        const double p = point(i);
        if (atom64(kind, a, k == 0 ? p : x, k == 1 ? p : y, k == 2 ? p : z)) sure |= 1ull << i;
    }
    return sure;
}

// One operator on masks: b is the top of the stack, a below it.
template <class M>
__device__ __forceinline__ M mask_op(uint32_t op, M a, M b) {
    if (op == OP_OR) return a | b;
    if (op == OP_AND) return a & b;
    if (op == OP_ANDNOT) return a & ~b;
    return ~a & b;  // OP_RANDNOT
}

// A program over such atoms as a mask over the points of a line; the stack
// below its top lies in LDS (slot i of this lane: stack[i * stride]).
template <bool UNI, class M, class CodeP, class F64P, class Point>
__device__ __forceinline__ M row_program(CodeP code, uint32_t n, F64P f64, int k, double x, double y, double z,
                                         double smax, double mag, double scale, double eta, int last, M want,
                                         M *stack, int stride, Point &&point) {
    M top = 0;
    int sp = 0;
    for (uint32_t pc = 0; pc < n; ++pc) {
        Insn in{code[pc].x, code[pc].y};
        if (UNI) in.x = (uint32_t)__builtin_amdgcn_readfirstlane((int)in.x);
        if (UNI) in.y = (uint32_t)__builtin_amdgcn_readfirstlane((int)in.y);
        const uint32_t op = insn_op(in.x);
        if (op == OP_ATOM || op == OP_TRUE || op == OP_FALSE) {
            if (sp > 0) stack[(sp - 1) * stride] = top;
            sp++;
            top = op == OP_ATOM ? (M)atom_mask(insn_kind(in.x), f64 + in.y, k, x, y, z, smax, mag, scale, eta, last,
                                               (uint64_t)want, point)
                                : (op == OP_TRUE ? ~(M)0 : (M)0);
        } else if (op == OP_NOT) {
            top = ~top;
        } else {
            sp--;
            top = mask_op<M>(op, stack[(sp - 1) * stride], top);
        }
    }
    return top;
}

}  // namespace mc3d
