// rows.h -- Solid.Contains along an axis-parallel line: where an atom is
// true on it, as an interval, so that one lane decides a whole row of
// corners (or all midpoints of an edge) instead of one point.
//
// A sphere, box, capsule or cylinder is convex, so the points of a line that
// lie in it are one interval.  atom_span bounds that interval from outside
// and from inside by more than the rounding of the reference's float64
// expressions (atom64) and of the computation here: a point past the outer
// bounds is false, a point within the inner bounds is true, and the points
// between the two, mostly few, are decided by atom64 itself.  A program over such
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

// 1 / x to the last digit or two (the bounds it goes into carry far more).
MC3D_HD inline double recip(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(x);
    y = __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
#else
    return 1 / x;
#endif
}

// ro >= sqrt(w') >= ri for every w' in [w - D, w + D] (w >= -D), with 1e-10 of
// itself more on each side; ri < 0: w' may be below zero.  (All in float64: D goes
// down to 1e-219 over the lengths that span_range admits.)
MC3D_HD inline void span_root(double w, double D, double &ro, double &ri) {
    if (w <= 4 * D) {  // the line grazes the surface
        ro = 5 * D * rsq_estimate(5 * D) * 1.001;
        ri = -1;
        return;
    }
    const double y = rsq_estimate(w);
    double r = w * y;
    r = r + 0.5 * y * __builtin_fma(-r, r, w);
    const double e = 1.1 * D * y + 1e-10 * r;
    ro = r + e;
    ri = r - e;
}

// Lengths that are neither so large nor so small that a square or a product of
// two leaves the float64 range.
MC3D_HD inline bool span_range(double M) { return M > 1e-100 && M < 1e100; }

// The axis of a line: known when the code is compiled (KX: the x axis), or
// a lane's own, then as the unit vector e_k, so that picking or leaving out a
// component is three multiply-adds instead of selects of scalar operands.
template <bool KX>
struct LineAxis {
    int k = 0;
    double v[3] = {1, 0, 0};
    MC3D_HD explicit LineAxis(int axis) : k(axis) {
        for (int a = 0; a < 3; a++) v[a] = a == axis ? 1.0 : 0.0;
    }
    MC3D_HD double along(double x, double y, double z) const {
        if (KX) return x;
        return __builtin_fma(z, v[2], __builtin_fma(y, v[1], x * v[0]));
    }
    MC3D_HD double across2(double x, double y, double z) const {  // the other components' squares
        if (KX) return __builtin_fma(z, z, y * y);
        const double a = __builtin_fma(-x, v[0], x), b = __builtin_fma(-y, v[1], y), c = __builtin_fma(-z, v[2], z);
        return __builtin_fma(c, c, __builtin_fma(b, b, a * a));
    }
};

// A vector's square, its component along the line's axis and the square of the
// rest, which rounding moves by a few half ulps of the whole square.
struct LineVec {
    double vv, along, across2;
};
template <bool KX>
MC3D_HD inline LineVec line_vec(const LineAxis<KX> &ax, double x, double y, double z) {
    LineVec r;
    r.along = ax.along(x, y, z);
    if (KX) {
        r.across2 = __builtin_fma(z, z, y * y);
        r.vv = __builtin_fma(x, x, r.across2);
    } else {
        r.vv = __builtin_fma(z, z, __builtin_fma(y, y, x * x));
        r.across2 = __builtin_fma(-r.along, r.along, r.vv);
    }
    return r;
}

// Sphere with threshold T (s <= T) whose centre is p - d, its squared distance s
// known to D.
MC3D_HD inline Span sphere_span(const LineVec &d, double T, double D) {
    const double w = T - d.across2, m = -d.along;
    if (w < -D) return span_none();
    double ro, ri;
    span_root(w, D, ro, ri);
    Span s{m - ro, m + ro, INFINITY, -INFINITY};
    if (ri > 0) s.ai = m - ri, s.bi = m + ri;
    return s;
}

// Cylinder from p - v along the unit vector d, length L, threshold T: with
// c = v.d and n = v - c d, the squared distance from its axis is |n|^2 +
// 2 s n_k + s^2 (1 - d_k^2), the position along it c + s d_k.  smax: the
// largest |s| asked about (nearly parallel lines, where the roots or the end
// planes are ill-defined, are bounded over that range instead).  M bounds the
// lengths it is made of, D the rounding of the squared distance.
template <bool KX>
MC3D_HD inline Span cylinder_span(const LineAxis<KX> &ax, const LineVec &v, double c, double dx, double dy, double dz, double L,
                                  double T, double smax, double M, double D) {
    const double dk = ax.along(dx, dy, dz), A = ax.across2(dx, dy, dz);
    const double nk = __builtin_fma(-c, dk, v.along), w = T - __builtin_fma(-c, c, v.vv);
    Span s;
    if (A < 1e-6) {  // along the axis: the distance hardly changes
        const double D2 = D + 2 * fabs(nk) * smax + A * smax * smax;
        if (w < -D2) return span_none();
        s = w > D2 ? span_all() : span_unsure();
    } else {
        // (n_k, at most |n| sqrt(A), carries a rounding of M: more than A D of
        // its square where the line is nearly parallel)
        const double disc = __builtin_fma(A, w, nk * nk);
        const double DD = __builtin_fma(fabs(nk), __builtin_fma(1e-14, fabs(nk), 4e-15 * M), A * D);
        if (disc < -DD) return span_none();
        double ro, ri;
        span_root(disc, DD, ro, ri);
        const double iA = recip(A), e = (1e-12 * (fabs(nk) + ro) + 1e-14 * M) * iA;
        s = Span{(-nk - ro) * iA - e, (-nk + ro) * iA + e, INFINITY, -INFINITY};
        if (ri > 0) s.ai = (-nk - ri) * iA + e, s.bi = (-nk + ri) * iA - e;
    }
    const double f = 1e-13 * M;  // rounding of the position along the axis
    if (dk == 0) {
        // Across the axis every point has this same sum, bit for bit (its k
        // term is a zero).  End faces mostly lie in planes of the grid, where
        // a margin would leave whole rows and edges open.
        if (c < 0 || c > L) return span_none();
    } else if (fabs(dk) < 1e-7) {
        const double f2 = f + fabs(dk) * smax;
        if (c < -f2 || c > L + f2) return span_none();
        if (!(c > f2 && c < L - f2)) s.ai = INFINITY, s.bi = -INFINITY;
    } else {
        const double i = recip(dk);
        const double t0 = (-f - c) * i, t1 = (L + f - c) * i, u0 = (f - c) * i, u1 = (L - f - c) * i;
        s.ao = fmax(s.ao, fmin(t0, t1)), s.bo = fmin(s.bo, fmax(t0, t1));
        s.ai = fmax(s.ai, dk > 0 ? u0 : u1), s.bi = fmin(s.bi, dk > 0 ? u1 : u0);
    }
    return s;
}

// Where an untransformed sphere, box, capsule or cylinder (params a, the
// layouts of AtomKind) is true on the line through (x, y, z) along the axis.
// mag: a bound of |x|, |y|, |z| and of the coordinates asked about.
template <bool KX, class F64P>
MC3D_HD inline Span atom_span(uint32_t kind, F64P a, const LineAxis<KX> &ax, double x, double y, double z, double smax,
                              double mag) {
    if (kind == A_RECT) {  // exact comparisons off the line's axis
        const int k = KX ? 0 : ax.k;
        const bool in = (int)(k == 0 || ((int)in_lo(x, a[0]) & (int)in_hi(x, a[3]))) &
                        (int)(k == 1 || ((int)in_lo(y, a[1]) & (int)in_hi(y, a[4]))) &
                        (int)(k == 2 || ((int)in_lo(z, a[2]) & (int)in_hi(z, a[5])));
        if (!in) return span_none();
        const double p = sel3(k, x, y, z), a0 = sel3(k, a[0], a[1], a[2]), a1 = sel3(k, a[3], a[4], a[5]);
        const double lo = a0 - p, hi = a1 - p;
        // (rounding of the differences; an infinite face has none)
        const double el = fabs(lo) < INFINITY ? 1e-15 * (mag + fabs(a0)) : 0;
        const double eh = fabs(hi) < INFINITY ? 1e-15 * (mag + fabs(a1)) : 0;
        return Span{lo - el, hi + eh, lo + el, hi - eh};
    }
    // Rounding is bounded by the lengths that are computed with, not by the
    // coordinates (a solid far from the origin has the same differences, each
    // rounded once): the squared distance moves by far less than 1e-13 of the
    // square of their sum, 3e-13 of the sum of three squares.
    const double vx = x - a[0], vy = y - a[1], vz = z - a[2];
    const LineVec v = line_vec(ax, vx, vy, vz);
    if (kind == A_SPHERE) {
        const double q = v.vv + __builtin_fma(smax, smax, a[4]);
        if (!(q > 1e-200 && q < 1e200)) return span_unsure();
        return sphere_span(v, a[4], 3e-13 * q);
    }
    // Contains of the other two takes the difference from the axis's nearest
    // point, rounded as a coordinate (at most G): 7 half ulps of G, at a distance
    // of up to M, move the square by less than 1e-15 M G.
    const bool cyl = kind == A_CYLINDER;
    const double L = cyl ? a[6] : a[9], M = fabs(vx) + fabs(vy) + fabs(vz) + smax + L + (cyl ? a[7] : a[10]), G = mag + M;
    const double D = __builtin_fma(1e-30 * G, G, M * __builtin_fma(1e-13, M, 4e-15 * G));
    const int dir = cyl ? 3 : 6;
    if (!(span_range(M) && G < 1e100 && fabs(a[dir]) + fabs(a[dir + 1]) + fabs(a[dir + 2]) < 2)) return span_unsure();
    const double T = cyl ? a[8] : a[11];
    const double c = vx * a[dir] + vy * a[dir + 1] + vz * a[dir + 2];  // (atom64's own sum)
    Span s = cylinder_span(ax, v, c, a[dir], a[dir + 1], a[dir + 2], L, T, smax, M, D);
    if (cyl) return s;
    // capsule: the cylinder between two spheres; it is convex, so the hull
    // of their intervals (and of the certain parts of those, each by the margin
    // of the points between the ends) is its own
    const Span u = sphere_span(v, T, D), e = sphere_span(line_vec(ax, x - a[3], y - a[4], z - a[5]), T, D);
    if (!(s.ao <= s.bo)) s = span_none();
    if (!(s.ai <= s.bi)) s.ai = INFINITY, s.bi = -INFINITY;
    s.ao = fmin(s.ao, fmin(u.ao, e.ao)), s.bo = fmax(s.bo, fmax(u.bo, e.bo));
    s.ai = fmin(s.ai, fmin(u.ai, e.ai)), s.bi = fmax(s.bi, fmax(u.bi, e.bi));
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

// How far the points of a row (64 additions of h, each rounded) and of a bracket
// (halvings, scale steps a unit) stray from even spacing, in steps.
MC3D_HD inline double row_eta(double mag, double inv_h) { return 1e-6 + 1e-11 * mag * inv_h; }
MC3D_HD inline double bracket_eta(double mag, double scale) { return 1e-6 + 1e-15 * mag * scale; }

// Bounds of a ray's interval are of use for points that stray less than this.
constexpr double RAY_ETA = 0.01;

// The point i / 2^levels of the bracket [a, b], as halvings reach it.
MC3D_HD inline double bracket_point(double a, double b, int levels, int i) {
    double m = a;
    for (int bit = 1 << (levels - 1), at = 0; bit; bit >>= 1) {
        m = (a + b) / 2;
        if (at + bit == i) break;
        if (i > at + bit) a = m, at += bit;
        else b = m;
    }
    return m;
}

// Open points that a lane evaluates one after another; a line with more of them
// (one that touches the surface all along, or whose bounds are no finer than its
// points) is decided otherwise.
constexpr int FEW_OPEN = 4;

// The atom's mask over the points: the sure ones, and those of the rest that
// rest(kind, a, open) finds inside.  Only the points of `want` matter.
template <bool KX, class F64P, class Rest>
__device__ __forceinline__ uint64_t atom_mask(uint32_t kind, F64P a, const LineAxis<KX> &ax, double x, double y, double z, double smax,
                                              double mag, double scale, double eta, int last, uint64_t want,
                                              Rest &&rest) {
    uint64_t sure, maybe;
    row_mask(atom_span(kind, a, ax, x, y, z, smax, mag), scale, eta, last, sure, maybe);
    return sure | rest(kind, a, maybe & ~sure & want);
}

// The open points at which atom64 is true, one after another (point(i): the
// i-th point's coordinate along the line's axis).
template <bool KX, class F64P, class Point>
__device__ __forceinline__ uint64_t open_points(uint32_t kind, F64P a, const LineAxis<KX> &ax, double x, double y, double z,
                                                uint64_t open, Point &&point) {
    uint64_t in = 0;
    for (; open; open &= open - 1) {
        const int i = __ffsll((unsigned long long)open) - 1;
        const int k = KX ? 0 : ax.k;
        const double p = point(i);
        if (atom64(kind, a, k == 0 ? p : x, k == 1 ? p : y, k == 2 ? p : z)) in |= 1ull << i;
    }
    return in;
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
template <bool UNI, class M, bool KX, class CodeP, class F64P, class Rest>
__device__ __forceinline__ M row_program(CodeP code, uint32_t n, F64P f64, const LineAxis<KX> &ax, double x, double y, double z,
                                         double smax, double mag, double scale, double eta, int last, M want,
                                         M *stack, int stride, Rest &&rest) {
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
            top = op == OP_ATOM ? (M)atom_mask(insn_kind(in.x), f64 + in.y, ax, x, y, z, smax, mag, scale, eta, last,
                                               (uint64_t)want, rest)
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
