// k_rays.hip -- a mesh collider's containment a row of corners at a time.
//
// ColliderContains (model3d/collisions.go:119-134) counts the triangles that
// a point's ray hits, all rays along one direction D.  Along a row of corners
// (a line in x) the conditions of Triangle.rayCollision (primitives.go:
// 207-249) are linear, so the corners whose ray hits one triangle are an
// interval of the row: it is bounded from outside and from inside by more than
// the rounding of the reference's expressions and of the ones here, and
// toggles the parity at its two ends.  The corners between the two bounds are
// decided by collider_contains itself, so every decision is the one it makes.
//
// The triangles that a row's rays can hit cross the plane of the row and D;
// the planes of all rows are parallel, so the triangles are binned by their
// extents across them.  A wave takes up to RAY_ROWS rows along z, whose planes
// lie within a bin's width of each other (every triangle is binned that much
// further), and a lane a triangle for all of them.  Looked up point by point,
// every triangle of a cell was 104 bytes read for each point, and the kernel
// waited for them; this one is bound by issue (286 vector and 137 scalar
// instructions for 64 triangles of 4 rows).  Measured (kernel trace, MI355X, a
// mesh made at spacing 0.02): 256^3 corners 993 -> 215 us, their vertices'
// bisection (8 halvings) 448 -> 192 us; the whole call at 40^3 corners 462 ->
// 180 us; the corners of a mesh with faces in the grid's planes, 1,410 -> 262 us
// (838 with a lane looking up all the undecided corners of its 32).
#include "launch.h"
#include "rows.h"

#include "kernels.h"

namespace mc3d {
namespace {

__device__ constexpr double RAY_D[3] = {0.5224892708603626, 0.10494477243214506, 0.43558938446126527};

constexpr double RAY_EPS = 64 * 0x1.0p-53;

// The linear forms of one kept triangle (ray_grid's record): bary1, bary2 and
// scale as a . p + c, with what |p| + |t0| has to be multiplied by for a bound
// of their errors: at most 14 roundings of the sums of the terms' magnitudes
// in the reference's order and here, 64 taken.  Its extent across the rows'
// planes, widened as its box in the ray grid is.
__global__ __launch_bounds__(256) void k_ray_forms(const double *__restrict__ rec, uint32_t n, RayPlanes R,
                                                   double *__restrict__ forms, double2 *__restrict__ extent,
                                                   uint32_t *__restrict__ bad) {
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const double *r = rec + (size_t)RAY_REC * i;
        const double *t0 = r, *c1 = r + 3, *v1 = r + 7, *v2 = r + 10, inv = r[6];
        double f[RAY_FORM];
        // D . (o x v1) = o . (v1 x D), v2 . (o x v1) = o . (v1 x v2)
        double m2[3], m3[3];
        for (int k = 0; k < 3; k++) {
            const int a = (k + 1) % 3, b = (k + 2) % 3;
            m2[k] = v1[a] * RAY_D[b] - v1[b] * RAY_D[a];
            m3[k] = v1[a] * v2[b] - v1[b] * v2[a];
        }
        f[9] = f[10] = f[11] = 0;
        for (int k = 0; k < 3; k++) {
            f[3 * k] = inv * c1[k], f[3 * k + 1] = inv * m2[k], f[3 * k + 2] = inv * m3[k];
            for (int q = 0; q < 3; q++) f[9 + q] -= f[3 * k + q] * t0[k];
        }
        const double one = fabs(c1[0]) + fabs(c1[1]) + fabs(c1[2]);
        const double v1m = fmax(fabs(v1[0]), fmax(fabs(v1[1]), fabs(v1[2])));
        const double v2s = fabs(v2[0]) + fabs(v2[1]) + fabs(v2[2]);
        const double ds = RAY_D[0] + RAY_D[1] + RAY_D[2];
        f[12] = RAY_EPS * fabs(inv) * one;
        f[13] = RAY_EPS * fabs(inv) * 2 * ds * v1m;
        f[14] = RAY_EPS * fabs(inv) * 2 * v2s * v1m;
        f[15] = 0;
        // |n . D| of the unit normal: grazing triangles lose digits
        const double nn = sqrt(m3[0] * m3[0] + m3[1] * m3[1] + m3[2] * m3[2]);
        const double dd = 1 / (fabs(inv) * nn);
        double lo = INFINITY, hi = -INFINITY, size = 0, mag = 0;
        for (int v = 0; v < 3; v++) {
            double p[3];
            for (int k = 0; k < 3; k++) {
                p[k] = t0[k] + (v == 1 ? v1[k] : v == 2 ? v2[k] : 0.0);
                mag = fmax(mag, fabs(p[k]));
                size = fmax(size, fmax(fabs(v1[k]), fmax(fabs(v2[k]), fabs(v2[k] - v1[k]))));
            }
            const double s = R.ny * p[1] + R.nz * p[2];
            lo = fmin(lo, s), hi = fmax(hi, s);
        }
        const double w = 2 * size * fmax(1e-6, 1e-13 / dd) + 2e-9 * mag + 1e-300;
        extent[i] = make_double2(lo - w, hi + w);
        // (far from overflow, or the collider keeps to point lookups)
        bool fine = fabs(lo) + fabs(hi) + w < 1e100;
        for (int k = 0; k < RAY_FORM; k++) fine = fine && fabs(f[k]) < 1e100, forms[(size_t)RAY_FORM * i + k] = f[k];
        if (!fine) atomicOr(bad, 1u);
    }
}

__device__ __forceinline__ int plane_bin(const RayPlanes &R, double s) {
    return (int)fmin((double)(R.bins - 1), fmax(0.0, floor((s - R.s0) * R.inv)));
}

// Entries of every bin (at[b]); then, with at the fill's cursors, the lists, in
// any order: the parity does not depend on it.  A block counts its triangles'
// entries in LDS and takes its places with one atomic a bin.
__global__ __launch_bounds__(1024) void k_ray_bins(const double2 *__restrict__ extent, uint32_t n, RayPlanes R,
                                                   uint32_t *__restrict__ at, uint32_t *__restrict__ list) {
    __shared__ uint32_t cnt[RAY_BINS];
    for (int b = threadIdx.x; b < R.bins; b += 1024) cnt[b] = 0;
    __syncthreads();
    const uint32_t i = blockIdx.x * 1024 + threadIdx.x;
    int b0 = 0, b1 = -1;
    if (i < n) {
        const double2 e = extent[i];
        b0 = plane_bin(R, e.x - R.width), b1 = plane_bin(R, e.y);
    }
    for (int b = b0; b <= b1; b++) atomicAdd(&cnt[b], 1u);
    __syncthreads();
    for (int b = threadIdx.x; b < R.bins; b += 1024)
        if (cnt[b]) cnt[b] = atomicAdd(&at[b], cnt[b]);
    if (!list) return;
    __syncthreads();
    for (int b = b0; b <= b1; b++) list[atomicAdd(&cnt[b], 1u)] = i;
}

// start[0, bins] and the fill's cursors from the bins' entries (one block).
__global__ __launch_bounds__(1024) void k_ray_scan(uint32_t *__restrict__ at, uint32_t bins, uint32_t *__restrict__ start,
                                                   unsigned long long *__restrict__ total) {
    __shared__ unsigned long long sh[1024];
    unsigned long long carry = 0;
    for (uint32_t b0 = 0; b0 < bins; b0 += 1024) {
        const uint32_t b = b0 + threadIdx.x, v = b < bins ? at[b] : 0u;
        __syncthreads();
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int d = 1; d < 1024; d <<= 1) {
            const unsigned long long t = (int)threadIdx.x >= d ? sh[threadIdx.x - d] : 0;
            __syncthreads();
            sh[threadIdx.x] += t;
            __syncthreads();
        }
        if (b < bins) at[b] = start[b] = (uint32_t)(carry + sh[threadIdx.x] - v);
        carry += sh[1023];
    }
    if (threadIdx.x == 0) start[bins] = (uint32_t)carry, *total = carry;
}

// Where A t + B(z) >= 0 along the rows of a wave (t: steps of a row's corners),
// B linear in z and everything known to e: t at least lo + lo_z z (A > 0) or at
// most hi + hi_z z (A < 0), give or take w.  A so small that w could reach over
// the row is flat: B alone decides.
struct RayBound {
    double lo, lo_z, hi, hi_z, w;
};
__device__ __forceinline__ bool ray_flat(double A, double e, double nx) { return !(fabs(A) * nx > 1e3 * e); }
__device__ __forceinline__ RayBound ray_bound(double A, double B, double slope, double e, bool flat) {
    const double q = recip(A), at = -B * q, z = -slope * q;
    const bool up = A > 0 && !flat, down = !up && !flat;
    return RayBound{up ? at : -1e9, up ? z : 0, down ? at : 1e9, down ? z : 0, flat ? 0 : e * fabs(q)};
}
// Corners that may be in ([p0, p1]) and that are ([s0, s1]).
struct RayRange {
    int p0, p1, s0, s1;
};
__device__ __forceinline__ RayRange ray_range(double lo, double hi, double w, int nx) {
    RayRange r;
    r.p0 = max((int)ceil(lo - w), 0), r.s0 = max((int)ceil(lo + w), 0);
    r.p1 = min((int)floor(hi + w), nx - 1), r.s1 = min((int)floor(hi - w), nx - 1);
    return r;
}

// bits [a, b] of the 32 from bit 32 w on
__device__ __forceinline__ uint32_t bit_range(int a, int b, int w) {
    const int lo = max(a - 32 * w, 0), hi = min(b - 32 * w, 31);
    return lo > hi ? 0u : (~0u >> (31 - hi)) & (~0u << lo);
}

// The occupancy words of a solid that is one collider without an inset: a wave
// per (1 << shift) rows along z by 1024 corners along x.
constexpr int RAY_SPAN = 1024;
__global__ __launch_bounds__(64) void k_ray_rows(const Seg sg, uint64_t *__restrict__ bits, Ctl *__restrict__ ctl,
                                                  SegOut *__restrict__ sout, int rows, uint64_t nunits) {
    __shared__ uint32_t ev[RAY_ROWS][RAY_SPAN / 32 + 1], open[RAY_ROWS][RAY_SPAN / 32];
    const int lane = threadIdx.x;
    const Grid &g = sg.g;
    const auto a = scalar_ptr(sg.P.f64) + scalar_ptr(sg.P.code)[0].y;
    const DevCollider &C = sg.P.colliders[(int)a[0]];
    const RayPlanes R = C.planes;
    const double *const forms = global_ptr(C.forms);
    const uint32_t *const pstart = global_ptr(C.pstart), *const plist = global_ptr(C.plist);
    const RowScale rs = row_scale(g);
    const uint32_t nchunk = (uint32_t)(g.nx + RAY_SPAN - 1) / RAY_SPAN;
    for (uint64_t u = blockIdx.x; u < nunits; u += gridDim.x) {
        const uint32_t c = (uint32_t)(u % nchunk), row = (uint32_t)(u / nchunk);
        const int y = (int)(row % (uint32_t)g.ny), z0 = (int)(row / (uint32_t)g.ny) * rows;
        const int x0 = (int)c * RAY_SPAN, nx = min(RAY_SPAN, g.nx - x0), nr = min(rows, g.nz - z0);
        const double py = g.ys[y];
        wave_sync();
        for (int i = lane; i < RAY_ROWS * (RAY_SPAN / 32 + 1); i += 64) (&ev[0][0])[i] = 0;
        for (int i = lane; i < RAY_ROWS * (RAY_SPAN / 32); i += 64) (&open[0][0])[i] = 0;
        wave_sync();
        double pz[RAY_ROWS];
        bool any = false;
        for (int r = 0; r < RAY_ROWS; r++) {
            pz[r] = g.zs[min(z0 + r, g.nz - 1)];
            any = any || (r < nr && in_lo(pz[r], a[3]) && in_hi(pz[r], a[6]));
        }
        any = any && in_lo(py, a[2]) && in_hi(py, a[5]);
        if (any) {
            // the rows' planes: from the least on, no more than a bin's width
            const double sa = R.ny * py + R.nz * pz[0], sb = R.ny * py + R.nz * g.zs[z0 + nr - 1];
            const int bin = plane_bin(R, fmin(sa, sb));
            const double px = g.xs[x0], em = rs.mag + C.mag;
            const uint32_t e = pstart[bin + 1], first = pstart[bin];
            double2 f[RAY_FORM / 2];
            auto entry = [&](uint32_t i) { return plist[i < e ? i : first]; };
            auto fetch = [&](uint32_t t) {
                const double2 *p = (const double2 *)(forms + (size_t)RAY_FORM * t);
                for (int k = 0; k < RAY_FORM / 2; k++) f[k] = p[k];
            };
            uint32_t t1 = 0;
            if (first < e) t1 = entry(first + lane);
            for (uint32_t i0 = first; i0 < e; i0 += 64) {
                const bool have = i0 + lane < e;
                fetch(t1);
                if (i0 + 64 < e) t1 = entry(i0 + 64 + lane);
                double q[RAY_FORM];
                for (int k = 0; k < RAY_FORM / 2; k++) q[2 * k] = f[k].x, q[2 * k + 1] = f[k].y;
                const double A1 = q[0] * rs.h, A2 = q[1] * rs.h, A3 = q[2] * rs.h;
                const double e1 = q[12] * em, e2 = q[13] * em, e3 = q[14] * em;
                const double c1 = q[0] * px + q[3] * py + q[9], c2 = q[1] * px + q[4] * py + q[10];
                const double c3 = q[2] * px + q[5] * py + q[11];
                const double A12 = -(A1 + A2), c12 = 1 - c1 - c2, q12 = -(q[6] + q[7]), e12 = e1 + e2 + 1e-15;
                // (edges along x: common in meshes of boxes and of grids)
                const bool f1 = ray_flat(A1, e1, nx), f2 = ray_flat(A2, e2, nx), f12 = ray_flat(A12, e12, nx), f3 = ray_flat(A3, e3, nx);
                const bool flat = __ballot(f1 || f2 || f12 || f3) != 0;
                const RayBound b1 = ray_bound(A1, c1, q[6], e1, f1), b2 = ray_bound(A2, c2, q[7], e2, f2);
                const RayBound b12 = ray_bound(A12, c12, q12, e12, f12), b3 = ray_bound(A3, c3, q[8], e3, f3);
                const double w = fmax(fmax(b1.w, b2.w), fmax(b12.w, b3.w)) + rs.eta;
                for (int r = 0; r < RAY_ROWS; r++) {
                    if (r >= nr) break;
                    const double z = pz[r];
                    const double lo = fmax(fmax(__builtin_fma(b1.lo_z, z, b1.lo), __builtin_fma(b2.lo_z, z, b2.lo)),
                                           fmax(__builtin_fma(b12.lo_z, z, b12.lo), __builtin_fma(b3.lo_z, z, b3.lo)));
                    const double hi = fmin(fmin(__builtin_fma(b1.hi_z, z, b1.hi), __builtin_fma(b2.hi_z, z, b2.hi)),
                                           fmin(__builtin_fma(b12.hi_z, z, b12.hi), __builtin_fma(b3.hi_z, z, b3.hi)));
                    RayRange g4 = ray_range(lo, hi, w, nx);
                    if (flat) {
                        bool may = true, sure = true;
                        auto check = [&](bool f, double A, double B, double e) {
                            const double m = e + fabs(A) * nx;
                            may = may && !(f && B < -m), sure = sure && !(f && !(B >= m));
                        };
                        check(f1, A1, c1 + q[6] * z, e1);
                        check(f2, A2, c2 + q[7] * z, e2);
                        check(f12, A12, c12 + q12 * z, e12);
                        check(f3, A3, c3 + q[8] * z, e3);
                        if (!may) g4.p1 = -1;
                        if (!sure) g4.s1 = -1;
                    }
                    const int p0 = g4.p0, p1 = g4.p1, s0 = g4.s0, s1 = g4.s1;
                    if (!have || p0 > p1) continue;
                    if (s0 <= s1) {
                        atomicXor(&ev[r][s0 >> 5], 1u << (s0 & 31));
                        atomicXor(&ev[r][(s1 + 1) >> 5], 1u << ((s1 + 1) & 31));
                        if (s0 == p0 && s1 == p1) continue;
                    }
                    for (int w = p0 >> 5; w <= p1 >> 5; w++) {
                        const uint32_t m = bit_range(p0, p1, w) & ~(s0 <= s1 ? bit_range(s0, s1, w) : 0u);
                        if (m) atomicOr(&open[r][w], m);
                    }
                }
            }
        }
        wave_sync();
        const bool col = lane < (nx + 31) / 32;  // this lane's 32 corners
        for (int r = 0; r < nr; r++) {
            const double z = pz[r];
            const bool in_row = in_lo(py, a[2]) && in_lo(z, a[3]) && in_hi(py, a[5]) && in_hi(z, a[6]);
            uint32_t v = 0, inside = 0;
            if (in_row) {
                // the parity of the toggles up to each corner
                v = lane < RAY_SPAN / 32 ? ev[r][lane] : 0u;
                for (int d = 1; d < 32; d <<= 1) v ^= v << d;
                const uint64_t odd = __ballot(v >> 31);
                if (__popcll(odd & ((1ull << lane) - 1)) & 1) v = ~v;
                // the corners within the collider's bounds, and the undecided
                // ones of them looked up, a lane a corner (a row in the plane
                // of a mesh face has them all the way along)
                uint32_t undecided = 0, found = 0;
                for (int w = 0; w < (nx + 63) / 64; w++) {
                    const int x = x0 + 64 * w + lane;
                    const double X = g.xs[min(x, g.nx - 1)];
                    const bool in = x < g.nx && in_lo(X, a[1]) && in_hi(X, a[4]);
                    const bool ask = in && ((open[r][2 * w + (lane >> 5)] >> (lane & 31)) & 1u);
                    const uint64_t m = __ballot(in), q = __ballot(ask);
                    uint64_t hit = 0;
                    if (q) hit = __ballot(ask && collider_contains(C, (const double *)(sg.P.f64 + sg.P.code[0].y), X, py, z));
                    if (lane >> 1 == w) {
                        const int half = 32 * (lane & 1);
                        inside = (uint32_t)(m >> half), undecided = (uint32_t)(q >> half), found = (uint32_t)(hit >> half);
                    }
                }
                v = (v & ~undecided) | found;
                v &= inside;
            }
            // (a word's two halves: an odd last half is written by the lane after it)
            if (lane < 2 * ((nx + 63) / 64)) ((uint32_t *)(bits + sg.word0 + word_index(g, x0 >> 6, y, z0 + r)))[lane] = col ? v : 0u;
            // panic("solid is true outside of bounds"), mc.go:687-689
            uint32_t face = 0;
            if (y == 0 || y == g.ny - 1 || z_face(g, z0 + r)) face = ~0u;
            if (x0 == 0 && lane == 0) face |= 1u;
            if ((g.nx - 1 - x0) >> 5 == lane) face |= 1u << ((g.nx - 1 - x0) & 31);
            if (col && (v & face)) atomicOr(&ctl->inside, 1u), atomicOr(&sout->inside, 1u);
        }
    }
}

// The points (of n, `step` apart along axis k from p on) whose ray hits a
// triangle, bound by bound.
__device__ __forceinline__ RayRange ray_points(const double *q, int k, const double *p, double step, double em, double eta,
                                               int n) {
    double lo = -1e9, hi = 1e9, w = eta;
    bool may = true, sure = true;
    auto bound = [&](double A, double B, double e) {
        if (ray_flat(A, e, n)) {
            const double m = e + fabs(A) * n;
            may = may && !(B < -m), sure = sure && B >= m;
        } else {
            const double i = recip(A), t = -B * i;
            if (A > 0) lo = fmax(lo, t);
            else hi = fmin(hi, t);
            w = fmax(w, e * fabs(i) + eta);
        }
    };
    const double A1 = sel3(k, q[0], q[3], q[6]) * step, A2 = sel3(k, q[1], q[4], q[7]) * step;
    const double A3 = sel3(k, q[2], q[5], q[8]) * step;
    const double B1 = q[0] * p[0] + q[3] * p[1] + q[6] * p[2] + q[9], B2 = q[1] * p[0] + q[4] * p[1] + q[7] * p[2] + q[10];
    const double B3 = q[2] * p[0] + q[5] * p[1] + q[8] * p[2] + q[11];
    const double e1 = q[12] * em, e2 = q[13] * em;
    bound(A1, B1, e1);
    bound(A2, B2, e2);
    bound(-(A1 + A2), 1 - B1 - B2, e1 + e2 + 1e-15);
    bound(A3, B3, q[14] * em);
    RayRange r = ray_range(lo, hi, w, n);
    if (!may) r.p1 = -1;
    if (!sure) r.s1 = -1;
    return r;
}

__device__ __forceinline__ uint64_t bit_range64(int a, int b) { return a > b ? 0 : (~0ull >> (63 - b)) & (~0ull << a); }

// mcSearchPoint (mc.go:223-258) of a collider's vertices: up to six halvings of
// an edge at a time from the parity at all the points that they can reach,
// RAY_LANES lanes a vertex and a triangle each.  The points are taken cell by
// cell of the ray grid.  Evaluating every halving was a chain of lookups, each a
// chain of loads over a cell's triangles.
//
// REST: the call halves on past the points' own rounding, where every halving is
// a lookup.  Those are left to k_bisect_rest, a lane a vertex, since all RAY_LANES
// of a vertex looked up the same point (a mesh made at spacing 0.05 on a grid of
// 0.0075, 60 halvings, device time: by points 3.2 ms, so 4.2, now 2.3): a vertex's
// place in the output holds its bracket and the halvings left.
constexpr int RAY_LANES = 8;
template <bool REST>
__global__ __launch_bounds__(256) void k_bisect_rays(const Seg sg, const uint64_t *__restrict__ bits_all,
                                                     const uint64_t *__restrict__ vkeys, double *__restrict__ verts,
                                                     double *__restrict__ interior, const Ctl *__restrict__ ctl,
                                                     uint64_t vcap) {
    const Grid &g = sg.g;
    const auto a = scalar_ptr(sg.P.f64) + scalar_ptr(sg.P.code)[0].y;
    const DevCollider &C = sg.P.colliders[(int)a[0]];
    const double *const forms = global_ptr(C.forms);
    const uint32_t *const cs = global_ptr(C.cell_start), *const ct = global_ptr(C.cell_tris);
    const double mag = row_scale(g).mag, em = mag + C.mag;
    const uint64_t *bits = bits_all + sg.word0;
    const uint32_t sub = threadIdx.x % RAY_LANES;
    const uint64_t nv = min((uint64_t)ctl->totals[0], vcap);
    const uint64_t per_grid = (uint64_t)gridDim.x * (256 / RAY_LANES);
    for (uint64_t v = (uint64_t)blockIdx.x * (256 / RAY_LANES) + threadIdx.x / RAY_LANES; v < nv; v += per_grid) {
        const uint64_t key = vkeys[v];
        const int k = (int)(key & 3);
        const int x = (int)((key >> 2) & 0xfffff), y = (int)((key >> 22) & 0xfffff), z = (int)((key >> 42) & 0xfffff);
        const double px = g.xs[x], py = g.ys[y], pz = g.zs[z];
        double lo = sel3(k, px, py, pz), hi = *(k == 0 ? g.xs + x + 1 : (k == 1 ? g.ys + y + 1 : g.zs + z + 1));
        const bool up = corner_bit(g, bits, x + (k == 0), y + (k == 1), z + (k == 2));
        int left = sg.iters;
        while (left > 0) {
            const int levels = min(left, 6), n = 1 << levels;
            const double step = (hi - lo) / n, eta = bracket_eta(mag, recip(step));
            if (REST && !(eta < RAY_ETA)) break;
            left -= levels;
            const double p[3] = {k == 0 ? lo : px, k == 1 ? lo : py, k == 2 ? lo : pz};
            uint64_t m = 0, open = 0;
            if (eta < RAY_ETA) {
                const double fu = (p[0] * C.u[0] + p[1] * C.u[1] + p[2] * C.u[2] - C.u0) * C.inv_cell;
                const double fv = (p[0] * C.v[0] + p[1] * C.v[1] + p[2] * C.v[2] - C.v0) * C.inv_cell;
                const double du = sel3(k, C.u[0], C.u[1], C.u[2]) * step * C.inv_cell;
                const double dv = sel3(k, C.v[0], C.v[1], C.v[2]) * step * C.inv_cell;
                // points so near a border that the lookup's rounding could put
                // them on its other side
                const double eu = 1e-6 + 1e-14 * (3 * mag + fabs(C.u0)) * C.inv_cell * recip(fabs(du));
                const double ev = 1e-6 + 1e-14 * (3 * mag + fabs(C.v0)) * C.inv_cell * recip(fabs(dv));
                auto border = [&](double t, double e) {
                    const int b0 = max((int)ceil(t - e), 1), b1 = min((int)floor(t + e), n - 1);
                    if (b0 <= b1) open |= bit_range64(b0, b1);
                };
                for (int i = 1; i < n;) {
                    const double cu = floor(fu + i * du), cv = floor(fv + i * dv);
                    // the last point before the cell's border
                    double tu = 64, tv = 64;
                    if (du != 0) {
                        const double t0 = (cu - fu) / du, t1 = (cu + 1 - fu) / du;
                        border(t0, eu), border(t1, eu);
                        tu = fmax(t0, t1);
                    }
                    if (dv != 0) {
                        const double t0 = (cv - fv) / dv, t1 = (cv + 1 - fv) / dv;
                        border(t0, ev), border(t1, ev);
                        tv = fmax(t0, t1);
                    }
                    const int end = max(i, (int)fmin(n - 1.0, fmin(tu, tv)));
                    if (cu >= 0 && cu < C.nu && cv >= 0 && cv < C.nv) {
                        const uint64_t run = bit_range64(i, end);
                        const uint32_t cell = (uint32_t)cv * (uint32_t)C.nu + (uint32_t)cu, e = cs[cell + 1];
                        for (uint32_t c = cs[cell] + sub; c < e; c += RAY_LANES) {
                            const double2 *f = (const double2 *)(forms + (size_t)RAY_FORM * ct[c]);
                            double q[RAY_FORM];
                            for (int j = 0; j < RAY_FORM / 2; j++) q[2 * j] = f[j].x, q[2 * j + 1] = f[j].y;
                            const RayRange r = ray_points(q, k, p, step, em, eta, n);
                            if (r.p0 > r.p1) continue;
                            const uint64_t may = bit_range64(r.p0, r.p1), in = bit_range64(r.s0, r.s1);
                            m ^= in & run, open |= may & ~in & run;
                        }
                    }
                    i = end + 1;
                }
            } else {
                open = ~0ull;
            }
            for (int d = 1; d < RAY_LANES; d <<= 1) {
                m ^= __shfl_xor(m, d, RAY_LANES);
                open |= __shfl_xor(open, d, RAY_LANES);
            }
            for (int bit = n >> 1, at = 0; bit; bit >>= 1) {
                const double mid = (lo + hi) / 2;
                const double qx = k == 0 ? mid : px, qy = k == 1 ? mid : py, qz = k == 2 ? mid : pz;
                bool in = (m >> (at + bit)) & 1;
                if ((open >> (at + bit)) & 1) in = collider_contains(C, sg.P.f64 + sg.P.code[0].y, qx, qy, qz);
                in = in && in_lo(qx, a[1]) && in_lo(qy, a[2]) && in_lo(qz, a[3]) && in_hi(qx, a[4]) && in_hi(qy, a[5]) &&
                     in_hi(qz, a[6]);
                if (in == up) hi = mid;  // the inside end moves
                else lo = mid, at += bit;
            }
        }
        if (REST) {
            if (sub < 3) verts[3 * v + sub] = sub == 0 ? lo : sub == 1 ? hi : (double)left;
        } else if (sub < 3) {
            const double res = (lo + hi) / 2, in = up ? hi : lo;  // the bracket's inside end (mc.go:252-255)
            const double at = sub == 0 ? px : sub == 1 ? py : pz;
            verts[3 * v + sub] = (int)sub == k ? res : at;
            if (interior) interior[3 * v + sub] = (int)sub == k ? in : at;
        }
    }
}

// The halvings that k_bisect_rays<true> left.
__global__ __launch_bounds__(256) void k_bisect_rest(const Seg sg, const uint64_t *__restrict__ bits_all,
                                                     const uint64_t *__restrict__ vkeys, double *__restrict__ verts,
                                                     double *__restrict__ interior, const Ctl *__restrict__ ctl,
                                                     uint64_t vcap) {
    const Grid &g = sg.g;
    const double *a = sg.P.f64 + sg.P.code[0].y;
    const DevCollider &C = sg.P.colliders[(int)a[0]];
    const uint64_t *bits = bits_all + sg.word0;
    const uint64_t nv = min((uint64_t)ctl->totals[0], vcap);
    for (uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x; v < nv; v += (uint64_t)gridDim.x * 256) {
        const uint64_t key = vkeys[v];
        const int k = (int)(key & 3);
        const int x = (int)((key >> 2) & 0xfffff), y = (int)((key >> 22) & 0xfffff), z = (int)((key >> 42) & 0xfffff);
        const double px = g.xs[x], py = g.ys[y], pz = g.zs[z];
        const bool up = corner_bit(g, bits, x + (k == 0), y + (k == 1), z + (k == 2));
        double lo = verts[3 * v], hi = verts[3 * v + 1];
        for (int left = (int)verts[3 * v + 2]; left > 0; left--) {
            const double mid = (lo + hi) / 2;
            const bool in = collider_contains(C, a, k == 0 ? mid : px, k == 1 ? mid : py, k == 2 ? mid : pz);
            if (in == up) hi = mid;
            else lo = mid;
        }
        const double res = (lo + hi) / 2, in = up ? hi : lo;
        for (int c = 0; c < 3; c++) {
            const double at = sel3(c, px, py, pz);
            verts[3 * v + c] = c == k ? res : at;
            if (interior) interior[3 * v + c] = c == k ? in : at;
        }
    }
}

}  // namespace

hipError_t launch_bisect_rays(const Pipe &p, const Bufs &b, double *verts, double *interior, uint64_t vcap,
                              hipStream_t st) {
    const unsigned grid = grid_for(vcap, 256 / RAY_LANES, 1u << 14);
    if (!p.ray_rest) {
        k_bisect_rays<false><<<grid, 256, 0, st>>>(p.seg0, b.bits, b.vkeys, verts, interior, p.ctl, vcap);
    } else {
        k_bisect_rays<true><<<grid, 256, 0, st>>>(p.seg0, b.bits, b.vkeys, verts, interior, p.ctl, vcap);
        k_bisect_rest<<<grid_for(vcap, 256, 1u << 14), 256, 0, st>>>(p.seg0, b.bits, b.vkeys, verts, interior, p.ctl, vcap);
    }
    return hipGetLastError();
}

hipError_t launch_ray_forms(const double *rec, uint32_t n, const RayPlanes &R, double *forms, double *extent, uint32_t *at,
                            uint32_t *bad, hipStream_t st) {
    hipError_t e = launch_zero(at, ((size_t)R.bins * 4 + 15) / 16 * 16, st);
    if (e != hipSuccess) return e;
    if ((e = launch_zero(bad, 16, st)) != hipSuccess) return e;
    const unsigned grid = grid_for(n, 256, 4096);
    k_ray_forms<<<grid, 256, 0, st>>>(rec, n, R, forms, (double2 *)extent, bad);
    k_ray_bins<<<(n + 1023) / 1024, 1024, 0, st>>>((const double2 *)extent, n, R, at, nullptr);
    return hipGetLastError();
}

hipError_t launch_ray_scan(uint32_t *at, uint32_t bins, uint32_t *start, unsigned long long *total, hipStream_t st) {
    k_ray_scan<<<1, 1024, 0, st>>>(at, bins, start, total);
    return hipGetLastError();
}

hipError_t launch_ray_fill(const double *extent, uint32_t n, const RayPlanes &R, uint32_t *at, uint32_t *list,
                           hipStream_t st) {
    k_ray_bins<<<(n + 1023) / 1024, 1024, 0, st>>>((const double2 *)extent, n, R, at, list);
    return hipGetLastError();
}

hipError_t launch_ray_rows(const Pipe &p, const Bufs &b, hipStream_t st) {
    const Grid &g = p.seg0.g;
    const uint64_t nunits = (uint64_t)((g.nx + RAY_SPAN - 1) / RAY_SPAN) * g.ny * ((g.nz + p.ray_rows - 1) / p.ray_rows);
    k_ray_rows<<<grid_for(nunits, 1, 1u << 18), 64, 0, st>>>(p.seg0, b.bits, p.ctl, p.sout, p.ray_rows, nunits);
    return hipGetLastError();
}

}  // namespace mc3d
