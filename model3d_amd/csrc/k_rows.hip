// k_rows.hip -- Solid.Contains at the grid's corners a row at a time, for
// solids whose atoms are all untransformed spheres, boxes, capsules and
// cylinders (rows.h): a lane decides the 64 corners of one occupancy word.
//
// An atom costs a row one interval (15 to 120 float64 operations, a square
// root or three) instead of one evaluation (9 to 25) at each of its 64
// corners, and a wave walks a brick's program once instead of once per row.
// The kernel that evaluates corners was bound by issue on the scalar and
// vector units; this one waits for its chain of loads (list entry, brick
// record, code, params, coordinates), which several waves per SIMD hide.
// Measured against it (kernel trace, MI355X): 64 primitives at 402^3 corners
// 50 -> 12 us in 8 x 8 bricks (3,500 active), 93 -> 19 us in 4 x 4; 512
// primitives at 1.0 G corners 1,192 -> 129 us; a batch of 32 solids 168 ->
// 33 us; one sphere without culling at 102^3 8.9 -> 3.6 us.
#include "launch.h"
#include "rows.h"

#include "kernels.h"

namespace mc3d {
namespace {

// The corners of one word (from x0, in row (y, z)) that a program holds for,
// each lane its own word (live: it has one).  A word with more than a few open
// corners is taken by the whole wave, a lane a corner: one lane after another's
// 64 evaluations is what a wave would wait for (a row along a cylinder's side).
template <bool UNI, class CodeP, class F64P>
__device__ __forceinline__ uint64_t word_bits(CodeP code, uint32_t n, F64P f64, const Grid &g, int x0, int y, int z,
                                              bool live, uint64_t *stack) {
    const RowScale rs = row_scale(g);
    const int lane = threadIdx.x & 63, last = min(63, g.nx - 1 - x0);
    const double *xs = g.xs + x0;
    const double py = g.ys[y], pz = g.zs[z];
    const LineAxis<true> ax(0);
    auto rest = [&](uint32_t kind, auto a, uint64_t open) {
        if (__ballot(open != 0) == 0) return (uint64_t)0;
        uint64_t in = 0;
        for (uint64_t many = __ballot(__popcll(open) > FEW_OPEN); many; many &= many - 1) {
            const int j = __ffsll((unsigned long long)many) - 1;
            const double x = g.xs[min(__shfl(x0, j) + lane, g.nx - 1)];
            const uint64_t m = __ballot(atom64(kind, a, x, __shfl(py, j), __shfl(pz, j)));
            if (lane == j) in = m & open, open = 0;
        }
        return in | open_points(kind, a, ax, 0, py, pz, open, [&](int i) { return xs[i]; });
    };
    const uint64_t m = row_program<UNI, uint64_t>(code, n, f64, ax, xs[0], py, pz, 64 * rs.h, rs.mag, rs.inv_h, rs.eta, last,
                                                  live ? ~0ull : 0ull, stack, 64, rest);
    return m & (~0ull >> (63 - last));
}

// panic("solid is true outside of bounds"), mc.go:687-689: a corner of the
// word on a face of the grid is inside.
__device__ __forceinline__ void check_faces(const Grid &g, uint64_t m, int x0, int y, int z, Ctl *__restrict__ ctl,
                                            SegOut *__restrict__ so) {
    uint64_t face = 0;
    if (y == 0 || y == g.ny - 1 || z_face(g, z)) face = ~0ull;
    if (x0 == 0) face |= 1;
    if (g.nx - 1 - x0 < 64) face |= 1ull << (g.nx - 1 - x0);
    if (m & face) atomicOr(&ctl->inside, 1u), atomicOr(&so->inside, 1u);
}

// A wave per active brick, a lane per row: the brick's program is walked
// once with scalar loads for its 64 rows (8 x 8), each atom an interval test
// per row instead of one evaluation per corner.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_rows_act(const Seg *__restrict__ segs, const Seg seg0,
                                                  const uint32_t *__restrict__ brick_seg,
                                                  const uint32_t *__restrict__ act, uint64_t *__restrict__ bits_all,
                                                  Ctl *__restrict__ ctl, SegOut *__restrict__ sout, uint32_t nbricks,
                                                  int depth) {
    extern __shared__ __align__(16) uint64_t row_stack[];
    const int lane = threadIdx.x & 63, wave = wave_id();
    uint64_t *stack = row_stack + (size_t)wave * depth * 64 + lane;
    // the wave's first list entry loaded beside the count (the list holds
    // nbricks entries)
    const uint32_t k0 = blockIdx.x * 4 + wave;
    const uint32_t gb0 = k0 < nbricks ? scalar_ptr(act)[k0] : 0;
    const uint32_t nact = ctl->nact_bricks;
    for (uint32_t k = k0; k < nact; k += gridDim.x * 4) {
        const uint32_t gb = k == k0 ? gb0 : scalar_ptr(act)[k];
        const uint32_t si = wave_seg<MULTI>(brick_seg, gb, SEG_BRICK_SHIFT);
        const Seg sg = pick_seg<MULTI>(segs, seg0, si);
        const Grid &g = sg.g;
        const Bricks &B = sg.B;
        const uint32_t b = gb - (uint32_t)sg.brick0, r = b / (uint32_t)g.W;
        const int bx = (int)(b - r * (uint32_t)g.W);
        const int bz = (int)(r / (uint32_t)B.nby), by = (int)(r - (uint32_t)bz * (uint32_t)B.nby);
        const uint64_t biw = scalar_ptr((const uint64_t *)B.info)[gb];
        const uint2 bi = make_uint2((uint32_t)biw, (uint32_t)(biw >> 32));
        const auto code = scalar_ptr(brick_code(sg.P, B, bi));
        const int nrows = B.BY * B.BZ;
        for (int j0 = 0; j0 < nrows; j0 += 64) {
            const int j = j0 + lane, jz = j / B.BY, y = by * B.BY + (j - jz * B.BY), z = bz * B.BZ + jz;
            const bool live = j < nrows && y < g.ny && z < g.nz;
            const uint64_t m = word_bits<true>(code, bi.y, scalar_ptr(sg.P.f64), g, bx * 64, min(y, g.ny - 1), min(z, g.nz - 1),
                                               live, stack);
            if (!live) continue;
            bits_all[sg.word0 + word_index(g, bx, y, z)] = m;
            check_faces(g, m, bx * 64, y, z, ctl, &sout[si]);
        }
    }
}

// Without culling: a lane per occupancy word, the whole program.
template <bool MULTI>
__global__ __launch_bounds__(256) void k_rows_all(const Seg *__restrict__ segs, const Seg seg0,
                                                  const uint32_t *__restrict__ word_seg, uint64_t *__restrict__ bits,
                                                  Ctl *__restrict__ ctl, SegOut *__restrict__ sout, uint64_t nwords,
                                                  int depth) {
    extern __shared__ __align__(16) uint64_t row_stack[];
    uint64_t *stack = row_stack + (size_t)wave_id() * depth * 64 + (threadIdx.x & 63);
    // (word ranges are aligned to 64: a wave's words are one segment's)
    for (uint64_t w0 = (uint64_t)blockIdx.x * 256 + wave_id() * 64; w0 < nwords; w0 += (uint64_t)gridDim.x * 256) {
        const uint64_t gw = w0 + (threadIdx.x & 63);
        const uint32_t si = wave_seg<MULTI>(word_seg, gw, SEG_WORD_SHIFT);
        const Seg sg = pick_seg<MULTI>(segs, seg0, si);
        const Grid &g = sg.g;
        const uint64_t w = gw - sg.word0;
        const bool live = w < sg.nwords;  // else alignment padding
        int wx, y, z;
        word_coords(g, live ? w : 0, wx, y, z);
        const uint64_t m = word_bits<true>(scalar_ptr(sg.P.code), sg.P.ncode, scalar_ptr(sg.P.f64), g, wx * 64, y, z, live, stack);
        if (live) check_faces(g, m, wx * 64, y, z, ctl, &sout[si]);
        if (gw < nwords) bits[gw] = live ? m : 0;
    }
}

// The program as a mask over the dyadic points of the bracket [lo, hi] on
// axis k of the line through p: bit i is the point that halving the bracket
// reaches at i / 2^levels.  dense: an atom leaves more than a few points open,
// and the mask says nothing.
template <bool UNI, class CodeP, class F64P>
__device__ __forceinline__ uint64_t bracket_bits(CodeP code, uint32_t n, F64P f64, const Grid &g,
                                                 const LineAxis<false> &ax, double lo, double hi, double x, double y,
                                                 double z, int levels, uint64_t *stack, bool &dense) {
    const int k = ax.k;
    const double scale = (double)(1 << levels) * recip(hi - lo);
    const double mag = row_scale(g).mag, eta = bracket_eta(mag, scale);
    const double qx = k == 0 ? lo : x, qy = k == 1 ? lo : y, qz = k == 2 ? lo : z;
    auto rest = [&](uint32_t kind, auto a, uint64_t open) -> uint64_t {
        if (open == 0) return 0;
        if (__popcll(open) > FEW_OPEN) {
            dense = true;
            return 0;
        }
        return open_points(kind, a, ax, qx, qy, qz, open, [&](int i) { return bracket_point(lo, hi, levels, i); });
    };
    const int last = (1 << levels) - 1;
    return row_program<UNI, uint64_t>(code, n, f64, ax, qx, qy, qz, hi - lo, mag, scale, eta, last, ~1ull, stack, 256, rest);
}

// `left` halvings of the bracket [lo, hi] of a vertex (mcSearchPoint, mc.go:
// 223-258): up to six are decided at a time by the program's mask over the
// points they can reach, the last one or two by evaluating it (a second mask
// costs more than two evaluations, the last of three or more would not: 8
// halvings as 6 + 2 took 31.6 -> 28.4 us, 573 -> 531 us against two masks).
// Where an atom leaves more than a few of a bracket's points open -- its bounds
// are no finer than the points after some 28 halvings, or far from the origin;
// an edge may touch a cylinder's side -- the wave evaluates all further
// halvings: deciding open points one by one is up to 63 evaluations for six
// halvings (one sphere at 102^3 corners, 64 halvings, whole calls: 357 us so, 75
// with the evaluations alone, 51 us for 8 halvings).
//
// Evaluating every halving is a chain of dependent program walks, bound by the
// latency of its loads where few waves run (a small part) and by the walks'
// scalar and vector issue where many do; one walk decides six halvings here.
// Bound by vector issue now, at 3 waves per SIMD (138 registers; 159 for several
// solids).  UNI: one program for the wave.
template <bool UNI>
__device__ __forceinline__ void halve(const Insn *code, uint32_t n, const DevProg &P, const Grid &g, int k, double px, double py,
                                      double pz, bool up, int left, double &lo, double &hi, uint64_t *stack) {
    const LineAxis<false> ax(k);
    bool dense = false;  // (then the wave halves on point by point)
    while (left > 2 && __ballot(dense) == 0) {
        const int levels = min(left, 6);
        uint64_t m;
        if constexpr (UNI) m = bracket_bits<true>(scalar_ptr(code), n, scalar_ptr(P.f64), g, ax, lo, hi, px, py, pz, levels, stack, dense);
        else m = bracket_bits<false>(code, n, P.f64, g, ax, lo, hi, px, py, pz, levels, stack, dense);
        if (dense) continue;
        for (int bit = 1 << (levels - 1), at = 0; bit; bit >>= 1) {
            const double mid = (lo + hi) / 2;
            const bool in = (m >> (at + bit)) & 1;
            if (in == up) hi = mid;  // the inside end moves
            else lo = mid, at += bit;
        }
        left -= levels;
    }
    for (; left > 0; left--) {
        const double mid = (lo + hi) / 2;
        GStats gs;
        const bool in = eval_code<0, false, UNI>(code, n, P, k == 0 ? mid : px, k == 1 ? mid : py, k == 2 ? mid : pz, gs);
        if (in == up) hi = mid;
        else lo = mid;
    }
}

// One vertex.  Measured (kernel trace, MI355X, 8 halvings, against a walk for each
// halving): 1,100 vertices 23 -> 12 us, 411k vertices of 64 primitives 43 -> 31 us
// (with the float32 guard 64 -> 35 us), a batch of 32 solids 173 -> 109 us, 10.1M
// vertices of 512 primitives 819 -> 670 us.
__device__ __forceinline__ void bisect_rows(const Seg &sg, const uint64_t *__restrict__ bits_all, const uint64_t key,
                                            double *__restrict__ verts, double *__restrict__ interior, uint64_t v,
                                            uint64_t *stack) {
    const DevProg &P = sg.P;
    const Grid &g = sg.g;
    const Bricks &B = sg.B;
    const uint64_t *bits = bits_all + sg.word0;
    const int k = (int)(key & 3);
    const int x = (int)((key >> 2) & 0xfffff), y = (int)((key >> 22) & 0xfffff), z = (int)((key >> 42) & 0xfffff);
    const double px = g.xs[x], py = g.ys[y], pz = g.zs[z];
    double lo = sel3(k, px, py, pz), hi = *(k == 0 ? g.xs + x + 1 : (k == 1 ? g.ys + y + 1 : g.zs + z + 1));
    // the high corner decides which end is inside
    const bool up = corner_bit(g, bits, x + (k == 0), y + (k == 1), z + (k == 2));
    if (sg.iters > 0) {
        // the edge's brick program (an edge crossed in a brick that the plan
        // found constant is decided by that constant, as in bisect_vertex)
        uint2 bi = make_uint2(BRICK_FULL, P.ncode);
        if (B.info) bi = B.info[sg.brick0 + ((size_t)(z / B.BZ) * B.nby + (y / B.BY)) * g.W + (x >> 6)];
        const uint32_t at0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)bi.x);
        const uint32_t n0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)bi.y);
        const bool uni = __ballot(bi.x != at0 || bi.y != n0) == 0;  // one program for the wave: scalar loads
        int left = sg.iters;
        if (brick_constant(bi.y))  // (no halvings are left for a walk of its record's length)
            for (; left > 0; left--) ((bi.y == BRICK_TRUE) == up ? hi : lo) = (lo + hi) / 2;
        if (uni) halve<true>(brick_code(P, B, make_uint2(at0, n0)), n0, P, g, k, px, py, pz, up, left, lo, hi, stack);
        else halve<false>(brick_code(P, B, bi), bi.y, P, g, k, px, py, pz, up, left, lo, hi, stack);
    }
    const double res = (lo + hi) / 2;
    verts[3 * v] = k == 0 ? res : px;
    verts[3 * v + 1] = k == 1 ? res : py;
    verts[3 * v + 2] = k == 2 ? res : pz;
    if (interior) {
        const double in = up ? hi : lo;  // the bracket's inside end (mc.go:252-255)
        interior[3 * v] = k == 0 ? in : px;
        interior[3 * v + 1] = k == 1 ? in : py;
        interior[3 * v + 2] = k == 2 ? in : pz;
    }
}

template <bool MULTI>
__global__ __launch_bounds__(256) void k_bisect_rows(const Seg *__restrict__ segs, const Seg seg0,
                                                     const uint32_t *__restrict__ vseg,
                                                     const uint64_t *__restrict__ bits_all,
                                                     const uint64_t *__restrict__ vkeys, double *__restrict__ verts,
                                                     double *__restrict__ interior, const Ctl *__restrict__ ctl,
                                                     uint64_t vcap) {
    extern __shared__ __align__(16) uint64_t row_stack[];
    uint64_t *stack = row_stack + threadIdx.x;
    // the first vertex's key (and solid) loaded beside the vertex count: the
    // arrays hold vcap entries, so the loads stay in bounds
    const uint64_t v0 = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t key0 = v0 < vcap ? vkeys[v0] : 0;
    const uint32_t mine0 = MULTI && v0 < vcap ? vseg[v0] : 0u;
    const uint64_t nv = min((uint64_t)ctl->totals[0], vcap);
    for (uint64_t v = v0; v < nv; v += (uint64_t)gridDim.x * 256) {
        const uint64_t key = v == v0 ? key0 : vkeys[v];
        // lanes may belong to different solids: one solid at a time (every
        // lane stays in the loop, so the solid is one for the wave in it)
        const uint32_t mine = MULTI ? (v == v0 ? mine0 : vseg[v]) : 0u;
        for (uint64_t todo = __ballot(true); todo;) {
            const uint32_t si =
                MULTI ? (uint32_t)__builtin_amdgcn_readlane((int)mine, __ffsll((unsigned long long)todo) - 1) : 0u;
            const bool here = !MULTI || mine == si;
            if (here) bisect_rows(pick_seg<MULTI>(segs, seg0, si), bits_all, key, verts, interior, v, stack);
            todo &= ~__ballot(here);
        }
    }
}

}  // namespace

hipError_t launch_bisect_rows(const Pipe &p, const Bufs &b, double *verts, double *interior, uint64_t vcap,
                              hipStream_t st) {
    const int depth = p.stack > 1 ? p.stack - 1 : 1;
    const size_t lds = (size_t)depth * 256 * sizeof(uint64_t);
    const unsigned grid = grid_for(vcap, 256, 1u << 14);
    if (p.nsegs > 1)
        k_bisect_rows<true><<<grid, 256, lds, st>>>(p.segs, p.seg0, b.vseg, b.bits, b.vkeys, verts, interior, p.ctl, vcap);
    else
        k_bisect_rows<false><<<grid, 256, lds, st>>>(p.segs, p.seg0, nullptr, b.bits, b.vkeys, verts, interior, p.ctl,
                                                     vcap);
    return hipGetLastError();
}

hipError_t launch_rows(const Pipe &p, const Bufs &b, hipStream_t st) {
    const int depth = p.stack > 1 ? p.stack - 1 : 1;  // masks below the top
    const size_t lds = (size_t)4 * depth * 64 * sizeof(uint64_t);
    if (p.cull) {
        const unsigned grid = grid_for(p.nbricks, 4, 4096);
        if (p.nsegs > 1)
            k_rows_act<true><<<grid, 256, lds, st>>>(p.segs, p.seg0, p.brick_seg, b.actb, b.bits, p.ctl, p.sout,
                                                     (uint32_t)p.nbricks, depth);
        else
            k_rows_act<false><<<grid, 256, lds, st>>>(p.segs, p.seg0, p.brick_seg, b.actb, b.bits, p.ctl, p.sout,
                                                      (uint32_t)p.nbricks, depth);
    } else {
        const unsigned grid = grid_for(p.nwords, 256, 1u << 16);
        if (p.nsegs > 1)
            k_rows_all<true><<<grid, 256, lds, st>>>(p.segs, p.seg0, p.word_seg, b.bits, p.ctl, p.sout, p.nwords, depth);
        else
            k_rows_all<false><<<grid, 256, lds, st>>>(p.segs, p.seg0, p.word_seg, b.bits, p.ctl, p.sout, p.nwords,
                                                      depth);
    }
    return hipGetLastError();
}

}  // namespace mc3d
