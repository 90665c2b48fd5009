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

// The corners of one word (from x0, in row (y, z)) that a program holds for.
template <bool UNI, class CodeP, class F64P>
__device__ __forceinline__ uint64_t word_bits(CodeP code, uint32_t n, F64P f64, const Grid &g, int x0, int y, int z,
                                              uint64_t *stack) {
    const int last = min(63, g.nx - 1 - x0);
    const double *xs = g.xs + x0;
    const uint64_t m = row_program<UNI, uint64_t>(code, n, f64, 0, xs[0], g.ys[y], g.zs[z], 64 / g.inv_h, g.mag, g.inv_h,
                                                  g.eta, last, ~0ull, stack, 64, [&](int i) { return xs[i]; });
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
        for (int j = lane; j < nrows; j += 64) {
            const int jz = j / B.BY, y = by * B.BY + (j - jz * B.BY), z = bz * B.BZ + jz;
            if (y >= g.ny || z >= g.nz) continue;
            const uint64_t m = word_bits<true>(code, bi.y, scalar_ptr(sg.P.f64), g, bx * 64, y, z, stack);
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
    for (uint64_t gw = (uint64_t)blockIdx.x * 256 + threadIdx.x; gw < nwords; gw += (uint64_t)gridDim.x * 256) {
        const uint32_t si = wave_seg<MULTI>(word_seg, gw, SEG_WORD_SHIFT);
        const Seg sg = pick_seg<MULTI>(segs, seg0, si);
        const Grid &g = sg.g;
        const uint64_t w = gw - sg.word0;
        uint64_t m = 0;
        if (w < sg.nwords) {  // else alignment padding
            int wx, y, z;
            word_coords(g, w, wx, y, z);
            m = word_bits<true>(scalar_ptr(sg.P.code), sg.P.ncode, scalar_ptr(sg.P.f64), g, wx * 64, y, z, stack);
            check_faces(g, m, wx * 64, y, z, ctl, &sout[si]);
        }
        bits[gw] = m;
    }
}

}  // namespace

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
