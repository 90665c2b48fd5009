// launch.h -- host-side launchers of the device stages (kernels.h).  Each
// group of kernels is compiled in a translation unit of its own (the corner
// kernel once per precision and statistics mode), so the library builds in
// parallel; mc3d.hip only sees these declarations.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "pipeline.h"

namespace mc3d {

// Device buffers of one call: the context's grow-only buffers, or pieces of
// the fixed scratch array of the allocation-free entry point.
struct Bufs {
    uint64_t *bits = nullptr;    // occupancy, one word per 64 x corners of a row
    uint32_t *counts = nullptr;  // packed per scan position
    uint2 *offs = nullptr;       // scanned {first vertex, first triangle}
    uint32_t *actw = nullptr;    // listed (emitting) words
    uint4 *tiles = nullptr;      // classify block sums
    ScanAgg *agg = nullptr;      // classify block sums of the one-pass scan (SCAN_ONE_PASS entries)
    uint2 *binfo = nullptr;      // per brick {code offset, length}
    uint32_t *actb = nullptr;    // active bricks
    Insn *bcode = nullptr;       // folded brick programs
    uint64_t *vkeys = nullptr;   // owning edge of each vertex
    uint32_t *vseg = nullptr;    // segment of each vertex (calls of several solids)
    const uint8_t *table = nullptr;   // 256-case table
    const uint8_t *etable = nullptr;  // the same with edges decoded for emit
    const uint64_t *keep = nullptr;   // block filter cube mask (one filtered solid)
};

// One call as the stage kernels see it.
struct Pipe {
    const Seg *segs = nullptr;
    uint32_t nsegs = 0;
    Seg seg0{};
    const uint32_t *word_seg = nullptr, *brick_seg = nullptr;  // segment tables (calls of several)
    const uint32_t *pos_seg = nullptr;  // segment per 64 scan positions (word_seg unless brick-major)
    Ctl *ctl = nullptr;
    SegOut *sout = nullptr;
    uint64_t nwords = 0, nbricks = 0, nscan = 0;
    uint32_t cap = 0;
    bool cull = false, bm = false, stats = false;
    int mode = 0, rows_per_walk = 1, wpb = 4;
    uint32_t plan_blocks = 0;  // 64-node blocks of the longest program that the plan lists
    uint32_t plan_gsz = 64;  // bricks per plan wave
    bool plan_tile = false;  // plan waves take compact tiles of bricks (one solid)
    bool scan_one_pass = false;  // classify scans its counts itself (at most SCAN_ONE_PASS blocks)
    bool rows = false;  // every atom has a row form: corners and bisection decide lines, not points
    int ray_rows = 0;   // the solid is a collider decided by rows, so many a wave (0: no)
    bool ray_rest = false;  // its last halvings are lookups, a launch of their own
    int stack = 1;      // boolean stack entries of the call's programs
    uint32_t emit_div = 1024;  // emit blocks: occupancy words / emit_div, in [512, 4096]
};

hipError_t launch_plan(const Pipe &p, const Bufs &b, hipStream_t st);
// Instantiated once per (MODE, STATS) in k_corners.hip.
template <int MODE, bool STATS>
hipError_t launch_corners_ms(const Pipe &p, const Bufs &b, hipStream_t st);
template <>
hipError_t launch_corners_ms<0, false>(const Pipe &p, const Bufs &b, hipStream_t st);
template <>
hipError_t launch_corners_ms<0, true>(const Pipe &p, const Bufs &b, hipStream_t st);
template <>
hipError_t launch_corners_ms<1, false>(const Pipe &p, const Bufs &b, hipStream_t st);
template <>
hipError_t launch_corners_ms<1, true>(const Pipe &p, const Bufs &b, hipStream_t st);
hipError_t launch_rows(const Pipe &p, const Bufs &b, hipStream_t st);
hipError_t launch_ray_rows(const Pipe &p, const Bufs &b, hipStream_t st);
inline hipError_t launch_corners(const Pipe &p, const Bufs &b, hipStream_t st) {
    if (p.rows) return launch_rows(p, b, st);
    if (p.ray_rows) return launch_ray_rows(p, b, st);
    if (p.mode == 0) return p.stats ? launch_corners_ms<0, true>(p, b, st) : launch_corners_ms<0, false>(p, b, st);
    return p.stats ? launch_corners_ms<1, true>(p, b, st) : launch_corners_ms<1, false>(p, b, st);
}
// zeroes bytes (a multiple of 16) of device memory with a kernel
hipError_t launch_zero(void *p, size_t bytes, hipStream_t st);
hipError_t launch_classify(const Pipe &p, const Bufs &b, hipStream_t st);
// the scan of classify's counts, the list of emitting words and (calls of
// several solids) each solid's output ranges
hipError_t launch_scan(const Pipe &p, const Bufs &b, hipStream_t st);
// A collider's triangles by planes (k_rays.hip): n ray-grid records into forms
// and extents, at[b] = the entries of bin b, *bad if one is too large for it;
// start and *total from at (left as the fill's cursors); the lists.
hipError_t launch_ray_forms(const double *rec, uint32_t n, const RayPlanes &R, double *forms, double *extent, uint32_t *at,
                            uint32_t *bad, hipStream_t st);
hipError_t launch_ray_scan(uint32_t *at, uint32_t bins, uint32_t *start, unsigned long long *total, hipStream_t st);
hipError_t launch_ray_fill(const double *extent, uint32_t n, const RayPlanes &R, uint32_t *at, uint32_t *list,
                           hipStream_t st);
hipError_t launch_emit(const Pipe &p, const Bufs &b, uint32_t *tris, uint64_t vcap, uint64_t tcap, hipStream_t st);
hipError_t launch_bisect_rows(const Pipe &p, const Bufs &b, double *verts, double *interior, uint64_t vcap,
                              hipStream_t st);
hipError_t launch_bisect_rays(const Pipe &p, const Bufs &b, double *verts, double *interior, uint64_t vcap,
                              hipStream_t st);
hipError_t launch_bisect(const Pipe &p, const Bufs &b, double *verts, double *interior, uint64_t vcap,
                         hipStream_t st);
hipError_t launch_bisect_host(int mode, const DevProg &P, const Grid &g, const uint64_t *bits,
                              const uint64_t *vkeys, double *state, double *probe, double *verts, double *interior,
                              uint64_t nv, int phase, hipStream_t st);
hipError_t launch_host_points(const DevProg &P, const Grid &g, const double *pts, uint32_t frame, uint64_t start,
                              uint64_t n, double *out, hipStream_t st);
hipError_t launch_contains(int mode, const DevProg &P, const double *pts, uint8_t *out, uint64_t n, hipStream_t st);
hipError_t launch_inverse_apply(const double *recs, uint32_t nops, double *verts, const Ctl *ctl, uint64_t vcap,
                                hipStream_t st);
// reads (write false) or writes `items` 16-byte items of buf; the read form
// writes one word per block (8192 blocks) to out
hipError_t launch_stream(bool write, void *buf, uint64_t items, uint32_t *out, hipStream_t st);
hipError_t launch_encode_stl(const double *verts, const uint32_t *tris, uint64_t nt, uint16_t *body,
                             hipStream_t st);

// A triangle's box.
struct GroupBox {
    double mn[3], mx[3];
};
// A mesh collider's triangles (9 doubles each) binned by their boxes in a
// uniform grid of n[0] x n[1] x n[2] cells: cell (x, y, z) holds
// cell_tris[cell_start[c], cell_start[c + 1]), c = (z * n[1] + y) * n[0] + x;
// point p is in cell floor((p - o) * inv), clamped to the grid.
// Beside it, a finer grid of the vertices that are a segment's origin (all
// but a triangle's largest, NewSegment's order) as a summed-volume table:
// vsat[(z * vn[1] + y) * vn[0] + x] counts those in cells <= (x, y, z).
struct RectGridDev {
    const double *tris = nullptr;
    const GroupBox *box = nullptr;
    uint32_t ntris = 0;
    const uint32_t *cell_start = nullptr, *cell_tris = nullptr;
    double o[3] = {0, 0, 0}, inv = 1;
    int n[3] = {1, 1, 1};
    const uint32_t *vsat = nullptr;
    double vo[3] = {0, 0, 0}, vinv = 1;
    int vn[3] = {1, 1, 1};
    const uint32_t *csat = nullptr;  // the same over the cells' list lengths
};
// A block of cubes [mn, mx) of MarchingCubesFilter's recursion (corner indices).
struct FBlock {
    int mn[3], mx[3];
};
// The recursion's filter: RectCollision of R with a block's bounds grown by
// eps, then by extra; accepted leaves set their cubes in keep (occupancy
// word layout, W words per row, ny rows per plane).
struct BlockFilter {
    RectGridDev R;
    const double *xs, *ys, *zs;
    double eps, extra;
    uint64_t *keep;
    int W, ny;
};
hipError_t launch_rgrid_gather(const double *verts, const uint32_t *tris, uint64_t nt, double *out, hipStream_t st);
// counts must start at zero
// (box: the triangles' boxes, R.box, are written here)
hipError_t launch_rgrid_count(const RectGridDev &R, GroupBox *box, uint32_t *counts, hipStream_t st);
// start (ncell + 1 entries) and cursor from the counts; tiles: ceil(ncell / 1024) <= 1024 entries
hipError_t launch_rgrid_scan(const uint32_t *counts, uint32_t ncell, uint32_t *tiles, uint32_t *start,
                             uint32_t *cursor, hipStream_t st);
hipError_t launch_rgrid_fill(const RectGridDev &R, uint32_t *cursor, uint32_t *cell_tris, hipStream_t st);
// R.vsat's table from the triangles: vsat must start at zero
hipError_t launch_vgrid(const RectGridDev &R, uint32_t *vsat, hipStream_t st);
// cell counts t of an n[0] x n[1] x n[2] grid into their summed-volume table
hipError_t launch_table(uint32_t *t, const int *n, hipStream_t st);
// the recursion from root, at most `depth` halvings deep, up to ocap (a multiple
// of 64, or 2^depth) leaves at a time (open: as many entries; nopen: 16 bytes)
hipError_t launch_block_filter(const BlockFilter &F, const FBlock &root, int depth, uint64_t *open, uint32_t *nopen,
                               uint32_t ocap, hipStream_t st);

// GroupTriangles (k_group.hip): one level of the recursion: the three orders, the axis of each of the level's 2^L nodes,
// the first-half flag of each triangle.
struct GroupLevel {
    uint32_t n = 0;
    int L = 0;
    const GroupBox *box = nullptr;
    const uint32_t *perm[3] = {nullptr, nullptr, nullptr};
    uint8_t *axis = nullptr;
    uint8_t *flag = nullptr;
};
// Entries first, first + step, ... of the three orders of n triangles (3 n of
// them, more than 32 bits from n = 2^32 / 3 on): f(axis, position).
template <class F>
MC3D_HD inline void each_order_entry(uint32_t n, uint64_t first, uint64_t step, F &&f) {
    for (uint64_t i = first; i < 3ull * n; i += step) {
        const int a = i >= 2ull * n ? 2 : (i >= n ? 1 : 0);
        f(a, (uint32_t)(i - (uint64_t)a * n));
    }
}
// boxes and midpoint keys of triangles (verts + tris, or 9 doubles each when
// tris is null): keys[a * n + t] with vals[a * n + t] = a * step + t
hipError_t launch_grp_boxes(const double *verts, const uint32_t *tris, uint32_t n, GroupBox *box, uint64_t *keys,
                            uint32_t *vals, uint32_t step, hipStream_t st);
// 3 n sorted values axis * n + triangle into the three orders, out[axis * n]
// on (counts: 3 * grp_tiles(3 n) entries of scratch)
hipError_t launch_grp_split(const uint32_t *vals, uint32_t n, uint32_t *counts, uint32_t *out, hipStream_t st);
// stable radix sort of (key, value) pairs (hipCUB; a null tmp asks for the
// temporary bytes)
hipError_t grp_sort(void *tmp, size_t &bytes, const uint64_t *keys_in, uint64_t *keys_out, const uint32_t *vals_in,
                    uint32_t *vals_out, uint32_t n, hipStream_t st);
// the axis of every node (slots: 36 keys per node)
hipError_t launch_grp_axis(const GroupLevel &G, unsigned long long *slots, hipStream_t st);
hipError_t launch_grp_flags(const GroupLevel &G, hipStream_t st);
// the three orders partitioned by the flags into out (counts: 3 *
// grp_tiles(n) entries of scratch)
uint32_t grp_tiles(uint32_t n);
hipError_t launch_grp_partition(const GroupLevel &G, uint32_t *counts, uint32_t *const out[3], hipStream_t st);
// all further levels of nodes of at most GROUP_LOCAL triangles: the x order
// into out (inv: n entries of scratch)
constexpr int GROUP_LOCAL = 1024;
hipError_t launch_grp_local(const GroupLevel &G, uint32_t *inv, uint32_t *out, hipStream_t st);
// out[k] = the three indices of triangle perm[k]
hipError_t launch_grp_apply(const uint32_t *tris, const uint32_t *perm, uint32_t n, uint32_t *out, hipStream_t st);

// z-slab stitching (k_slab.hip).  What a slab's rank pass leaves: the
// vertices on its bottom and its top plane, its own vertices, and whether a
// bottom vertex was missing below.
struct SlabEnd {
    uint32_t bottom, top, kept, bad;
};
// One slab's rank pass.  Vertices with keys vkeys; plane zbot is shared with
// the slab below and plane ztop with the one above (-1: none).  The slab's
// top plane goes into a table of 2^top_bits slots, at least twice the plane's
// vertices; the slab below left its own.  counts: slab_tiles(nv) entries of
// scratch.
struct SlabPart {
    const uint64_t *vkeys = nullptr;
    uint64_t nv = 0;
    uint32_t ntiles = 0;
    bool scanned = false;
    int zbot = -1, ztop = -1;
    uint64_t *top_keys = nullptr;
    uint32_t *top_vals = nullptr;
    int top_bits = 1;
    const uint64_t *below_keys = nullptr;
    const uint32_t *below_vals = nullptr;
    int below_bits = 1;
    const SlabEnd *below_end = nullptr;
    SlabEnd *end = nullptr;
    uint32_t *counts = nullptr, *rank = nullptr;
};
uint32_t slab_tiles(uint64_t nv);
hipError_t launch_slab_rank(SlabPart S, hipStream_t st);
// A slab's mesh and its place in the stitched one.
struct StitchPiece {
    const double *v, *in;
    const uint32_t *t, *rank;
    uint64_t nv, nt, tbase;
    uint32_t vbase, pad;
};
hipError_t launch_stitch(const StitchPiece *pieces, uint32_t npieces, uint64_t nv_max, uint64_t nt_max, double *fv,
                         double *fin, uint32_t *ft, hipStream_t st);

inline unsigned grid_for(uint64_t n, unsigned block, unsigned cap = 1u << 20) {
    uint64_t b = (n + block - 1) / block;
    if (b == 0) b = 1;
    return (unsigned)(b < cap ? b : cap);
}

}  // namespace mc3d
